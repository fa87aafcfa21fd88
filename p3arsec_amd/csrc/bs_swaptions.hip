// bs_swaptions.hip -- the swaptions map of p3arsec: HJM Monte-Carlo prices of
// a portfolio of swaptions (parsec-ff/pkgs/apps/swaptions/src).
//
// The reference maps HJM_Swaption_Blocking (HJM_Swaption_Blocking.cpp:20-222)
// over the swaptions with a FastFlow ParallelFor (HJM_Securities.cpp:311-323),
// each swaption simulating its trials serially in blocks of BLOCK_SIZE paths.
// Here every Monte-Carlo path of every swaption is one GPU work-item.
//
// Per path p of swaption i the reference draws (n-1) F uniforms from the
// counter seed_i + p (n-1) F + (s-1) F + k (time step s, factor k: its
// generator advances the counter by one per draw and draws path by path),
// maps them through Moro's inverse normal, evolves the forward curve
//   f(s, l) = f(s-1, l+1) + mu[l] dt + sqrt(dt) sum_k sigma_k[l] Z_k(s)
// for every step, discounts along the short rate f(s, 0) and prices the swap
// on the curve f(m, .) at the swaption's start m.
//
// Every exponent of that payoff is linear in the path's draws: the payoff
// reads the short rates before m and the curve at m, the model is Gaussian,
// and a discount factor is the exponential of a sum of rates.  So a path of
// k_sw_paths is
//   max(sum_c pay_c 2^(C_c + sum_j G_cj Z_j) - 1, 0) 2^(C_0 + sum_j G_0j Z_j)
// over the m F draws Z_j before the start and the swap's cash flows c (the
// reference multiplies the discount factors between them by zero), with C and
// G formed once per swaption on the host: one FMA per draw and cash flow and
// one exponential per cash flow, where the recursion takes them per curve
// point and step.  It holds wherever the reference's running products neither
// overflow nor underflow (pack_linear bounds them) and every draw is finite
// (a counter that is a multiple of 2^31-1 draws u = 0, whose normal is
// infinite); blocks of paths where it may not hold are left to
// k_sw_paths_steps, which follows the reference statement by statement.  The
// prices are the reference's up to rounding: measured against the oracle's
// restatement, 1e-15 relative.
//
// Generator: the reference's RanUnif (PARSEC 3.0 RanUnif.cpp, not in the
// reference tree) is the Park-Miller minimal standard generator applied to
// 1513517 c mod (2^31-1).  Both products together are A c mod (2^31-1) with
// A = 16807 * 1513517, the same residues as its Schrage factorisation, so the
// residue of the next counter is one 32-bit addition away.
//
// Kernels (the caller's stream): k_sw_paths, 2 to 32 paths per work-item, and,
// where it left paths out, k_sw_paths_steps, each unit's sums of payoff and
// payoff^2 (512 to 2048 paths) folded in a fixed order into one partial; a
// swaption's partials are added in a fixed order and its mean and standard error
// formed as the reference does, by its last block in a small launch and by
// k_sw_final else.  A swaption's results are the same bits in every call.
// The arithmetic is FP64 (the reference's FTYPE); this file is compiled
// without FMA contraction, so the step-by-step kernel rounds every product and
// sum as the reference does and the other one's FMAs are the ones written.
#include <climits>
#include <cmath>
#include <cstdio>
#include <cstring>

#include <algorithm>
#include <chrono>
#include <mutex>
#include <vector>

#include "bs_arrive.hpp"
#include "bs_fp64.hpp"
#include "bs_internal.hpp"
#include "bs_moro.hpp"
#include "bs_wave.hpp"

namespace bs {
namespace {

constexpr int kSwThreads = 256;
constexpr int kSwRows = 4;                // paths per work-item that limits are stated in
constexpr int kSwMaxSteps = 64;           // n_steps
constexpr int kSwMaxFactors = 8;          // n_factors
constexpr int kSwMaxDraws = 64;           // start index x n_factors
constexpr int64_t kSwCounterLimit = int64_t(1) << 42;

// How a launch's blocks cover the paths: block b takes swaption b / bps, its
// paths [(b % bps) kSwThreads rows, + kSwThreads rows), `rows` of them per
// work-item, kSwThreads apart.
struct SwGrid {
    int64_t paths;
    int32_t bps, rows;
};

// A swaption's paths are summed in units of kSwThreads unit_rows paths, each
// into a partial of its own.  The unit, and with it the order of the sums, comes
// from the swaption and its number of paths alone, so a swaption's results are
// the same bits in every call, whatever else the call prices and however its
// blocks are cut (`rows` is a multiple of every unit).
//
// A unit costs a wave 18 VALU instructions (two together 21) beside the 200 or
// more of each row of paths, and no work-item has fewer rows than a unit of its
// call, which leaves small calls with too few blocks.  Units of 2, 4 and 8 rows, us
// a call, swaptions of the driver (3 or 6 draws): 128 x 1M trials 790, 793, 774,
// 1 x 1M 41.6, 30.2, 25.8; 128 x 300,000 273, 274, 267; 8 x 262,144 36.3, 36.2,
// 33.5, 1 x 262,144 23.4, 20.9, 21.2; 64 x 20,000 42.5, 42.0, 42.5, 16 x 10,000
// 23.8, 25.2, 28.8.  With more draws (24 steps, 4 factors, starts at steps 1-12)
// 8 x 50,000 43.2, 58.2, 89.0, and 1 x 1M (start at step 8) 87.7, 87.4, 105, 16 x 1M
// 900, 897, 901.
constexpr int kSwMaxUnits = 16;   // of a block
constexpr int unit_rows(bool narrow, int64_t paths) {
    return narrow && paths >= (1 << 18) ? 8 : 2;
}

// One swaption as the step-by-step kernel reads it.  pool + off holds f0[n] (the forward
// curve at t = 0), mudt[n-1] (total drift x dt), sigma[F][n-1] and pay[L]
// (the swap's cash flows per unit notional).
struct SwHead {
    int64_t seed;        // counter of path 0's first draw
    double dt, sdt, dts; // HJM step, its square root, the swap curve's step
    int32_t n, m, L, off;
};
static_assert(sizeof(SwHead) == 48, "SwHead layout");

__device__ __forceinline__ uint64_t mod_m31(uint64_t x) {   // x < 2^63
    x = (x & kM31) + (x >> 31);
    x = (x & kM31) + (x >> 31);
    return x >= kM31 ? x - kM31 : x;
}

// RanUnif of counter c (0 <= c < 2^42).
__device__ __forceinline__ double ran_unif(int64_t c) {
    uint64_t x = mod_m31((uint64_t)c * 1513517u);
    x = mod_m31(x * 16807u);
    return (double)(int64_t)x * 4.656612875e-10;
}

// Loops over a path's steps are unrolled where its draws then fit registers.
constexpr int unrolled(int factors, int steps) {
    return steps <= 8 && steps * factors <= 32 ? steps : 1;
}

// The normal draws of path p: z[s][k] = Z_k(s + 1) for s < m <= MAXM.
template <int F, int MAXM>
__device__ __forceinline__ void draws(const SwHead& h, int64_t p, double (&z)[MAXM][F]) {
    constexpr int kUnroll = unrolled(F, MAXM);
    const int64_t c0 = h.seed + p * (int64_t)((h.n - 1) * F);
#pragma unroll kUnroll
    for (int s = 0; s < MAXM; ++s) {
        if (s >= h.m) break;
#pragma unroll
        for (int k = 0; k < F; ++k) z[s][k] = moro_inv(ran_unif(c0 + s * F + k));
    }
}

// Discounted payoff of a path from its draws z, the reference's arithmetic
// statement by statement: each forward chain d (f(0,d) -> f(1,d-1) -> ...)
// takes the steps 1..min(d, m) that the payoff reads, with the reference's
// additions in the reference's order.
template <int F, int MAXM>
__device__ __forceinline__ double path_payoff(const SwHead& h, const double* __restrict__ q,
                                              const double (&z)[MAXM][F]) {
    constexpr int kUnroll = unrolled(F, MAXM);
    const int n = h.n, m = h.m, L = h.L, w = n - 1;
    const double* f0 = q;
    const double* mudt = q + n;
    const double* sigma = q + n + w;
    const double* pay = q + n + w + F * w;
    double df = 1.0, sdf = 1.0, leg = 0.0;
    const int dend = min(n, m + L);
    for (int d = 0; d < dend; ++d) {
        double x = f0[d];
        const int steps = min(d, m);
#pragma unroll kUnroll
        for (int s = 1; s <= MAXM; ++s) {
            if (s > steps) break;
            const int l = d - s;
            double shock = 0.0;
#pragma unroll
            for (int k = 0; k < F; ++k) shock += sigma[k * w + l] * z[s - 1][k];
            x = x + mudt[l] + h.sdt * shock;
        }
        if (d < m) {
            df *= exp(-x * h.dt);
        } else {
            const int l = d - m;
            leg += pay[l] * sdf;
            if (l < L - 1) sdf *= exp(-x * h.dts);
        }
    }
    // curve points past the simulated horizon are zero rates: factor exp(-0) = 1
    for (int l = n - m; l < L; ++l) leg += pay[l] * sdf;
    const double payoff = leg - 1.0 > 0 ? leg - 1.0 : 0;
    return payoff * df;
}

// ---- the linear form --------------------------------------------------------------
// One swaption as k_sw_paths reads it; pool + off holds, for W = the width of
// its form (lin_width: at least `flows`, padded with zeros), C[W], pay[W],
// G[draws][W] and Gdf[draws].  Exponents are in base 2.
struct SwLin {
    int64_t seed;        // counter of path 0's first draw
    double c_df;         // C of the discount to the swaption's start
    uint32_t per_path;   // counters a path takes, (n-1) F
    uint32_t x_path;     // A per_path mod M: residue step to the next path
    uint32_t x_row;      // A kSwThreads per_path mod M: to a work-item's next path
    int32_t draws;       // m F, those the payoff reads
    int32_t df_draws;    // (m-1) F, those the discount to the start reads
    int32_t flows;       // cash flows
    int32_t off;
    int32_t linear;      // 0: every block is left to k_sw_paths_steps
    int32_t unit, units; // rows of a unit, and how many units hold the paths
    int32_t unit0;       // the first one's place among the launch's partials
    int32_t pad;
};
static_assert(sizeof(SwLin) == 64, "SwLin layout");

constexpr uint32_t kGenA = (uint32_t)(uint64_t(16807) * 1513517u % kM31);
constexpr uint32_t gen_step(uint64_t counters) {
    return (uint32_t)(counters % kM31 * kGenA % kM31);
}

// a + b mod M for residues a, b < M = 2^31-1.
__device__ __forceinline__ uint32_t add_m31(uint32_t a, uint32_t b) {
    const uint32_t t = a + b;
    return min(t, t - (uint32_t)kM31);   // t < M: t - M wraps past it
}

// Whether the linear form takes the kSwThreads rows paths from `first` on: the
// swaption is bounded and none of their counters draws u = 0.
__device__ __forceinline__ bool rows_linear(const SwLin& h, int64_t first, int rows) {
    const uint64_t span = (uint64_t)(kSwThreads * rows) * h.per_path;
    const uint64_t r = mod_m31((uint64_t)h.seed + (uint64_t)first * h.per_path);
    return h.linear && r != 0 && r + span <= kM31;
}

// A wave's sums of a unit, or of two next to one another, left in LDS: the two
// quantities are halved into one register (the lower lanes' of sumsq against the
// upper lanes' of sum), two units' registers into one (rows of 16 lanes against
// rows), and all fold at once within a row; 18 instructions for one unit, 21 for
// two.  The additions are the same ones either way.
using UnitSums = double[kSwThreads / 64][kSwMaxUnits][2];
__device__ __forceinline__ void wave_sums(double sum, double sumsq, double (&to)[2]) {
    const double a = swap_halves_add(sum, sumsq);
    const double x = row_sums(swap_rows_add(a, a));
    const int lane = threadIdx.x & 63;
    if ((lane & 31) == 15) to[lane >> 5] = x;
}
__device__ __forceinline__ void wave_sums(double sum, double sumsq, double sum2, double sumsq2,
                                          double (*to)[2]) {
    const double x = row_sums(
        swap_rows_add(swap_halves_add(sum, sumsq), swap_halves_add(sum2, sumsq2)));
    const int lane = threadIdx.x & 63, row = lane >> 4;
    if ((lane & 15) == 15) to[row & 1][row >> 1] = x;
}

// Sums of payoff and payoff^2.
struct SwSums {
    double sum = 0.0, sumsq = 0.0;
    __device__ __forceinline__ void add(double v) {
        sum += v;
        sumsq = __builtin_fma(v, v, sumsq);
    }
};

// A work-item's paths, a unit at a time: paths(at, s, s') adds the PP paths at,
// at + kSwThreads, ... and advances xb past them, the first half to s and the
// second to s'.  PAIRS: two units of PP / 2 rows at a time.  Units that hold a
// zero draw are left to k_sw_paths_steps (whole: none does; beside one that is
// summed their paths are drawn all the same, and the sums dropped).  Bit u of the
// result: unit u was summed into sums[u].
template <int PP, bool PAIRS, class Paths>
__device__ __forceinline__ uint32_t over_units(const SwLin& h, const SwGrid& grid, int64_t first,
                                               bool whole, uint32_t& xb,
                                               double (*__restrict__ sums)[2], Paths&& paths) {
    const int64_t end = min(first + kSwThreads * grid.rows, grid.paths);
    const int unit = PAIRS ? PP / 2 : h.unit, rows = PAIRS ? PP : unit;
    uint32_t done = 0;
    int u = 0;
#pragma unroll 1
    for (int64_t at = first; at < end; at += kSwThreads * rows, u += PAIRS ? 2 : 1) {
        uint32_t take = whole || rows_linear(h, at, unit) ? 1u : 0u;
        if constexpr (PAIRS) {
            const int64_t next = at + kSwThreads * unit;
            if (next < end && (whole || rows_linear(h, next, unit))) take |= 2u;
        }
        if (!take) {
            for (int row = 0; row < rows; ++row) xb = add_m31(xb, h.x_row);
            continue;
        }
        const int64_t p = at + (int)threadIdx.x;
        SwSums a;
        if constexpr (PAIRS) {
            SwSums b;
            paths(p, a, b);
            wave_sums(a.sum, a.sumsq, b.sum, b.sumsq, sums + u);
        } else {
#pragma unroll 1
            for (int row = 0; row < rows; row += PP) paths(p + row * kSwThreads, a, a);
            wave_sums(a.sum, a.sumsq, sums[u]);
        }
        done |= take << u;
    }
    return done;
}

// Keeps the compiler from moving the lanes' accesses to their wave's LDS list
// across this point; the hardware performs a wave's LDS accesses in order.
__device__ __forceinline__ void wave_lds_order() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// The h.draws <= DB draws of PP paths, added into the paths' exponents.  FULL:
// h.draws = DB.  xs holds each path's residue at its first draw.
//
// Moro's tail (16% of draws, but taken by nearly every wave at every draw when
// each lane branches on its own) is compacted over the batch: the lanes write
// the residues that need it to their wave's LDS list (ballot and mbcnt give
// the places), all lanes evaluate the list, and each owner reads its results
// back.  PP DB = 12 draws make 123 list entries a batch on average, so the
// last of its rounds of 64 wastes little.
template <int W, int PP, int DB, bool FULL>
__device__ __forceinline__ void linear_batch(const SwLin& h, const double* __restrict__ G,
                                             const double* __restrict__ gdf,
                                             const uint32_t (&xs)[PP], char* lds, uint32_t wl,
                                             const MoroCentral& central,
                                             double (&acc)[PP][W], double (&dfe)[PP]) {
    const int lane = __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
    double z[PP][DB];
    bool tail[PP][DB];
    uint32_t at[PP][DB];   // a tail draw's list entry (its offset in lds)
    int count = 0;       // the wave's list so far (uniform)
#pragma unroll
    for (int j = 0; j < DB; ++j) {
        if (FULL || j < h.draws) {
#pragma unroll
            for (int p = 0; p < PP; ++p) {
                const uint32_t x = add_m31(xs[p], gen_step(j));
                z[p][j] = central(x);
                tail[p][j] = x - (kTailLo + 1) >= kTailHi - (kTailLo + 1);
                const uint64_t b = __ballot(tail[p][j]);
                at[p][j] = (wl + 8 * (uint32_t)count) +
                           8 * __builtin_amdgcn_mbcnt_hi((uint32_t)(b >> 32),
                                                         __builtin_amdgcn_mbcnt_lo((uint32_t)b, 0u));
                if (tail[p][j]) *reinterpret_cast<uint32_t*>(lds + at[p][j]) = x;
                count += __popcll(b);
            }
        }
    }
    wave_lds_order();
    for (int r = 0; r < count; r += 64) {
        const int i = r + lane;
        if (i < count) {
            const uint32_t e = wl + 8 * (uint32_t)i;
            *reinterpret_cast<double*>(lds + e) = moro_tail_fma(
                *reinterpret_cast<const uint32_t*>(lds + e));
        }
    }
    wave_lds_order();
#pragma unroll
    for (int j = 0; j < DB; ++j) {
        if (FULL || j < h.draws) {
            const double* __restrict__ g = G + j * W;
#pragma unroll
            for (int p = 0; p < PP; ++p)
                if (tail[p][j]) z[p][j] = *reinterpret_cast<const double*>(lds + at[p][j]);
#pragma unroll
            for (int c = 0; c < W; ++c)
#pragma unroll
                for (int p = 0; p < PP; ++p)
                    acc[p][c] = __builtin_fma(g[c], z[p][j], acc[p][c]);
            if (j < h.df_draws) {
#pragma unroll
                for (int p = 0; p < PP; ++p)
                    dfe[p] = __builtin_fma(gdf[j], z[p][j], dfe[p]);
            }
        }
    }
    wave_lds_order();   // the list is rewritten by the next batch
}

// The paths of a work-item, PP at a time.
template <int W, int PP, int DB, bool PAIRS>
__device__ __forceinline__ uint32_t linear_paths(const SwLin& h, const double* __restrict__ q,
                                                 uint32_t xb, int64_t first, bool whole,
                                                 const SwGrid& grid, char* lds, uint32_t wl,
                                                 double (*__restrict__ sums)[2]) {
    const double* __restrict__ pay = q + W;
    const double* __restrict__ G = q + 2 * W;
    const double* __restrict__ gdf = G + h.draws * W;
    const double df0 = exp2_mid(h.c_df);
    const MoroCentral central;
    return over_units<PP, PAIRS>(h, grid, first, whole, xb, sums,
                                 [&](int64_t p0, SwSums& low, SwSums& high) {
        double acc[PP][W], dfe[PP];
        uint32_t xs[PP];
#pragma unroll
        for (int p = 0; p < PP; ++p) {
#pragma unroll
            for (int c = 0; c < W; ++c) acc[p][c] = q[c];
            dfe[p] = h.c_df;
            xs[p] = xb;
            xb = add_m31(xb, h.x_row);
        }
        if (h.draws == DB)
            linear_batch<W, PP, DB, true>(h, G, gdf, xs, lds, wl, central, acc, dfe);
        else
            linear_batch<W, PP, DB, false>(h, G, gdf, xs, lds, wl, central, acc, dfe);
        double leg[PP];
#pragma unroll
        for (int p = 0; p < PP; ++p) leg[p] = -1.0;
#pragma unroll
        for (int c = 0; c < W; ++c)
#pragma unroll
            for (int p = 0; p < PP; ++p)
                leg[p] = __builtin_fma(pay[c], exp2_mid(acc[p][c]), leg[p]);
        double df[PP];
#pragma unroll
        for (int p = 0; p < PP; ++p) df[p] = df0;
        if (h.df_draws > 0) {
#pragma unroll
            for (int p = 0; p < PP; ++p) df[p] = exp2_mid(dfe[p]);
        }
#pragma unroll
        for (int p = 0; p < PP; ++p) {
            double v = (leg[p] > 0 ? leg[p] : 0) * df[p];
            v = p0 + p * kSwThreads < grid.paths ? v : 0.0;
            (p < PP / 2 ? low : high).add(v);
        }
    });
}

// The paths of a work-item one at a time, for many draws or cash flows: only
// the W exponents stay in registers.  The draws of a batch live in LDS, slot
// j 64 + lane: a central draw's normal, or a tail draw's residue until the
// compacted evaluation (as in linear_batch, over a list of slots) replaces it.
constexpr int kWideDraws = 12;   // draws in a batch
constexpr uint32_t kWideBytes = kWideDraws * 64 * (8 + 2);   // a wave's slots and list

template <int W>
__device__ __forceinline__ uint32_t linear_wide(const SwLin& h, const double* __restrict__ q,
                                                uint32_t xb, int64_t first, bool whole,
                                                const SwGrid& grid, char* lds,
                                                double (*__restrict__ sums)[2]) {
    const double* __restrict__ pay = q + W;
    const double* __restrict__ G = q + 2 * W;
    const double* __restrict__ gdf = G + h.draws * W;
    const double df0 = exp2_mid(h.c_df);
    const MoroCentral central;
    const int lane = __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane(threadIdx.x / 64);
    char* slots = lds + wave * kWideBytes;
    uint16_t* list = reinterpret_cast<uint16_t*>(slots + kWideDraws * 64 * 8);
    char* mine = slots + lane * 8;
    return over_units<1, false>(h, grid, first, whole, xb, sums,
                                [&](int64_t p0, SwSums& to, SwSums&) {
        double acc[W], dfe = h.c_df;
#pragma unroll
        for (int c = 0; c < W; ++c) acc[c] = q[c];
        uint32_t x = xb;
        xb = add_m31(xb, h.x_row);
#pragma unroll 1
        for (int j0 = 0; j0 < h.draws; j0 += kWideDraws) {
            const int nj = min(kWideDraws, h.draws - j0);
            int count = 0;
#pragma unroll 2
            for (int j = 0; j < nj; ++j) {
                const bool tail = x - (kTailLo + 1) >= kTailHi - (kTailLo + 1);
                const uint64_t b = __ballot(tail);
                *reinterpret_cast<double*>(mine + j * 512) = central(x);
                if (tail) {
                    const uint32_t at = __builtin_amdgcn_mbcnt_hi(
                        (uint32_t)(b >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)b, 0u));
                    *reinterpret_cast<uint32_t*>(mine + j * 512) = x;
                    list[count + at] = (uint16_t)(j * 512 + lane * 8);
                }
                count += __popcll(b);
                x = add_m31(x, gen_step(1));
            }
            wave_lds_order();
            for (int r = 0; r < count; r += 64) {
                if (r + lane < count) {
                    char* slot = slots + list[r + lane];
                    *reinterpret_cast<double*>(slot) = moro_tail_fma(
                        *reinterpret_cast<const uint32_t*>(slot));
                }
            }
            wave_lds_order();
            const double* __restrict__ g = G + j0 * W;
#pragma unroll 2
            for (int j = 0; j < nj; ++j, g += W) {
                const double z = *reinterpret_cast<const double*>(mine + j * 512);
#pragma unroll
                for (int c = 0; c < W; ++c) acc[c] = __builtin_fma(g[c], z, acc[c]);
                if (j0 + j < h.df_draws) dfe = __builtin_fma(gdf[j0 + j], z, dfe);
            }
            wave_lds_order();   // the slots are rewritten by the next batch
        }
        double leg = -1.0;
#pragma unroll
        for (int c = 0; c < W; ++c)
            if (c < h.flows) leg = __builtin_fma(pay[c], exp2_mid(acc[c]), leg);
        double v = (leg > 0 ? leg : 0) * (h.df_draws > 0 ? exp2_mid(dfe) : df0);
        v = p0 < grid.paths ? v : 0.0;
        to.add(v);
    });
}

// A block's sums of payoff and payoff^2, in a fixed order (thread 0's to use).
__device__ __forceinline__ void block_sums(double* sum, double* sumsq) {
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) {
        *sum += __shfl_xor(*sum, o, 64);
        *sumsq += __shfl_xor(*sumsq, o, 64);
    }
    __shared__ double lds[2][kSwThreads / 64];
    __syncthreads();   // the last call's reads
    if ((threadIdx.x & 63) == 0) {
        lds[0][threadIdx.x / 64] = *sum;
        lds[1][threadIdx.x / 64] = *sumsq;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        *sum = lds[0][0];
        *sumsq = lds[1][0];
#pragma unroll
        for (int i = 1; i < kSwThreads / 64; ++i) {
            *sum += lds[0][i];
            *sumsq += lds[1][i];
        }
    }
}

// A swaption's mean and standard error (HJM_Swaption_Blocking.cpp:212-218) from
// its units' partials: work-item t takes t, t + 256, ... in order, then a fixed
// tree; thread 0 hands both to put().  lds: 2 kSwThreads doubles.
template <class Load, class Put>
__device__ __forceinline__ void mean_and_error(int units, int64_t trials, double* lds, Load&& load,
                                               Put&& put) {
    double a = 0.0, b = 0.0;
    for (int i = threadIdx.x; i < units; i += kSwThreads) {
        a += load(2 * i);
        b += load(2 * i + 1);
    }
    double* sums = lds;
    double* squares = lds + kSwThreads;
    sums[threadIdx.x] = a;
    squares[threadIdx.x] = b;
    __syncthreads();
    for (int half = kSwThreads / 2; half >= 1; half >>= 1) {
        if ((int)threadIdx.x < half) {
            sums[threadIdx.x] += sums[threadIdx.x + half];
            squares[threadIdx.x] += squares[threadIdx.x + half];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        const double sum = sums[0], sumsq = squares[0];
        put(sum / trials,
            sqrt((sumsq - sum * sum / trials) / (trials - 1.0)) / sqrt((double)trials));
    }
}

// How a launch ends by itself: the last block of a swaption forms its results
// and the last of those tells the host.
struct SwDone {
    uint32_t* counters;   // 64 words apart: the swaptions', then the launch's; NULL:
                          // k_sw_final follows
    double* out;          // pinned
    uint32_t* flag;       // pinned
    uint32_t seq;
    int32_t swaptions;
    int64_t trials;
};

// Ends a block of swaption sw whose unit u (bit u of summed) has its waves' sums
// in sums[wave][u]; mine: the partials from its first unit on, all: from the
// swaption's.  lds: as mean_and_error's, free to overwrite once the block has met.
__device__ __forceinline__ void finish_block(const UnitSums& sums, uint32_t summed, int sw,
                                             const SwLin& h, const SwGrid& grid, double* all,
                                             double* mine, const SwDone& done, double* lds) {
    static_assert(2 * kSwMaxUnits <= 64, "one wave stores a block's partials");
    __shared__ int last;
    __syncthreads();
    if (threadIdx.x < 64) {
        const int u = threadIdx.x / 2, q = threadIdx.x & 1;
        if (u < kSwMaxUnits && (summed >> u & 1)) {
            double v = sums[0][u][q];
#pragma unroll
            for (int w = 1; w < kSwThreads / 64; ++w) v += sums[w][u][q];
            agent_store(mine + 2 * u + q, v);
        }
        if (done.counters) {
            stores_done();
            const bool full = arrive(done.counters + 64 * sw, (uint32_t)grid.bps);
            if (threadIdx.x == 0) last = full;
        }
    }
    if (!done.counters) return;
    __syncthreads();
    if (!last) return;
    mean_and_error(h.units, done.trials, lds, [&](int i) { return agent_load(all + i); },
                   [&](double mean, double error) {
                       system_store(done.out + 2 * sw, mean);
                       system_store(done.out + 2 * sw + 1, error);
                       stores_done();
                       if (arrive_one(done.counters + 64 * done.swaptions,
                                      (uint32_t)done.swaptions))
                           system_store(done.flag, done.seq);
                   });
}

constexpr int kSwBatch = 12;     // draws of a work-item in one batch of the narrow form
constexpr int kNarrowFlows = 4;   // cash flows it takes

// Widths of the linear form's accumulators: the smallest that holds the cash
// flows.  A launch's kernel holds the forms up to the widest of its swaptions
// and each block takes its swaption's own.
constexpr int kLinWidths[] = {1, 2, 3, 4, 6, 8, 12, 16, 24, 32, 48, 64};
constexpr int lin_width(int flows) {
    for (int w : kLinWidths)
        if (flows <= w) return w;
    return 0;
}

// Few draws and cash flows (the reference driver's swaptions have 3 or 6 and 1
// to 3): several paths at a time in registers.  Otherwise the wide form.
template <int W>
__device__ __forceinline__ uint32_t linear_form(const SwLin& h, const double* __restrict__ q,
                                                uint32_t xb, int64_t first, bool whole,
                                                const SwGrid& grid, char* lds,
                                                double (*__restrict__ sums)[2]) {
    if constexpr (W <= kNarrowFlows) {
        const uint32_t wl = (uint32_t)__builtin_amdgcn_readfirstlane(threadIdx.x / 64) *
                            (kSwBatch * 64 * 8);
        if (h.draws <= 3 && grid.rows > 2)   // 12 draws in a batch
            return h.unit == 2
                       ? linear_paths<W, 4, 3, true>(h, q, xb, first, whole, grid, lds, wl, sums)
                       : linear_paths<W, 4, 3, false>(h, q, xb, first, whole, grid, lds, wl, sums);
        if (h.draws <= kSwBatch / 2)
            return linear_paths<W, 2, kSwBatch / 2, false>(h, q, xb, first, whole, grid, lds, wl,
                                                           sums);
    }
    return linear_wide<W>(h, q, xb, first, whole, grid, lds, sums);
}

// Bound by FP64 issue (parameters and partial sums are all it reads and
// writes): PARSEC's native run, 128 swaptions x 1M trials with 3 or 6 draws and
// 1 to 3 cash flows, takes 0.776 ms at 204 VALU instructions per path, and
// took 3.31 ms at 928 in the form that followed the forward-rate chains (a
// 64-bit generator, 6 draws for every swaption, an exponential per curve
// point); 32 swaptions x 50,000 trials with 4-40 draws 0.09 ms and 0.76 ms.
// With 3 waves per SIMD in place of 4 the native run takes 0.79 ms, with 5 the same.
template <int MAXW>
__global__ __launch_bounds__(kSwThreads)
__attribute__((amdgpu_waves_per_eu(MAXW <= 8 ? 4 : MAXW <= 32 ? 3 : 2))) void k_sw_paths(
    const SwLin* __restrict__ heads, const double* __restrict__ pool, SwGrid grid,
    double* partial, SwDone done) {
    __shared__ __align__(8) char lds[kSwThreads / 64 * kWideBytes];
    __shared__ UnitSums unit_sums;
    static_assert(kSwThreads * kSwBatch * 8 <= sizeof lds, "the narrow form's lists");
    const int sw = (int)(blockIdx.x / (unsigned)grid.bps);
    const int64_t chunk = blockIdx.x % (unsigned)grid.bps;
    const SwLin h = heads[sw];
    if (!h.linear) return;
    const double* q = pool + h.off;
    const int64_t first = chunk * (kSwThreads * grid.rows);
    const bool whole = rows_linear(h, first, grid.rows);
    // residue of this work-item's first draw: the block's (uniform) and the
    // work-item's path, A (seed + (first + t) per_path)
    const uint64_t xu = mod_m31(mod_m31((uint64_t)h.seed + (uint64_t)first * h.per_path) * kGenA);
    const uint32_t xb = add_m31((uint32_t)xu, (uint32_t)mod_m31((uint64_t)h.x_path * threadIdx.x));
    double (*sums)[2] = unit_sums[__builtin_amdgcn_readfirstlane(threadIdx.x / 64)];
    uint32_t summed = 0;
    const int W = h.flows;
    if (W <= 1) summed = linear_form<1>(h, q, xb, first, whole, grid, lds, sums);
    if (W == 2) summed = linear_form<2>(h, q, xb, first, whole, grid, lds, sums);
    if constexpr (MAXW >= 4) {
        if (W == 3) summed = linear_form<3>(h, q, xb, first, whole, grid, lds, sums);
        if (W == 4) summed = linear_form<4>(h, q, xb, first, whole, grid, lds, sums);
    }
    if constexpr (MAXW >= 8) {
        if (W > 4 && W <= 6) summed = linear_form<6>(h, q, xb, first, whole, grid, lds, sums);
        if (W > 6 && W <= 8) summed = linear_form<8>(h, q, xb, first, whole, grid, lds, sums);
    }
    if constexpr (MAXW >= 16) {
        if (W > 8 && W <= 12) summed = linear_form<12>(h, q, xb, first, whole, grid, lds, sums);
        if (W > 12 && W <= 16) summed = linear_form<16>(h, q, xb, first, whole, grid, lds, sums);
    }
    if constexpr (MAXW >= 32) {
        if (W > 16 && W <= 24) summed = linear_form<24>(h, q, xb, first, whole, grid, lds, sums);
        if (W > 24 && W <= 32) summed = linear_form<32>(h, q, xb, first, whole, grid, lds, sums);
    }
    if constexpr (MAXW >= 64) {
        if (W > 32 && W <= 48) summed = linear_form<48>(h, q, xb, first, whole, grid, lds, sums);
        if (W > 48) summed = linear_form<64>(h, q, xb, first, whole, grid, lds, sums);
    }
    static_assert(2 * kSwThreads * sizeof(double) <= sizeof lds, "finish_block's sums");
    // finish_block synchronises the block before it overwrites the lists
    double* all = partial + 2 * (int64_t)h.unit0;
    finish_block(unit_sums, summed, sw, h, grid, all, all + 2 * (first / (kSwThreads * h.unit)),
                 done, reinterpret_cast<double*>(lds));
}

// The units that k_sw_paths left out, one path at a time per work-item: block b
// takes the units b % bps, + bps, ... of swaption b / bps.
template <int F, int MAXM>
__global__ __launch_bounds__(kSwThreads) void k_sw_paths_steps(
    const SwLin* __restrict__ lin, const SwHead* __restrict__ heads,
    const double* __restrict__ pool, int64_t paths, int bps, double* __restrict__ partial) {
    const int sw = (int)(blockIdx.x / (unsigned)bps);
    const SwLin x = lin[sw];
#pragma unroll 1
    for (int u = (int)(blockIdx.x % (unsigned)bps); u < x.units; u += bps) {
        const int64_t first = (int64_t)u * (kSwThreads * x.unit);
        if (rows_linear(x, first, x.unit)) continue;
        const SwHead h = heads[sw];
        const double* q = pool + h.off;
        double sum = 0.0, sumsq = 0.0;
#pragma unroll 1
        for (int j = 0; j < x.unit; ++j) {
            const int64_t p = first + j * kSwThreads + threadIdx.x;
            if (p < paths) {
                double z[MAXM][F];
                draws<F, MAXM>(h, p, z);
                const double v = path_payoff<F, MAXM>(h, q, z);
                sum += v;
                sumsq += v * v;
            }
        }
        block_sums(&sum, &sumsq);
        if (threadIdx.x == 0) {
            double* mine = partial + 2 * ((int64_t)x.unit0 + u);
            mine[0] = sum;
            mine[1] = sumsq;
        }
    }
}

// A call's parameters from pinned host memory (16-byte words); counters (64
// words apart) to zero.
__global__ __launch_bounds__(kSwThreads) void k_sw_stage(const uint4* __restrict__ host,
                                                         uint4* __restrict__ dev, int words,
                                                         uint32_t* counters, int ncounters) {
    const int stride = gridDim.x * kSwThreads, first = blockIdx.x * kSwThreads + threadIdx.x;
    for (int i = first; i < words; i += stride) dev[i] = host[i];
    for (int i = first; i < ncounters; i += stride) counters[64 * i] = 0;
}

// Block i forms swaption i's results from its units' partials.
__global__ __launch_bounds__(kSwThreads) void k_sw_final(const SwLin* __restrict__ heads,
                                                         const double* __restrict__ partial,
                                                         int64_t trials,
                                                         double* __restrict__ out) {
    __shared__ double lds[2 * kSwThreads];
    const double* in = partial + 2 * (int64_t)heads[blockIdx.x].unit0;
    mean_and_error(heads[blockIdx.x].units, trials, lds, [&](int i) { return in[i]; },
                   [&](double mean, double error) {
                       out[2 * blockIdx.x] = mean;
                       out[2 * blockIdx.x + 1] = error;
                   });
}

using LaunchLin = void (*)(unsigned, hipStream_t, const SwLin*, const double*, const SwGrid&,
                           double*, const SwDone&);
template <int MAXW>
void launch_linear(unsigned blocks, hipStream_t st, const SwLin* heads, const double* pool,
                   const SwGrid& grid, double* partial, const SwDone& done) {
    hipLaunchKernelGGL((k_sw_paths<MAXW>), dim3(blocks), dim3(kSwThreads), 0, st, heads, pool,
                       grid, partial, done);
}
LaunchLin linear_kernel(int flows) {
    return flows <= 2    ? launch_linear<2>
           : flows <= 4  ? launch_linear<4>
           : flows <= 8  ? launch_linear<8>
           : flows <= 16 ? launch_linear<16>
           : flows <= 32 ? launch_linear<32>
                         : launch_linear<64>;
}

// What the step-by-step kernel covers.  Its form goes by the latest start of the
// swaptions: up to 2, 4 or (4 factors at most) 8 steps the draws stay in registers
// (56-116 VGPRs), beyond they live in scratch.  32 swaptions x 50,000 trials whose
// rates are past the linear form's bound, us a call with the registers' form and
// with the scratch's throughout: 3 factors, starts at steps 1-2 124 and 156; 4
// factors, 1-4 243 and 438, 1-8 344 and 621; 1-10 (scratch) 672.  A linear
// portfolio with a zero draw in one unit of each swaption, 128 x 1M: 867, and 769
// without.
struct SwSteps {
    int64_t paths;
    int start, units;   // the latest start and the most units of the swaptions
};
template <int F, int MAXM>
void launch_steps_of(unsigned n, hipStream_t st, const SwLin* lin, const SwHead* heads,
                     const double* pool, const SwSteps& x, double* partial) {
    // a launch holds fewer than 2^32 work-items
    const unsigned bps = std::min<unsigned>(x.units, std::max(1u, 0xffffffffu / kSwThreads / n));
    hipLaunchKernelGGL((k_sw_paths_steps<F, MAXM>), dim3(n * bps), dim3(kSwThreads), 0, st, lin,
                       heads, pool, x.paths, (int)bps, partial);
}
template <int F>
void launch_steps(unsigned n, hipStream_t st, const SwLin* lin, const SwHead* heads,
                  const double* pool, const SwSteps& x, double* partial) {
    if (x.start <= 2) return launch_steps_of<F, 2>(n, st, lin, heads, pool, x, partial);
    if (x.start <= 4) return launch_steps_of<F, 4>(n, st, lin, heads, pool, x, partial);
    if constexpr (F <= 4)
        if (x.start <= 8) return launch_steps_of<F, 8>(n, st, lin, heads, pool, x, partial);
    launch_steps_of<F, kSwMaxDraws / F>(n, st, lin, heads, pool, x, partial);
}
using LaunchSteps = void (*)(unsigned, hipStream_t, const SwLin*, const SwHead*, const double*,
                             const SwSteps&, double*);
constexpr LaunchSteps kStepsByFactors[kSwMaxFactors] = {
    launch_steps<1>, launch_steps<2>, launch_steps<3>, launch_steps<4>,
    launch_steps<5>, launch_steps<6>, launch_steps<7>, launch_steps<8>};

bool finite_all(const bs_swaption_t& s) {
    return std::isfinite(s.strike) && std::isfinite(s.compounding) && std::isfinite(s.maturity) &&
           std::isfinite(s.tenor) && std::isfinite(s.payment_interval) && std::isfinite(s.years);
}

// (int)(x + 0.5) as the reference rounds, or INT32_MIN when x is out of range.
int round_index(double x) {
    const double y = x + 0.5;
    return (y > -1e9 && y < 1e9) ? (int)y : INT32_MIN;
}

// Index sizes of a swaption (HJM_Swaption_Blocking.cpp:48-70).
struct SwShape {
    double dt;
    int m, L, freq, points;
    int unit;
};

// Validates swaption i of `paths` paths.
int shape_of(const bs_swaption_t& s, int64_t i, int64_t paths, SwShape* x) {
    const int n = s.n_steps, F = s.n_factors;
    char msg[160];
    auto bad = [&](const char* why) {
        snprintf(msg, sizeof msg, "swaption %lld: %s", (long long)i, why);
        return set_error(BS_ERR_INVALID, msg);
    };
    if (n < 2 || n > kSwMaxSteps) return bad("n_steps must be in [2, 64]");
    if (F < 1 || F > kSwMaxFactors) return bad("n_factors must be in [1, 8]");
    if (!s.yield || !s.factors) return bad("NULL yield or factors");
    if (!finite_all(s) || !(s.years > 0)) return bad("non-finite parameter or years <= 0");
    const double dt = (double)(s.years / n);
    const int freq = round_index(s.payment_interval / dt);
    const int L = round_index(n - s.maturity / dt);
    const int m = round_index(s.maturity / dt);
    const int points = round_index(s.tenor / dt);
    if (freq < 1) return bad("payment interval rounds to less than one step");
    if (m < 0 || m >= n) return bad("maturity outside the simulated horizon");
    if (L < 1 || points < 0 || points > L - 1) return bad("swap tenor outside the horizon");
    if (m * F > kSwMaxDraws) return bad("start step x n_factors exceeds 64");
    const bool narrow = m * F <= kSwBatch / 2 && points / freq <= kNarrowFlows;
    *x = {dt, m, L, freq, points, unit_rows(narrow, paths)};
    return BS_OK;
}

// Appends a swaption's head and data (the per-swaption set-up of
// HJM_Swaption_Blocking.cpp:48-150 and HJM.cpp's forward curve and drifts, in
// host FP64 without contraction, as the reference computes them).
void pack_swaption(const bs_swaption_t& s, const SwShape& x, int64_t seed, SwHead* h,
                   std::vector<double>* pool) {
    const int n = s.n_steps, F = s.n_factors, m = x.m, L = x.L, freq = x.freq, points = x.points;
    const double dt = x.dt;
    const double strike_cont = s.compounding == 0
                                   ? s.strike
                                   : (1 / s.compounding) * log(1 + s.strike * s.compounding);
    const int w = n - 1;
    h->seed = seed;
    h->dt = dt;
    h->sdt = sqrt(dt);
    h->dts = (double)((double)(L * dt) / L);
    h->n = n;
    h->m = m;
    h->L = L;
    h->off = (int32_t)pool->size();
    const size_t base = pool->size();
    pool->resize(base + n + w + (size_t)F * w + L, 0.0);
    double* f0 = pool->data() + base;
    double* mudt = f0 + n;
    double* sig = mudt + w;
    double* pay = sig + (size_t)F * w;
    // forward curve from the yield curve
    f0[0] = s.yield[0];
    for (int j = 1; j < n; ++j) f0[j] = (j + 1) * s.yield[j] - j * s.yield[j - 1];
    // drifts: sum_{l<=j} mu_k[l] = dt/2 (sum_{l<=j} sigma_k[l])^2, then the total;
    // the running sums d and vol add in the order of the reference's own loops
    double drift[kSwMaxFactors][kSwMaxSteps];
    for (int k = 0; k < F; ++k) {
        const double* fk = s.factors + (size_t)k * w;
        double* dk = drift[k];
        dk[0] = 0.5 * dt * fk[0] * fk[0];
        double d = 0, vol = 0 + fk[0];
        for (int j = 1; j < w; ++j) {
            d -= dk[j - 1];
            vol += fk[j];
            dk[j] = d + 0.5 * dt * vol * vol;
        }
        for (int l = 0; l < w; ++l) sig[(size_t)k * w + l] = fk[l];
    }
    for (int l = 0; l < w; ++l) {
        double t = 0;
        for (int k = 0; k < F; ++k) t += drift[k][l];
        mudt[l] = t * dt;
    }
    for (int l = 0; l < L; ++l) pay[l] = 0.0;
    const double grow = exp(strike_cont * s.payment_interval);
    for (int l = freq; l <= points; l += freq) pay[l] = l != points ? grow - 1 : grow;
}

// Appends the linear form of the swaption that pack_swaption packed at h:
// every exponent of its payoff, in base 2, as a constant and one coefficient
// per draw.
// It holds if the running products of discount factors that the reference
// forms stay far from overflow and underflow: with every finite draw below 7
// in size (Moro at u = 4.66e-10 is 6.2), the rates times their times sum to at
// most 400 in base 2 over the whole curve, so every product is within 2^+-400.
// (Their terms are then finite too, and the factors past the last cash flow,
// which the reference multiplies by zero, contribute +0.)
void pack_linear(const SwHead& h, int F, int freq, int points, SwLin* x,
                 std::vector<double>* pool) {
    const int n = h.n, m = h.m, w = n - 1, D = m * F;
    x->seed = h.seed;
    x->per_path = (uint32_t)(w * F);
    x->x_path = gen_step(x->per_path);
    x->x_row = gen_step((uint64_t)kSwThreads * x->per_path);
    x->draws = D;
    x->df_draws = m > 0 ? (m - 1) * F : 0;
    x->flows = points / freq;
    const int W = lin_width(x->flows);
    pool->resize((pool->size() + 7) & ~(size_t)7);   // scalar loads of whole lines
    x->off = (int32_t)pool->size();
    const size_t base = pool->size(), old = (size_t)h.off;
    pool->resize(base + 2 * W + (size_t)D * W + D, 0.0);
    const double* f0 = pool->data() + old;
    const double* mudt = f0 + n;
    const double* sig = mudt + w;
    const double* cash = sig + (size_t)F * w;
    double* C = pool->data() + base;
    double* pay = C + W;
    double* G = pay + W;
    double* gdf = G + (size_t)D * W;
    constexpr long double kLog2eL = 1.442695040888963407359924681001892137L;
    // sqrt(dt) sigma log2 e per rate step and factor, and their sizes
    double g[kSwMaxSteps * kSwMaxFactors], size_of[kSwMaxSteps];
    for (int l = 0; l < w; ++l) {
        size_of[l] = 0.0;
        for (int k = 0; k < F; ++k) {
            g[l * F + k] = (double)(h.sdt * kLog2eL * sig[(size_t)k * w + l]);
            size_of[l] += std::fabs(g[l * F + k]);
        }
    }
    long double base_sum = 0.0L;   // the running exponent: its constant,
    double sum[kSwMaxDraws] = {};  // and per draw, both before the factor -t
    double size = 0.0;             // bound on the sum of |rate| x time, in base 2
    int c = 0;
    for (int d = 0; d < n; ++d) {
        if (d == m) {   // the discount to the start is complete
            x->c_df = (double)(-h.dt * base_sum);
            for (int j = 0; j < D; ++j) gdf[j] = -h.dt * sum[j];
            base_sum = 0.0L;
            std::fill(sum, sum + D, 0.0);
        }
        const int steps = std::min(d, m);
        long double rate = f0[d];
        double shocks = 0.0;
        for (int s = 1; s <= steps; ++s) {
            const int l = d - s;
            rate += mudt[l];
            shocks += size_of[l];
            for (int k = 0; k < F; ++k) sum[(s - 1) * F + k] += g[l * F + k];
        }
        base_sum += kLog2eL * rate;
        size += (d < m ? h.dt : h.dts) * (1.4427 * std::fabs((double)rate) + 7.0 * shocks);
        const int l = d - m + 1;   // the swap curve's point whose discount this completes
        if (d >= m && l <= points && l % freq == 0) {
            C[c] = (double)(-h.dts * base_sum);
            pay[c] = cash[l];
            for (int j = 0; j < D; ++j) G[(size_t)j * W + c] = -h.dts * sum[j];
            ++c;
        }
    }
    for (; c < x->flows; ++c) {   // cash flows past the simulated curve: zero rates there
        C[c] = (double)(-h.dts * base_sum);
        pay[c] = cash[(c + 1) * freq];
        for (int j = 0; j < D; ++j) G[(size_t)j * W + c] = -h.dts * sum[j];
    }
    x->linear = size <= 400.0 ? 1 : 0;   // false for NaN
}

// Whether counters [c, c + count) hold a multiple of 2^31-1.
bool draws_zero(int64_t c, int64_t count) {
    const int64_t m = (int64_t)kM31;
    return c % m == 0 || c / m != (c + count - 1) / m;
}

// A call's buffers.  Most calls take one of up to kSwSpaces workspaces that the
// library keeps per device, given back after the call's stream has been
// synchronised: pinned memory, from which a kernel fetches the parameters and
// into which the last kernel writes the results, and device memory for the
// parameters and partial sums.  Stream-ordered allocation (22 us with its
// free), a pageable upload (14 us) and a pageable download (20 us) cost more
// than the kernels of a small call: 64 swaptions x 20,000 trials take 42 us
// and took 91.
constexpr int kSwDevices = 64;
constexpr int kSwSpaces = 4;
constexpr size_t kSpaceHost = size_t(1) << 20, kSpaceDev = size_t(16) << 20;
constexpr size_t kSpaceFlag = 64;   // the end of the pinned memory

// Launches that end by themselves (SwDone) save k_sw_final and the stream's
// synchronisation, 4 to 6 us a call (1 x 1000 trials 23.3 and 17.7 us, 32 x 50,000
// 125 and 119, 128 x 300,000, 4736 blocks, 272 and 268), but every block then
// waits for its partials' acknowledgement, which over many rounds costs as much
// (128 x 550,000, 8704 blocks, 453 and 448 us, 128 x 1M, 15,744 blocks, 775 both).
constexpr size_t kSwSelfMax = 512;
constexpr int64_t kSwSelfBlocks = 8192;

struct SwSpace {
    char* host = nullptr;       // pinned
    char* host_dev = nullptr;   // the same memory, device address
    char* dev = nullptr;        // kSpaceDev bytes, then the counters
    uint32_t seq = 0;           // of the last launch that ended by itself
};

// Spins until that launch has ended, for at most `us` microseconds.
bool spin_for(const SwSpace& x, int64_t us) {
    const uint32_t* flag = reinterpret_cast<const uint32_t*>(x.host + kSpaceHost - kSpaceFlag);
    const auto until = std::chrono::steady_clock::now() + std::chrono::microseconds(us);
    while (__atomic_load_n(flag, __ATOMIC_ACQUIRE) != x.seq) {
        if (std::chrono::steady_clock::now() >= until) return false;
        __builtin_ia32_pause();
    }
    return true;
}

struct SwSpaces {
    std::mutex mu;
    std::vector<SwSpace> idle;   // room for all of them is reserved before the first
    int made = 0;
};

SwSpaces& spaces_of(int dev) {
    static SwSpaces* s = new SwSpaces[kSwDevices];   // lives until the process ends
    return s[dev];
}

// Takes an idle workspace or makes one; false when all are in use or there is
// no memory for another.
bool take_space(int dev, SwSpace* x) {
    if (dev < 0 || dev >= kSwDevices) return false;
    SwSpaces& all = spaces_of(dev);
    std::lock_guard<std::mutex> lk(all.mu);
    all.idle.reserve(kSwSpaces);
    if (!all.idle.empty()) {
        *x = all.idle.back();
        all.idle.pop_back();
        return true;
    }
    if (all.made == kSwSpaces) return false;
    const RelaxedCapture relaxed;
    void* p = nullptr;
    if (hipHostMalloc(reinterpret_cast<void**>(&x->host), kSpaceHost, hipHostMallocCoherent) !=
        hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    if (hipHostGetDevicePointer(&p, x->host, 0) != hipSuccess ||
        hipMalloc(reinterpret_cast<void**>(&x->dev), kSpaceDev + (kSwSelfMax + 1) * 256) !=
            hipSuccess) {
        (void)hipGetLastError();
        (void)hipHostFree(x->host);
        return false;
    }
    memset(x->host + kSpaceHost - kSpaceFlag, 0, kSpaceFlag);
    x->seq = 0;
    x->host_dev = static_cast<char*>(p);
    ++all.made;
    return true;
}

void give_space(int dev, const SwSpace& x) {
    SwSpaces& all = spaces_of(dev);
    std::lock_guard<std::mutex> lk(all.mu);
    all.idle.push_back(x);
}

// Calls that no workspace holds allocate from one stream-ordered pool per
// device that keeps freed memory up to 1 GiB: they end with a stream
// synchronisation, at which the default pool would hand its memory back to the
// device and the next call would allocate anew.

hipError_t pool_of(int dev, hipMemPool_t* out) {
    static std::mutex mu;
    static hipMemPool_t pools[kSwDevices] = {};
    if (dev < 0 || dev >= kSwDevices) return hipErrorInvalidDevice;
    std::lock_guard<std::mutex> lk(mu);
    if (!pools[dev]) {
        const RelaxedCapture relaxed;
        hipMemPoolProps props = {};
        props.allocType = hipMemAllocationTypePinned;
        props.location.type = hipMemLocationTypeDevice;
        props.location.id = dev;
        hipMemPool_t p = nullptr;
        hipError_t e = hipMemPoolCreate(&p, &props);
        if (e != hipSuccess) return e;
        uint64_t keep = uint64_t(1) << 30;
        e = hipMemPoolSetAttribute(p, hipMemPoolAttrReleaseThreshold, &keep);
        if (e != hipSuccess) {
            (void)hipMemPoolDestroy(p);
            return e;
        }
        pools[dev] = p;
    }
    *out = pools[dev];
    return hipSuccess;
}

// Swaptions of one launch.
struct SwBatch {
    std::vector<SwLin> lins;
    std::vector<SwHead> heads;
    std::vector<double> pool;
    std::vector<int32_t> index;   // places in the caller's array
    int flows = 0;
    int32_t units = 0;
    int start = 0, most = 0;      // the latest start and the most units of a swaption
    bool steps = false;           // some unit needs the step-by-step kernel

    void add(const bs_swaption_t& s, const SwShape& x, int64_t seed, int32_t i, int64_t paths) {
        heads.emplace_back();
        lins.emplace_back();
        index.push_back(i);
        pack_swaption(s, x, seed, &heads.back(), &pool);
        pack_linear(heads.back(), s.n_factors, x.freq, x.points, &lins.back(), &pool);
        SwLin& l = lins.back();
        flows = std::max(flows, l.flows);
        // swaptions that the step-by-step kernel prices whole: units of 2 rows
        l.unit = l.linear ? x.unit : unit_rows(false, paths);
        l.units = (int32_t)((paths + kSwThreads * l.unit - 1) / (kSwThreads * l.unit));
        l.unit0 = units;
        units += l.units;
        start = std::max(start, x.m);
        most = std::max(most, l.units);
        steps = steps || !l.linear ||
                draws_zero(seed, (int64_t)l.units * kSwThreads * l.unit * l.per_path);
    }
};

// The places of a call's parts: heads of both kernels | pool | partials.
struct SwLayout {
    size_t heads, pool, partial, bytes;   // offsets of the step-by-step heads, pool and
                                          // partials, and what all of it takes
    explicit SwLayout(const SwBatch& b) {
        auto up = [](size_t n) { return (n + 255) & ~(size_t)255; };
        heads = up(b.lins.size() * sizeof(SwLin));
        pool = heads + up(b.heads.size() * sizeof(SwHead));
        partial = pool + up(b.pool.size() * sizeof(double));
        bytes = partial + (size_t)b.units * 2 * sizeof(double);
    }
    // Writes the parameters (everything before the partials), laid out as on the device.
    void write(const SwBatch& b, char* to) const {
        memcpy(to, b.lins.data(), b.lins.size() * sizeof(SwLin));
        memcpy(to + heads, b.heads.data(), b.heads.size() * sizeof(SwHead));
        memcpy(to + pool, b.pool.data(), b.pool.size() * sizeof(double));
    }
};

// The kernels of a launch whose parameters are on the device at base; k_sw_final
// only without done.counters.
hipError_t launch_batch(const SwBatch& b, const SwLayout& at, int F, const SwGrid& grid,
                        int64_t trials, char* base, double* out, const SwDone& done,
                        hipStream_t st) {
    const unsigned n = (unsigned)b.lins.size();
    const unsigned blocks = (unsigned)grid.bps * n;
    const SwLin* dl = reinterpret_cast<const SwLin*>(base);
    const SwHead* dh = reinterpret_cast<const SwHead*>(base + at.heads);
    const double* dp = reinterpret_cast<const double*>(base + at.pool);
    double* dq = reinterpret_cast<double*>(base + at.partial);
    linear_kernel(b.flows)(blocks, st, dl, dp, grid, dq, done);
    if (b.steps)
        kStepsByFactors[F - 1](n, st, dl, dh, dp, {grid.paths, b.start, b.most}, dq);
    if (!done.counters)
        hipLaunchKernelGGL(k_sw_final, dim3(n), dim3(kSwThreads), 0, st, dl, dq, trials, out);
    return hipGetLastError();
}

int price_batch(const SwBatch& b, int F, const SwGrid& grid, int64_t trials, double* price,
                double* std_error, hipStream_t st) {
    const size_t n = b.lins.size();
    const SwLayout at(b);
    const size_t ob = n * 2 * sizeof(double);
    auto deliver = [&](const double* out) {
        for (size_t k = 0; k < n; ++k) {
            price[b.index[k]] = out[2 * k];
            std_error[b.index[k]] = out[2 * k + 1];
        }
        return BS_OK;
    };
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return hip_error(e, "hipGetDevice");
    SwSpace space;
    if (at.partial + ob <= kSpaceHost - kSpaceFlag && at.bytes <= kSpaceDev &&
        take_space(dev, &space)) {
        at.write(b, space.host);
        double* out = reinterpret_cast<double*>(space.host_dev + at.partial);
        const bool self = n <= kSwSelfMax && (int64_t)grid.bps * (int64_t)n <= kSwSelfBlocks &&
                          !b.steps;   // (blocks left out count in nowhere)
        SwDone done = {};
        if (self)
            done = {reinterpret_cast<uint32_t*>(space.dev + kSpaceDev), out,
                    reinterpret_cast<uint32_t*>(space.host_dev + kSpaceHost - kSpaceFlag),
                    ++space.seq, (int32_t)n, trials};
        const int words = (int)(at.partial / sizeof(uint4));
        hipLaunchKernelGGL(k_sw_stage, dim3(std::min((words + kSwThreads - 1) / kSwThreads, 64)),
                           dim3(kSwThreads), 0, st, reinterpret_cast<const uint4*>(space.host_dev),
                           reinterpret_cast<uint4*>(space.dev), words, done.counters,
                           self ? (int)n + 1 : 0);
        e = hipGetLastError();
        if (e == hipSuccess)
            e = launch_batch(b, at, F, grid, trials, space.dev, out, done, st);
        hipError_t es = hipSuccess;
        if (!self || e != hipSuccess || !spin_for(space, 500))
            es = hipStreamSynchronize(st);
        if (e == hipSuccess && es == hipSuccess)
            deliver(reinterpret_cast<const double*>(space.host + at.partial));
        if (es == hipSuccess) give_space(dev, space);   // else its work may still run
        if (e != hipSuccess) return hip_error(e, "bs_swaptions_host_f64");
        return es == hipSuccess ? BS_OK : hip_error(es, "hipStreamSynchronize");
    }
    hipMemPool_t mem = nullptr;
    e = pool_of(dev, &mem);
    if (e != hipSuccess) return hip_error(e, "hipMemPoolCreate");
    std::vector<double> out(n * 2);
    std::vector<char> staged(at.partial);
    at.write(b, staged.data());
    char* base = nullptr;
    const size_t results = (at.bytes + 255) & ~(size_t)255;
    e = hipMallocFromPoolAsync(reinterpret_cast<void**>(&base), results + ob, mem, st);
    if (e != hipSuccess) return hip_error(e, "hipMallocFromPoolAsync");
    double* dout = reinterpret_cast<double*>(base + results);
    e = hipMemcpyAsync(base, staged.data(), staged.size(), hipMemcpyHostToDevice, st);
    if (e == hipSuccess) e = launch_batch(b, at, F, grid, trials, base, dout, SwDone{}, st);
    if (e == hipSuccess) e = hipMemcpyAsync(out.data(), dout, ob, hipMemcpyDeviceToHost, st);
    const hipError_t ef = hipFreeAsync(base, st);
    const hipError_t es = hipStreamSynchronize(st);
    if (e != hipSuccess) return hip_error(e, "bs_swaptions_host_f64");
    if (ef != hipSuccess) return hip_error(ef, "hipFreeAsync");
    if (es != hipSuccess) return hip_error(es, "hipStreamSynchronize");
    return deliver(out.data());
}

}  // namespace
}  // namespace bs

using namespace bs;

extern "C" int bs_swaptions_host_f64(const bs_swaption_t* sw, int64_t n, int64_t trials,
                                     int64_t seed, int32_t block_size, double* price,
                                     double* std_error, bs_stream_t stream) {
    return guarded("bs_swaptions_host_f64", [&]() -> int {
        if (n < 0) return set_error(BS_ERR_INVALID, "n < 0");
        if (n == 0) return BS_OK;
        if (!sw || !price || !std_error) return set_error(BS_ERR_INVALID, "NULL array");
        if (n > (1 << 20)) return set_error(BS_ERR_INVALID, "more than 2^20 swaptions");
        if (trials < 1 || trials > (int64_t(1) << 40))
            return set_error(BS_ERR_INVALID, "trials must be in [1, 2^40]");
        if (block_size < 1) return set_error(BS_ERR_INVALID, "block_size < 1");
        if (seed < 0 || seed >= kSwCounterLimit)
            return set_error(BS_ERR_INVALID, "seed must be in [0, 2^42)");
        const int F = sw[0].n_factors;
        const int64_t paths = (trials + block_size - 1) / block_size * block_size;
        std::vector<SwShape> shapes((size_t)n);
        for (int64_t i = 0; i < n; ++i) {
            if (sw[i].n_factors != F)
                return set_error(BS_ERR_INVALID, "every swaption must have the same n_factors");
            const int rc = shape_of(sw[i], i, paths, &shapes[(size_t)i]);
            if (rc) return rc;
            const int64_t draws = (int64_t)(sw[i].n_steps - 1) * F;
            if (paths > (kSwCounterLimit - (seed + i)) / draws)
                return set_error(BS_ERR_INVALID, "seed + paths x draws exceeds 2^42");
        }
        // A synchronous call waits for its results, which recorded kernels never
        // write: a workspace taken for them would be lost.
        if (capturing(static_cast<hipStream_t>(stream)))
            return hip_error(hipErrorStreamCaptureUnsupported, "bs_swaptions_host_f64");
        // one launch of at most 2^32 work-items: 2^24 blocks of 1024 paths
        const int64_t bps_most = (paths + kSwThreads * kSwRows - 1) / (kSwThreads * kSwRows);
        if (bps_most * n > (int64_t(1) << 24))
            return set_error(BS_ERR_INVALID,
                             "more than 2^24 blocks of 1024 paths (2^34 paths) in one call");
        // Paths per work-item: enough of them to spread the 100 or so
        // instructions of its set-up and its units' sums while several rounds of
        // blocks are left (1024 are resident at once), and 2 where 4 would leave
        // the chip idle.  us a call with rows 2, 4, 8, 16 and 32, swaptions of the
        // driver: 16 x 10,000 (160 blocks of 4 rows) 24.0, 25.5, 30.0, 39, 57; 64 x
        // 20,000 (1280) 44.9, 41.9, 42.8, 49, 68; 128 x 50,000 (6272) 110, 88.7,
        // 85.0, 86.8, 98; 128 x 131,000 (16,384) 210, 162, 150, 144.5, 148; 128 x
        // 300,000 (37,504) -, -, 287, 275, 274; 128 x 1M (125,056) -, -, 823, 783,
        // 774.  Of a desk with starts at steps 1-10 and 4 factors: 8 x 50,000 (392)
        // 44.8, 60.5, 95.7, 165, 300; 32 x 50,000 (1568) 118.9, 119.1, 132, 224, 411.
        const int64_t blocks4 = bps_most * n;
        int rows = blocks4 >= 32768   ? 32
                   : blocks4 >= 12288 ? 16
                   : blocks4 >= 4096  ? 8
                   : blocks4 >= 1024  ? 4
                                      : 2;
        for (const SwShape& x : shapes) rows = std::max(rows, x.unit);
        const int64_t bps = (paths + kSwThreads * rows - 1) / (kSwThreads * rows);
        // the swaptions whose paths cost most first, so that the launch ends on
        // its cheapest blocks
        std::vector<int32_t> order((size_t)n), cost((size_t)n);
        bool even = true;
        for (int64_t i = 0; i < n; ++i) {
            const SwShape& x = shapes[(size_t)i];
            const int W = lin_width(x.points / x.freq);
            order[(size_t)i] = (int32_t)i;
            cost[(size_t)i] = x.m * F * (45 + W) + 20 * W;
            even = even && cost[(size_t)i] == cost[0];
        }
        if (!even)
            std::stable_sort(order.begin(), order.end(), [&](int32_t a, int32_t b) {
                return cost[(size_t)a] > cost[(size_t)b];
            });
        // parameters of more than 2^24 doubles go in several launches
        for (size_t first = 0; first < (size_t)n;) {
            SwBatch batch;
            for (; first < (size_t)n && batch.pool.size() < (size_t(1) << 24); ++first) {
                const int32_t i = order[first];
                batch.add(sw[i], shapes[(size_t)i], seed + i, i, paths);
            }
            const int rc = price_batch(batch, F, {paths, (int32_t)bps, rows}, trials, price,
                                       std_error, static_cast<hipStream_t>(stream));
            if (rc) return rc;
        }
        return BS_OK;
    });
}
