// bs_kernels.hip -- gfx950 streaming kernels of the Black-Scholes map.
//
// Layout in HBM: structure of arrays, one array per field (s, k, r, v, t as
// float or double, the option type as one byte).  A work-item handles a group
// of VW consecutive options: one VW*4-byte load per float array, one VW-byte
// load of the type bytes and one store per output array, so every wave64
// instruction moves a contiguous 64*VW*4-byte span (fully coalesced).  VW is 4
// (128-bit accesses) or 2 (64-bit): 2 for the prices, for the Greeks below 2^22
// options, 4 from there and for CNDF.  Groups are walked grid-stride, optionally
// software-pipelined (the next group's loads issued before the current group's
// math).  Every byte is touched once: loads of aligned streams are non-temporal,
// those of unaligned ones go through the caches, and stores have the policy that
// bs_ops.hpp gives their size.
//
// The pricing arithmetic lives in bs_math.hpp; this file only moves data.
#include <algorithm>

#include "bs_internal.hpp"
#include "bs_math.hpp"
#include "bs_ops.hpp"

namespace bs {
namespace {

// ---- argument packs ------------------------------------------------------------
struct PriceArgs {
    SoaIn<float> in;
    const uint8_t* type;
    float* out;
};
struct PriceI32Args {
    SoaIn<float> in;
    const int32_t* type;
    float* out;
};
struct PriceF64Args {
    SoaIn<double> in;
    const uint8_t* type;
    double* out;
};
struct GreeksArgs {
    SoaIn<float> in;
    const uint8_t* type;
    GreeksOut out;
};
template <class T>
struct CndfArgs {
    const T* x;
    T* out;
};

template <class T>
SoaIn<T> from(const SoaIn<T>& a, int64_t h) {
    return {a.s + h, a.k + h, a.r + h, a.v + h, a.t + h};
}
template <class A>   // the three price packs
A from(const A& a, int64_t h) {
    return {from(a.in, h), a.type + h, a.out + h};
}
GreeksArgs from(const GreeksArgs& a, int64_t h) {
    return {from(a.in, h), a.type + h,
            {a.out.price + h, a.out.delta + h, a.out.vega + h, a.out.rho + h, a.out.theta + h}};
}
template <class T>
CndfArgs<T> from(const CndfArgs<T>& a, int64_t h) {
    return {a.x + h, a.out + h};
}

// Calls f(array) for every array of a call, an output first.
template <class T, class F>
void each(const SoaIn<T>& a, F&& f) {
    f(a.s), f(a.k), f(a.r), f(a.v), f(a.t);
}
template <class A, class F>
void each(const A& a, F&& f) {
    f(a.out), each(a.in, f), f(a.type);
}
template <class F>
void each(const GreeksArgs& a, F&& f) {
    f(a.out.price), f(a.out.delta), f(a.out.vega), f(a.out.rho), f(a.out.theta);
    each(a.in, f), f(a.type);
}
template <class T, class F>
void each(const CndfArgs<T>& a, F&& f) {
    f(a.out), f(a.x);
}

template <class Op, class A>
Op make_op(const A& a) { return Op{a.in, a.type, a.out}; }
template <class Op, class T>
Op make_op(const CndfArgs<T>& a) { return Op{a.x, a.out}; }

// ---- generic streaming kernels ----------------------------------------------
// Grid-stride over the whole groups of VW options in the n from the op's arrays
// on; the `head` options before them and the last n % VW, which do not fill a
// group, are priced one per work-item by the first blocks.  PIPE
// issues the loads of a work-item's next group before pricing the current one
// (register double buffering), so a wave overlaps its own HBM latency with its
// arithmetic; it holds one more group of registers, so its occupancy target
// is two waves lower.  Ix is the group index type: uint32_t when every array
// spans less than 4 GiB (32-bit offsets on the arrays' SGPR bases; fewer than
// 2^30 groups there, so g + stride cannot wrap), int64_t otherwise.
template <class Op, bool NT, bool PIPE, class Ix>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(waves_for<Op, PIPE>())))
void k_stream(Op op, int64_t n, int head) {
    constexpr int VW = Op::kVW;
    const Ix stride = (Ix)gridDim.x * blockDim.x;
    const Ix gid = (Ix)blockIdx.x * blockDim.x + threadIdx.x;
    const Ix ng = (Ix)n / VW;
    Ix g = gid;
    if constexpr (PIPE) {
        if (g < ng) {
            typename Op::Group cur = op.template load<NT>(g);
            for (Ix gn = g + stride; gn < ng; gn += stride) {
                const typename Op::Group nxt = op.template load<NT>(gn);
                op.template finish<NT>(g, cur);
                cur = nxt;
                g = gn;
            }
            op.template finish<NT>(g, cur);
        }
    } else {
        for (; g < ng; g += stride) {
            const typename Op::Group x = op.template load<NT>(g);
            op.template finish<NT>(g, x);
        }
    }
    const int rest = (int)((Ix)n % VW);
    if ((int64_t)gid < head + rest)
        op.scalar((int64_t)gid < head ? (int64_t)gid - head : n - rest + ((int64_t)gid - head));
}

// Blocks of a grid-stride kernel; a launch holds fewer than 2^32 work-items.
inline unsigned grid_for(int64_t work_items, int64_t cap, int threads = kThreads) {
    int64_t blocks = (work_items + threads - 1) / threads;
    if (cap > 0 && blocks > cap) blocks = cap;
    blocks = std::min<int64_t>(blocks, 0xffffffff / threads);
    return (unsigned)(blocks < 1 ? 1 : blocks);
}

template <class Op, bool NT, bool PIPE>
hipError_t launch_form(const Op& op, int64_t n, int head, hipStream_t st) {
    constexpr int VW = Op::kVW;
    const int64_t mb = config().max_blocks.load(std::memory_order_relaxed);
    const int bt = config().block_threads.load(std::memory_order_relaxed);
    const int64_t cap = mb > 0 ? mb : Op::kBlocks;
    const int nt = bt > 0 ? bt : Op::kThreadsPref;
    const unsigned grid = grid_for(std::max<int64_t>(n / VW, head + VW), cap, nt);
    // LDS reserved per block caps the waves resident on a CU (none is used)
    const int lw = config().lds_per_wave.load(std::memory_order_relaxed);
    const size_t lds = std::min<size_t>(
        (size_t)(lw < 0 ? Op::kLdsPerWave : lw) * (size_t)((nt + 63) / 64), 65536);
    if (n < (int64_t(1) << 32) / Op::kElemBytes)
        hipLaunchKernelGGL((k_stream<Op, NT, PIPE, uint32_t>), dim3(grid), dim3(nt), lds, st, op,
                           n, head);
    else
        hipLaunchKernelGGL((k_stream<Op, NT, PIPE, int64_t>), dim3(grid), dim3(nt), lds, st, op,
                           n, head);
    return hipGetLastError();
}

template <class Op>
hipError_t launch_op(const Op& op, int64_t n, int head, hipStream_t st) {
    const bool nt = config().nontemporal.load(std::memory_order_relaxed) != 0;
    const int pl = config().pipeline.load(std::memory_order_relaxed);
    const bool pipe = pl < 0 ? Op::kPipe : pl != 0;
    if (pipe)
        return nt ? launch_form<Op, true, true>(op, n, head, st)
                  : launch_form<Op, false, true>(op, n, head, st);
    return nt ? launch_form<Op, true, false>(op, n, head, st)
              : launch_form<Op, false, false>(op, n, head, st);
}

template <class T>
uintptr_t address(const T* p) { return reinterpret_cast<uintptr_t>(p); }

// Elements to leave before the first group so that the arrays start on
// 128-byte lines: those up to the first output's next line.  *aligned: every
// array's groups of vw elements are then aligned to their size.
template <class Args>
int head_for(const Args& a, int64_t n, int vw, bool* aligned) {
    uintptr_t low = 0;
    each(a, [&](auto* p) { low |= address(p); });
    if (low % 128 == 0) {   // whole arrays from the allocator: nothing to align
        *aligned = true;
        return 0;
    }
    int64_t head = -1;
    bool as_is = true;
    each(a, [&](auto* p) {
        as_is = as_is && address(p) % (sizeof(*p) * vw) == 0;
        if (head < 0)   // the first output
            head = address(p) % sizeof(*p) == 0
                       ? (int64_t)((128 - address(p) % 128) % 128 / sizeof(*p)) : 0;
    });
    head = std::min(head, n);
    bool shifted = true, lines = true;
    each(a, [&](auto* p) {
        const uintptr_t q = address(p + head);
        shifted = shifted && q % (sizeof(*p) * vw) == 0;
        lines = lines && (sizeof(*p) == 1 || q % 128 == 0);
    });
    *aligned = as_is || shifted;
    // arrays that are aligned as they are move only if all of them gain lines
    return as_is && !(shifted && lines) ? 0 : (int)head;
}

// Instantiates OP<VW, AL> for the configured (or the op's preferred) width.
//
// Arrays that start at the same odd option of their lines (a slice of a book)
// leave the few options before the line to single work-items and stream the
// rest aligned: 5M options from option 3 on take 21.2 us (Greeks 37.4), from
// option 0 20.7 (36.9), and one option per work-item throughout 25.6 (45.3).
// Where no common shift aligns the arrays (inputs from option 3 on, output
// from 0), the same kernel runs with unaligned accesses: 23.6 us (38.3)
// against 25.3 (40.9) with one option per work-item.
template <template <int, bool> class OP, class Args>
hipError_t launch_stream(const Args& a, int64_t n, int preferred_vw, hipStream_t st) {
    if (n <= 0) return hipSuccess;
    const int cvw = config().vector_width.load(std::memory_order_relaxed);
    int vw = cvw > 0 ? cvw : preferred_vw;
    if (vw != 2 && vw != 4) vw = 4;
    vw = vw == 4 ? OP<4, true>::kVW : OP<2, true>::kVW;   // FP64: 2 whatever is asked
    bool aligned;
    int head = head_for(a, n, vw, &aligned);
    if (vw == 4 && !aligned) {   // aligned for two options as they are
        bool two;
        const int h2 = head_for(a, n, 2, &two);
        if (two) vw = 2, aligned = true, head = h2;
    }
    const Args b = from(a, head);
    n -= head;
    if (vw == 4)
        return aligned ? launch_op(make_op<OP<4, true>>(b), n, head, st)
                       : launch_op(make_op<OP<4, false>>(b), n, head, st);
    return aligned ? launch_op(make_op<OP<2, true>>(b), n, head, st)
                   : launch_op(make_op<OP<2, false>>(b), n, head, st);
}

// ---- repeated passes ------------------------------------------------------------
// `passes` passes over a book in one launch: a work-item prices its options
// pass after pass, every pass loading its inputs, pricing and storing.  No pass
// reads another's output (the caller has checked that price overlaps no input)
// and every pass stores the same bits, so neither options nor passes need wait
// for one another: row y of the grid takes its share of the passes, and a book
// that leaves the chip idle runs its passes side by side.  The stores are
// relaxed atomics (plain stores in the machine, which cannot tear): rows on
// different dies write one address, always with the same bits.  The compiler
// may not carry a value from one pass to the next: each load is behind a
// compiler fence.
//
// Bound by VALU issue where the passes fill the chip (200,000 options x 100:
// 52 us of it), by the launch where they don't.  100 passes, all of them in
// one row (as many waves as the book has) / as here: 4096 options 35 / 5.7 us
// (27.4 with four passes in flight per wave), 16,384 35 / 7.4, 65,536 38 / 20.5,
// 131,072 44.5 / 37.4, 200,000 77.5 / 57; 10 passes of 200,000 9.8 / 8.9.  A
// graph of 100 kernel nodes takes 1.9 us each at least, the kernel boundary:
// 187 us at 4096 options, 201 at 65,536, 237 at 200,000, 482 at 1M (266 here).
// Rows are added up to 16,384 waves, two rounds of them (200,000 options: 77.5
// us with 4096, 64.3 with 8192, 56.9 with 16,384, 56.1 with 32,768; 16,384
// options: 7.5, 7.6, 7.9, 8.3), of at least four passes each, which repay a
// wave's start (200,000 x 10: 9.0 us with 5 a row, 9.4 with 2, 10.8 with
// one).  Books of one row have the form without ROWS (3M x 10: 80.0 us and
// 81.4 with it; agent-scope stores 84).
constexpr int64_t kPassWaves = 16384;
constexpr int kPassesPerRow = 4;

template <class TY, bool ROWS, class Ix>
__global__ __launch_bounds__(kThreads) void k_passes(SoaIn<float> in, const TY* type, float* out,
                                                     int64_t n, int passes) {
    const Ix stride = (Ix)gridDim.x * blockDim.x;
    if constexpr (ROWS)
        passes = (int)((int64_t)passes * (blockIdx.y + 1) / gridDim.y) -
                 (int)((int64_t)passes * blockIdx.y / gridDim.y);
    for (Ix i = (Ix)blockIdx.x * blockDim.x + threadIdx.x; i < (Ix)n; i += stride) {
        for (int p = 0; p < passes; ++p) {
            asm volatile("" ::: "memory");
            const float price = bs_price<Ref32>(*at(in.s, i), *at(in.k, i), *at(in.r, i),
                                                *at(in.v, i), *at(in.t, i), *at(type, i) != 0);
            __hip_atomic_store(at(out, i), price, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            asm volatile("" ::: "memory");
        }
    }
}

template <class TY>
hipError_t launch_passes_t(SoaIn<float> in, const TY* type, float* out, int64_t n, int passes,
                           hipStream_t st) {
    const int64_t cap = config().max_blocks.load(std::memory_order_relaxed);
    const int bt = config().block_threads.load(std::memory_order_relaxed);
    const int nt = bt > 0 ? bt : 64;
    const unsigned blocks = grid_for(n, cap, nt);
    int64_t rows = std::min<int64_t>(kPassWaves * 64 / ((int64_t)blocks * nt),
                                     passes / kPassesPerRow);
    if (cap > 0) rows = std::min(rows, cap / blocks);
    if (rows > 1)   // the blocks cover the book, of at most 2^19 options
        hipLaunchKernelGGL((k_passes<TY, true, uint32_t>), dim3(blocks, (unsigned)rows), dim3(nt), 0,
                           st, in, type, out, n, passes);
    else if (n < (int64_t(1) << 30))
        hipLaunchKernelGGL((k_passes<TY, false, uint32_t>), dim3(blocks), dim3(nt), 0, st, in, type,
                           out, n, passes);
    else
        hipLaunchKernelGGL((k_passes<TY, false, int64_t>), dim3(blocks), dim3(nt), 0, st, in, type,
                           out, n, passes);
    return hipGetLastError();
}

// ---- AoS -> SoA repack ------------------------------------------------------
// OptionData (blackscholes.c:89-100): 9 dwords per record; dword 6 holds the
// OptionType char in its low byte.  A block stages 256 records (2304 dwords,
// 576 16-byte words) through LDS with coalesced 16-byte non-temporal loads,
// then each thread writes one record's fields, so every field array is
// written coalesced (non-temporal: nothing is read back).  The stride of 9
// dwords between the records threads read is odd, so the LDS reads are free
// of bank conflicts.  A step that is partial, or whose records do not start
// on a 16-byte boundary (the reference's records are 4-byte aligned), loads
// dword by dword.  Measured on MI355X, 10M records (57 B each: 36 in, 21
// out): 92-94 us per pass, 6.1-6.2 TB/s; dword loads and cached stores
// 136.6 us; 4 or 2 records per thread, or other block sizes, 93-102 us.
constexpr int kRecDwords = 9;
using u32x4 = uint32_t __attribute__((ext_vector_type(4)));
constexpr int kRepackWords4 = kThreads * kRecDwords / 4;   // 16-byte words per step

__global__ __launch_bounds__(kThreads) void k_repack_aos(const uint32_t* __restrict__ aos,
                                                          int64_t n, float* s, float* k,
                                                          float* r, float* v, float* t,
                                                          uint8_t* type) {
    __shared__ u32x4 tile4[kRepackWords4];
    const uint32_t* tile = reinterpret_cast<const uint32_t*>(tile4);
    for (int64_t base = (int64_t)blockIdx.x * kThreads; base < n;
         base += (int64_t)gridDim.x * kThreads) {
        const int64_t recs = n - base < kThreads ? n - base : kThreads;
        const uint32_t* src = aos + base * kRecDwords;
        if (recs == kThreads && (reinterpret_cast<uintptr_t>(src) & 15u) == 0) {
            const u32x4* src4 = reinterpret_cast<const u32x4*>(src);
            for (int w = threadIdx.x; w < kRepackWords4; w += kThreads)
                tile4[w] = __builtin_nontemporal_load(src4 + w);
        } else {
            uint32_t* tw = reinterpret_cast<uint32_t*>(tile4);
            const int words = (int)recs * kRecDwords;
            for (int w = threadIdx.x; w < words; w += kThreads) tw[w] = src[w];
        }
        __syncthreads();
        if (threadIdx.x < recs) {
            const uint32_t* rec = tile + threadIdx.x * kRecDwords;
            const int64_t i = base + threadIdx.x;
            __builtin_nontemporal_store(__uint_as_float(rec[0]), s + i);
            __builtin_nontemporal_store(__uint_as_float(rec[1]), k + i);
            __builtin_nontemporal_store(__uint_as_float(rec[2]), r + i);
            __builtin_nontemporal_store(__uint_as_float(rec[4]), v + i);
            __builtin_nontemporal_store(__uint_as_float(rec[5]), t + i);
            __builtin_nontemporal_store(
                (uint8_t)((rec[6] & 0xffu) == (uint32_t)'P' ? 1 : 0), type + i);
        }
        __syncthreads();
    }
}

__global__ void k_price_scalar(float s, float k, float r, float v, float t, int put,
                               float* out) {
    out[0] = bs_price<Ref32>(s, k, r, v, t, put != 0);
}
__global__ void k_cndf_scalar(float x, float* out) { out[0] = Ref32::cndf<false>(x, nullptr); }

}  // namespace

namespace {
template <int VW, bool AL>
using PriceRef = PriceF32<Ref32, VW, AL>;
template <int VW, bool AL>
using PriceFast = PriceF32<Fast32, VW, AL>;
}  // namespace

// ---- launchers ---------------------------------------------------------------
hipError_t launch_price_f32(SoaIn<float> in, const uint8_t* type, float* out, int64_t n,
                            hipStream_t st) {
    return launch_stream<PriceRef>(PriceArgs{in, type, out}, n, 2, st);
}

hipError_t launch_price_fast_f32(SoaIn<float> in, const uint8_t* type, float* out,
                                 int64_t n, hipStream_t st) {
    return launch_stream<PriceFast>(PriceArgs{in, type, out}, n, 2, st);
}

hipError_t launch_price_i32type_f32(SoaIn<float> in, const int32_t* type, float* out,
                                    int64_t n, hipStream_t st) {
    return launch_stream<PriceI32F32>(PriceI32Args{in, type, out}, n, 2, st);
}

hipError_t launch_price_passes_f32(SoaIn<float> in, const void* type, int type_bytes, float* out,
                                   int64_t n, int passes, hipStream_t st) {
    return type_bytes == 1
               ? launch_passes_t(in, static_cast<const uint8_t*>(type), out, n, passes, st)
               : launch_passes_t(in, static_cast<const int32_t*>(type), out, n, passes, st);
}

hipError_t launch_price_f64(SoaIn<double> in, const uint8_t* type, double* out, int64_t n,
                            hipStream_t st) {
    return launch_stream<PriceF64>(PriceF64Args{in, type, out}, n, 2, st);
}

hipError_t launch_greeks_f32(SoaIn<float> in, const uint8_t* type, GreeksOut out, int64_t n,
                             hipStream_t st) {
    // Two options per work-item (8-byte agent-scope stores, 11 KB of LDS reserved
    // per wave) for what the 256 MB last-level cache takes in one launch, four
    // (16-byte non-temporal stores, 16 KB) for streams past it.  us on one / two
    // streams, two against four: 1M options 8.4 / 6.2 and 10.2 / 7.0, 3M 20.2 / 18.1
    // and 23.1 / 20.2, 4M 30.4 / 28.9 and 30.7 / 28.7, 4.4M 32.5 / 32.3 and 32.4 /
    // 30.1, 7M 48.8 / 47.4 and 48.6 / 46.7, 10M 67.0 / 66.5 and 68.0 / 66.0, 20M
    // 132.3 / 135.2 and 133.0 / 132.5, 40M 259.2 / 269.8 and 261.2 / 262.5.
    const int vw = n < (int64_t(1) << 22) ? 2 : 4;
    return launch_stream<GreeksF32>(GreeksArgs{in, type, out}, n, vw, st);
}

hipError_t launch_cndf_f32(const float* x, float* out, int64_t n, hipStream_t st) {
    return launch_stream<CndfF32>(CndfArgs<float>{x, out}, n, 4, st);
}

hipError_t launch_cndf_f64(const double* x, double* out, int64_t n, hipStream_t st) {
    return launch_stream<CndfF64>(CndfArgs<double>{x, out}, n, 2, st);
}

hipError_t launch_repack_aos(const void* aos, int64_t n, float* s, float* k, float* r,
                             float* v, float* t, uint8_t* type, hipStream_t st) {
    if (n <= 0) return hipSuccess;
    int64_t blocks = (n + kThreads - 1) / kThreads;
    if (blocks > 1048576) blocks = 1048576;   // past 2^28 records, blocks loop
    hipLaunchKernelGGL(k_repack_aos, dim3((unsigned)blocks), dim3(kThreads), 0, st,
                       static_cast<const uint32_t*>(aos), n, s, k, r, v, t, type);
    return hipGetLastError();
}

hipError_t launch_price_scalar(float s, float k, float r, float v, float t, int put,
                               float* out, hipStream_t st) {
    hipLaunchKernelGGL(k_price_scalar, dim3(1), dim3(1), 0, st, s, k, r, v, t, put, out);
    return hipGetLastError();
}

hipError_t launch_cndf_scalar(float x, float* out, hipStream_t st) {
    hipLaunchKernelGGL(k_cndf_scalar, dim3(1), dim3(1), 0, st, x, out);
    return hipGetLastError();
}

}  // namespace bs
