// bs_portfolio.hip -- portfolio reductions over a book: the MapReduce step
// after the map (SkePU2 MapReduce, skepu2/backend/impl/mapreduce/).
//
// sums[0] = sum_i w_i * price_i and, with Greeks, sums[1..4] = the same sums of
// delta, vega, rho and theta, where each per-option value is exactly the one
// the map computes (the same per-option code, bs_math.hpp) and w_i is the
// position (1 when no weights are given).
//
// One kernel on the caller's stream, k_pf_rows: a block owns `rows` consecutive
// rows of 256 two-option groups (the map's loads: one 8-byte load per array per
// lane, so each wave instruction reads 512 contiguous bytes), wave w of it the
// w-th run of `rows` rows of 64; a lane walks its column of those rows in order,
// the next row's loads issued before the current row's arithmetic, and adds
// w*value to FP64 accumulators; each wave folds its lanes with a fixed
// wave sum and the block its waves in order into one partial.  The last block
// of every 64 to arrive folds their partials with one wave sum, and the last
// of those folds the groups of 64 (bs_arrive.hpp): no second launch, and nothing
// waits.  The
// shape of the sum depends only on n, so the sums are bit-reproducible for a
// given book, wherever its arrays start.
//
// Scratch (counters and partials): slots of a fixed device array, claimed on
// the host by a flag in pinned memory that the kernel's last block clears, so
// calls on any threads and streams never share one.  With no slot free, and
// under stream capture (a graph may be replayed at any time), the partials go
// to stream-ordered memory and a second launch, k_pf_final, adds them in the
// same order; bs_portfolio_f32_noalloc does the same with an array of its own.
//
// Traffic: 21 bytes per option read (25 with weights), 8 or 40 bytes written
// in all, plus 8 or 40 bytes per block.
#include <algorithm>
#include <atomic>
#include <mutex>
#include <type_traits>

#include "bs_arrive.hpp"
#include "bs_internal.hpp"
#include "bs_math.hpp"
#include "bs_ops.hpp"
#include "bs_wave.hpp"

namespace bs {
namespace {

constexpr int kPfThreads = 256;
constexpr int kPfWaves = kPfThreads / 64;
constexpr int kPfGroup = 64;            // blocks per group of partials
constexpr int64_t kPfMaxBlocks = 8192;  // 128 groups: two per lane of the last fold
constexpr int kPfMaxGroups = kPfMaxBlocks / kPfGroup;

struct PfArgs {
    SoaIn<float> in;
    const uint8_t* type;
    const float* w;   // NULL: every weight is 1
    int64_t n;
    int64_t rows;     // rows of 64 groups per wave
    double* partial;  // [blocks][NQ]
};

// A call's scratch in the one-launch form; the counters are zero between calls,
// 256 bytes apart.
struct PfCounter {
    uint32_t done;
    uint32_t pad[63];
};
struct PfSlot {
    PfCounter groups;
    PfCounter blocks[kPfMaxGroups];
    double group[kPfMaxGroups * 5];
    double partial[kPfMaxBlocks * 5];
};

template <bool kGreeks>
__device__ __forceinline__ void add_option(double* acc, float s, float k, float r, float v,
                                           float t, bool put, float w) {
    const double dw = (double)w;
    if constexpr (kGreeks) {
        const Greeks32 g = bs_greeks<Ref32>(s, k, r, v, t, put);
        acc[0] += dw * (double)g.price;
        acc[1] += dw * (double)g.delta;
        acc[2] += dw * (double)g.vega;
        acc[3] += dw * (double)g.rho;
        acc[4] += dw * (double)g.theta;
    } else {
        acc[0] += dw * (double)bs_price<Ref32>(s, k, r, v, t, put);
    }
}

// One group's inputs.  Ix = uint32_t when every array of the call spans less
// than 4 GiB (32-bit offsets on the arrays' bases), else int64_t.  AL false:
// some array is not aligned for two options (cached loads, as in the maps).
using F2 = vec<float, 2>;
struct PfOptions {
    F2 s, k, r, v, t, w;
    uint32_t ty;
};

template <bool AL, class Ix>
__device__ __forceinline__ PfOptions pf_load(const PfArgs& a, Ix g) {
    PfOptions x;
    x.s = ld<AL>(at(reinterpret_cast<const F2*>(a.in.s), g));
    x.k = ld<AL>(at(reinterpret_cast<const F2*>(a.in.k), g));
    x.r = ld<AL>(at(reinterpret_cast<const F2*>(a.in.r), g));
    x.v = ld<AL>(at(reinterpret_cast<const F2*>(a.in.v), g));
    x.t = ld<AL>(at(reinterpret_cast<const F2*>(a.in.t), g));
    x.ty = ld<AL>(at(reinterpret_cast<const uint16_t*>(a.type), g));
    if (a.w) x.w = ld<AL>(at(reinterpret_cast<const F2*>(a.w), g));
    else x.w = F2(1.0f);
    return x;
}

template <bool kGreeks>
__device__ __forceinline__ void pf_add(double* acc, const PfOptions& x) {
#pragma unroll
    for (int j = 0; j < 2; ++j)
        add_option<kGreeks>(acc, x.s[j], x.k[j], x.r[j], x.v[j], x.t[j], put_of(x.ty, j), x.w[j]);
}

// One wave's sums of NQ quantities: of group g's partials, and of the groups'.
// load(i, q) gives quantity q of partial (group) i; both launch forms fold in
// these shapes.
template <int NQ, class Load>
__device__ __forceinline__ void fold_blocks(int g, int blocks, int lane, double (&x)[NQ],
                                            Load&& load) {
    const int b = g * kPfGroup + lane;
#pragma unroll
    for (int q = 0; q < NQ; ++q) x[q] = b < blocks ? load(b, q) : 0.0;
#pragma unroll
    for (int q = 0; q < NQ; ++q) x[q] = wave_sum(x[q]);
}
template <int NQ, class Load>
__device__ __forceinline__ void fold_groups(int groups, int lane, double (&x)[NQ], Load&& load) {
    double hi[NQ];
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
        x[q] = lane < groups ? load(lane, q) : 0.0;
        hi[q] = lane + 64 < groups ? load(lane + 64, q) : 0.0;
    }
#pragma unroll
    for (int q = 0; q < NQ; ++q) x[q] = wave_sum(x[q] + hi[q]);
}

// x[q] for q = lane, the same for every lane past NQ.
template <int NQ>
__device__ __forceinline__ double pick(const double (&x)[NQ], int lane) {
    double v = x[0];
#pragma unroll
    for (int q = 1; q < NQ; ++q) v = lane == q ? x[q] : v;
    return v;
}

// slot: the one-launch form's scratch, its host flag and the sums' place; NULL
// leaves the partials in a.partial for k_pf_final.
template <bool kGreeks, bool AL, class Ix>
__global__ __launch_bounds__(kPfThreads) __attribute__((amdgpu_waves_per_eu(kGreeks ? 4 : 5)))
void k_pf_rows(PfArgs a, PfSlot* slot, uint32_t* busy, double* __restrict__ sums) {
    constexpr int NQ = kGreeks ? 5 : 1;
    double acc[NQ];
#pragma unroll
    for (int q = 0; q < NQ; ++q) acc[q] = 0.0;
    const Ix ngroups = (Ix)(a.n / 2);
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x / 64;
    const Ix span = (Ix)a.rows * 64;
    Ix g = ((Ix)blockIdx.x * kPfWaves + wave) * span + lane;
    const Ix g_end = g + span;
    if (g < ngroups) {
        PfOptions cur = pf_load<AL>(a, g);
        for (Ix gn = g + 64; gn < g_end && gn < ngroups; gn += 64) {
            const PfOptions nxt = pf_load<AL>(a, gn);
            pf_add<kGreeks>(acc, cur);
            cur = nxt;
            g = gn;
        }
        pf_add<kGreeks>(acc, cur);
        g += 64;
    }
    if ((a.n & 1) && g == ngroups && g < g_end) {   // the last option of an odd book
        const int64_t i = a.n - 1;
        add_option<kGreeks>(acc, a.in.s[i], a.in.k[i], a.in.r[i], a.in.v[i], a.in.t[i],
                            a.type[i] != 0, a.w ? a.w[i] : 1.0f);
    }
    __shared__ double lds[kPfWaves][NQ];
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
        const double x = wave_sum(acc[q]);
        if (lane == 0) lds[wave][q] = x;
    }
    __syncthreads();
    if (wave != 0) return;
    if (lane < NQ) {
        double v = lds[0][lane];
#pragma unroll
        for (int w = 1; w < kPfWaves; ++w) v += lds[w][lane];
        agent_store(a.partial + (int64_t)blockIdx.x * NQ + lane, v);
    }
    if (!slot) return;
    stores_done();
    const int blocks = gridDim.x, groups = (blocks + kPfGroup - 1) / kPfGroup;
    const int gr = blockIdx.x / kPfGroup;
    if (!arrive(&slot->blocks[gr].done, min(kPfGroup, blocks - gr * kPfGroup))) return;
    double x[NQ];
    fold_blocks(gr, blocks, lane, x, [&](int b, int q) {
        return agent_load(a.partial + (int64_t)b * NQ + q);
    });
    if (lane < NQ) agent_store(&slot->group[gr * NQ + lane], pick(x, lane));
    if (lane == 0) agent_store(&slot->blocks[gr].done, 0u);
    stores_done();
    if (!arrive(&slot->groups.done, groups)) return;
    fold_groups(groups, lane, x, [&](int i, int q) { return agent_load(&slot->group[i * NQ + q]); });
    if (lane < NQ) sums[lane] = pick(x, lane);
    if (lane == 0) agent_store(&slot->groups.done, 0u);
    stores_done();
    if (lane == 0) system_store(busy, 0u);
}

// The second launch of the two-launch form: one block folds the partials, a
// wave per group up to 16.
constexpr int kPfFinalThreads = 1024;

template <int NQ>
__global__ __launch_bounds__(kPfFinalThreads) void k_pf_final(const double* __restrict__ in,
                                                              int blocks,
                                                              double* __restrict__ out) {
    __shared__ double lds[kPfMaxGroups][NQ];
    const int lane = threadIdx.x & 63;
    const int groups = (blocks + kPfGroup - 1) / kPfGroup;
    double x[NQ];
    for (int g = threadIdx.x / 64; g < groups; g += (int)blockDim.x / 64) {
        fold_blocks(g, blocks, lane, x, [&](int b, int q) { return in[(int64_t)b * NQ + q]; });
        if (lane < NQ) lds[g][lane] = pick(x, lane);
    }
    __syncthreads();
    if (threadIdx.x >= 64) return;
    fold_groups(groups, lane, x, [&](int i, int q) { return lds[i][q]; });
    if (lane < NQ) out[lane] = pick(x, lane);
}

// Rows per wave: one while that makes fewer than kPfSpread blocks, so that a
// small book spreads over the chip (1280 blocks of the price form are resident at
// once); then up to kPfMostRows, which keeps the blocks' counting in rare against
// their options; more only to stay within kPfMaxBlocks.  With and without Greeks
// alike, so that the sum of prices has the same bits in both.  us a call, price
// sums / with Greeks / with Greeks and weights, for (rows, spread), one stream:
//         (4, 1024)            (6, 1536)            (6, 2048)            (8, 2048)
//   1M     8.5 / 13.2 / 13.3    8.5 / 13.1 / 13.2    8.5 / 13.2 / 13.2    8.6 / 13.2 / 13.3
//   1.5M  10.3 / 15.0 / 15.1   10.2 / 15.6 / 15.7   10.2 / 15.6 / 15.7   10.2 / 15.6 / 15.7
//   2.5M  13.7 / 19.3 / 19.6   13.9 / 19.4 / 20.0   13.2 / 19.7 / 20.1   13.2 / 19.6 / 20.2
//   4M    18.7 / 25.9 / 26.2   19.8 / 26.6 / 26.9   18.7 / 26.0 / 26.4   18.7 / 26.1 / 26.4
//   6M    25.1 / 34.0 / 34.2   25.4 / 33.5 / 33.9   25.5 / 34.4 / 34.4   25.6 / 34.4 / 34.4
//   10M   38.3 / 49.6 / 51.6   38.3 / 47.6 / 50.1   38.1 / 47.8 / 50.1   38.9 / 48.7 / 51.1
// and on two streams 10M 34.8 / 45.2, 34.4 / 44.0, 34.4 / 44.0, 34.4 / 43.5; price
// sums of 10M with weights 41.3, 41.7, 41.6, 43.2, and with 16 rows 44 without.
//
// The whole call, against one wave per 8 rows and one final block in two
// launches with stream-ordered scratch: 65,537 options 5.9 us and 23.4 (the
// host's allocation); 1M 8.5 and 25, with Greeks 13.2 and 25; 10M 38.1 and
// 47.1, with Greeks and weights 50.1 and 61 (the final block alone 8.8).
// Bound by HBM (price) and VALU issue (Greeks).
constexpr int64_t kPfSpread = 2048;
constexpr int64_t kPfMostRows = 6;

struct PfShape {
    int64_t rows, blocks;
};
constexpr PfShape pf_shape(int64_t n) {
    const int64_t items = n / 2 + (n & 1);
    auto up = [](int64_t a, int64_t b) { return (a + b - 1) / b; };
    int64_t rows = std::min(kPfMostRows, std::max<int64_t>(1, items / (kPfThreads * kPfSpread)));
    rows = std::max(rows, up(items, kPfThreads * kPfMaxBlocks));
    return {rows, std::max<int64_t>(1, up(items, kPfThreads * rows))};
}

// slot NULL: the two-launch form with a.partial.
template <bool kGreeks, bool AL>
hipError_t launch_pf(PfArgs a, PfSlot* slot, uint32_t* busy, double* sums, hipStream_t st) {
    const PfShape shape = pf_shape(a.n);
    a.rows = shape.rows;
    if (slot) a.partial = slot->partial;
    // LDS reserved per block caps the waves resident on a CU: none by default
    // (a block holds its LDS while its last wave counts it in: 10M options with
    // Greeks and weights took 57.8 us with 8 KB per wave and 56.2 with none)
    const int lw = config().lds_per_wave.load(std::memory_order_relaxed);
    const size_t lds = std::min<size_t>((size_t)std::max(lw, 0) * kPfWaves, 65536 - 512);
    const dim3 grid((unsigned)shape.blocks), block(kPfThreads);
    if (a.n < (int64_t(1) << 30))
        hipLaunchKernelGGL((k_pf_rows<kGreeks, AL, uint32_t>), grid, block, lds, st, a, slot, busy,
                           sums);
    else
        hipLaunchKernelGGL((k_pf_rows<kGreeks, AL, int64_t>), grid, block, lds, st, a, slot, busy,
                           sums);
    if (!slot)
        hipLaunchKernelGGL((k_pf_final<kGreeks ? 5 : 1>), dim3(1),
                           dim3((unsigned)std::min<int64_t>(
                               (shape.blocks + kPfGroup - 1) / kPfGroup * 64, kPfFinalThreads)),
                           0, st, a.partial, (int)shape.blocks, sums);
    return hipGetLastError();
}

bool pf_aligned(const PfArgs& a) {
    auto al = [](const void* p, uintptr_t b) { return (reinterpret_cast<uintptr_t>(p) & (b - 1)) == 0; };
    return al(a.in.s, 8) && al(a.in.k, 8) && al(a.in.r, 8) && al(a.in.v, 8) && al(a.in.t, 8) &&
           al(a.type, 2) && (a.w == nullptr || al(a.w, 8));
}

hipError_t launch_pf_any(const PfArgs& a, bool greeks, PfSlot* slot, uint32_t* busy, double* sums,
                         hipStream_t st) {
    if (pf_aligned(a))
        return greeks ? launch_pf<true, true>(a, slot, busy, sums, st)
                      : launch_pf<false, true>(a, slot, busy, sums, st);
    return greeks ? launch_pf<true, false>(a, slot, busy, sums, st)
                  : launch_pf<false, false>(a, slot, busy, sums, st);
}

// ---- scratch ---------------------------------------------------------------------
// Fixed device arrays, held on every device the library runs on until the
// process ends: kPfSlots slots of the one-launch form (12 MB in all) and the
// partials of bs_portfolio_f32_noalloc (0.3 MB).  In host code the arrays'
// names are not device addresses: their addresses on each device come from
// hipGetSymbolAddress, resolved once per device with that device current, and
// only those reach a kernel.
constexpr int kPfSlots = 32;
__device__ __align__(256) PfSlot g_pf_slots[kPfSlots];
__device__ __align__(256) double g_pf_scratch[kPfMaxBlocks * 5];

constexpr int kPfMaxDevices = 64;
struct PfDevice {
    std::mutex mu;
    PfSlot* slots = nullptr;
    double* scratch = nullptr;
    uint32_t* busy = nullptr;       // pinned, one flag per slot, a cache line apart
    uint32_t* busy_dev = nullptr;   // the same memory, device address
    std::atomic<unsigned> next{0};
};
constexpr int kPfFlagStride = 64 / sizeof(uint32_t);

PfDevice& pf_device(int dev) {
    static PfDevice* d = new PfDevice[kPfMaxDevices];   // lives until the process ends
    return d[dev];
}

template <class T, class S>
hipError_t symbol_address(T** p, const S& symbol) {
    void* a = nullptr;
    const hipError_t e = hipGetSymbolAddress(&a, symbol);
    if (e == hipSuccess) *p = static_cast<T*>(a);
    return e;
}

hipError_t pf_scratch_of(int dev, double** out) {
    if (dev < 0 || dev >= kPfMaxDevices) return hipErrorInvalidDevice;
    PfDevice& d = pf_device(dev);
    std::lock_guard<std::mutex> lk(d.mu);
    hipError_t e = hipSuccess;
    if (!d.scratch) e = symbol_address(&d.scratch, HIP_SYMBOL(g_pf_scratch));
    *out = d.scratch;
    return e;
}

// Claims a free slot of the device, or returns -1 (none free, or no flags).
int claim_slot(PfDevice& d) {
    {
        std::lock_guard<std::mutex> lk(d.mu);
        if (!d.slots && symbol_address(&d.slots, HIP_SYMBOL(g_pf_slots)) != hipSuccess) {
            (void)hipGetLastError();
            return -1;
        }
        if (!d.busy) {
            const RelaxedCapture relaxed;
            uint32_t* p = nullptr;
            void* q = nullptr;
            if (hipHostMalloc(reinterpret_cast<void**>(&p), kPfSlots * 64, hipHostMallocCoherent) !=
                hipSuccess) {
                (void)hipGetLastError();
                return -1;
            }
            if (hipHostGetDevicePointer(&q, p, 0) != hipSuccess) {
                (void)hipGetLastError();
                (void)hipHostFree(p);
                return -1;
            }
            std::fill(p, p + kPfSlots * kPfFlagStride, 0u);
            d.busy_dev = static_cast<uint32_t*>(q);
            d.busy = p;
        }
    }
    const unsigned first = d.next.fetch_add(1, std::memory_order_relaxed);
    for (unsigned i = 0; i < kPfSlots; ++i) {
        const unsigned s = (first + i) % kPfSlots;
        uint32_t idle = 0;
        if (__atomic_compare_exchange_n(d.busy + s * kPfFlagStride, &idle, 1u, false,
                                        __ATOMIC_ACQUIRE, __ATOMIC_RELAXED))
            return (int)s;
    }
    return -1;
}

}  // namespace

// bs_portfolio_f32 with the device's fixed partials: no allocation.  The caller
// has checked n <= kPfNoAllocMaxOptions.  Calls that overlap on one device
// share the array and race (the two-launch form: a race leaves no counter
// behind that a later call could meet).
hipError_t launch_portfolio_f32_noalloc(SoaIn<float> in, const uint8_t* type, const float* w,
                                        int64_t n, bool greeks, double* sums, hipStream_t st) {
    if (n > kPfNoAllocMaxOptions) return hipErrorInvalidValue;
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    PfArgs a{in, type, w, n, 0, nullptr};
    e = pf_scratch_of(dev, &a.partial);
    if (e != hipSuccess) return e;
    return launch_pf_any(a, greeks, nullptr, nullptr, sums, st);
}

hipError_t launch_portfolio_f32(SoaIn<float> in, const uint8_t* type, const float* w, int64_t n,
                                bool greeks, double* sums, hipStream_t st) {
    PfArgs a{in, type, w, n, 0, nullptr};
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    if (dev < kPfMaxDevices && !capturing(st)) {
        PfDevice& d = pf_device(dev);
        const int s = claim_slot(d);
        if (s >= 0) {
            e = launch_pf_any(a, greeks, d.slots + s, d.busy_dev + s * kPfFlagStride, sums, st);
            if (e != hipSuccess)   // nothing will run that clears the flag
                __atomic_store_n(d.busy + s * kPfFlagStride, 0u, __ATOMIC_RELEASE);
            return e;
        }
    }
    e = hipMallocAsync(reinterpret_cast<void**>(&a.partial),
                       (size_t)pf_shape(n).blocks * (greeks ? 5 : 1) * sizeof(double), st);
    if (e != hipSuccess) return e;
    e = launch_pf_any(a, greeks, nullptr, nullptr, sums, st);
    const hipError_t f = hipFreeAsync(a.partial, st);
    return e != hipSuccess ? e : f;
}

}  // namespace bs
