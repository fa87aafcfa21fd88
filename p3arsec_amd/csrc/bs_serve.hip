// bs_serve.hip -- the serving loop: resident books, continuous batching,
// fused launches of every queued request.
//
// A context owns
//   * one device arena (hipMalloc of the HBM budget) holding resident books
//     and request outputs, carved by serve::Core's segregated-fit allocator;
//   * six descriptor slots, each a pinned host table plus its device copy;
//   * per batch, a stage kernel that copies the slot's table from pinned host
//     memory to the device, then one fused kernel per section (the batch's
//     price requests, its Greeks requests): a block prices one tile of 512
//     options of one request, found by a 64-ary wave search of the table.  A
//     batch of at most 32 requests and 2048 tiles that finds little or nothing in
//     flight is one kernel with the table as its argument.
//     Launched directly (the default) each section's grid is one block per
//     tile.  With use_graph the three kernels are captured once per slot and
//     each batch is one hipGraphLaunch; before it, each section's node gets
//     the batch's grid (hipGraphExecKernelNodeSetParams).  On ROCm 7.2 the
//     direct form measured 15 us launch-to-completion against 31 us;
//   * a dispatcher thread (serve_loop.hpp): it admits queued requests as arena
//     memory allows, writes a table into a free slot and launches it, and
//     retires each batch when its event completes.  Requests of at most 64K
//     options (bs_serve_opts.small_request_options) form batches of their own
//     on a stream of their own (two in flight), so they complete beside large
//     requests rather than behind them; the rest alternate over two streams
//     (four in flight).  Requests that arrive while batches run go into the
//     next batch of their lane.
// Results are bit-identical to bs_price_f32 / bs_price_greeks_f32: the fused
// kernels run the batch map's own per-group code (bs_ops.hpp).
#include <stddef.h>
#include <string.h>
#include <time.h>

#include <algorithm>
#include <mutex>
#include <string>
#include <vector>

#include "bs_arrive.hpp"
#include "bs_internal.hpp"
#include "bs_math.hpp"
#include "bs_ops.hpp"
#include "serve_core.hpp"
#include "serve_loop.hpp"

namespace bs {
namespace {

constexpr int kVW = 2;                 // options per work-item (the batch map's width)
// Threads per block of the fused kernels, chosen per context from
// BS_CFG_BLOCK_THREADS (64, 128 or 256; 0 = kServeThreads); a tile is one
// block step, threads x kVW options.
constexpr int kServeThreads = 256;
constexpr int kMaxDesc = 4096;         // requests per batch: 64 x 64 for find_desc
constexpr int64_t kMaxGrid = int64_t(1) << 20;  // default section grid cap (blocks loop)
constexpr int kStageBlocks = 32;

// One request of a batch: 112 bytes, a multiple of the stage kernel's 16-byte words.
struct Desc {
    const float* in[5];   // s, k, r, v, t
    const uint8_t* type;
    float* out[5];        // price, delta, vega, rho, theta (Greeks only use 1..4)
    int64_t n;
    int64_t tile_begin;   // first tile of this request within its section
    int32_t kind;
    int32_t pad;
};
static_assert(sizeof(Desc) == 112, "Desc layout");

// A batch's table: the header, then the price requests' descriptors, then the
// Greeks requests' descriptors.  Section 0 is price, section 1 Greeks.
struct SlotHeader {
    int32_t ndesc[2];
    int64_t tiles[2];
    int64_t seq;
    int64_t pad[4];
};
static_assert(sizeof(SlotHeader) == 64, "SlotHeader layout");

constexpr size_t kSlotBytes = sizeof(SlotHeader) + sizeof(Desc) * kMaxDesc;

// Copies header + descriptors from the pinned table to device memory.
__global__ __launch_bounds__(kThreads) void k_stage(const uint4* __restrict__ host,
                                                    uint4* __restrict__ dev) {
    const SlotHeader* h = reinterpret_cast<const SlotHeader*>(host);
    const int np = h->ndesc[0], ng = h->ndesc[1];
    const int ndesc = (np < 0 || ng < 0 || np + ng > kMaxDesc) ? 0 : np + ng;
    const int64_t words = (int64_t)(sizeof(SlotHeader) + sizeof(Desc) * ndesc) / 16;
    for (int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x; i < words;
         i += (int64_t)gridDim.x * kThreads)
        dev[i] = host[i];
}

// The request of tile t among d[0, nd): the last descriptor whose tile_begin
// <= t.  A 64-ary search over tile_begin (increasing, d[0].tile_begin == 0):
// each wave resolves 64 x 64 = 4096 descriptors with two loads per lane.
__device__ __forceinline__ int find_desc(const Desc* d, int nd, int64_t t) {
    const int lane = threadIdx.x & 63;
    int j = lane * 64;
    const int base = (__popcll(__ballot(j < nd && d[j].tile_begin <= t)) - 1) * 64;
    j = base + lane;
    return base + __popcll(__ballot(j < nd && d[j].tile_begin <= t)) - 1;
}

template <class Op>
__device__ __forceinline__ Op op_of(const Desc& x);
template <>
__device__ __forceinline__ PriceF32<Ref32, kVW> op_of(const Desc& x) {
    return {SoaIn<float>{x.in[0], x.in[1], x.in[2], x.in[3], x.in[4]}, x.type, x.out[0]};
}
template <>
__device__ __forceinline__ GreeksF32<kVW> op_of(const Desc& x) {
    return {SoaIn<float>{x.in[0], x.in[1], x.in[2], x.in[3], x.in[4]}, x.type,
            GreeksOut{x.out[0], x.out[1], x.out[2], x.out[3], x.out[4]}};
}

// Fused kernel of one section: a block prices tile t (kThr x kVW options of
// one request, one kVW-group per work-item) for t = blockIdx.x, + gridDim.x, ...
// The grid has one block per tile up to the context's cap (kMaxGrid unless
// bs_serve_opts.grid_blocks sets it), in both launch forms.
// Every access is bounded by the request's n.
// The per-group code is the batch map's own (bs_ops.hpp).
template <class Op, int kSection, int kThr>
__global__ __launch_bounds__(kThr) __attribute__((amdgpu_waves_per_eu(waves_for<Op, false>())))
void k_serve(const uint8_t* __restrict__ slot) {
    const SlotHeader* h = reinterpret_cast<const SlotHeader*>(slot);
    const int np = h->ndesc[0], ng = h->ndesc[1];
    if (np < 0 || ng < 0 || np + ng > kMaxDesc) return;
    const int nd = kSection == 0 ? np : ng;
    if (nd <= 0) return;
    const Desc* d = reinterpret_cast<const Desc*>(slot + sizeof(SlotHeader)) + (kSection ? np : 0);
    const int64_t tiles = h->tiles[kSection];
    for (int64_t t = blockIdx.x; t < tiles; t += gridDim.x) {
        const Desc& x = d[find_desc(d, nd, t)];
        const Op op = op_of<Op>(x);
        const int64_t n = x.n;
        const int64_t g = (t - x.tile_begin) * kThr + threadIdx.x;
        if ((g + 1) * kVW <= n) {
            op.template finish<true>(g, op.template load<true>(g));
        } else {
            for (int64_t i = g * kVW; i < n; ++i) op.scalar(i);
        }
    }
}

// ---- replies -----------------------------------------------------------------
// bs_result_copy's way to the host: one kernel writes the wanted outputs of a
// request (one span of the arena where they lie side by side) into pinned memory
// and then the reply's sequence number, on which the caller spins; the arrays go
// on to the caller's from there.  The runtime's own copies take 11-35 us each to pageable memory (copy
// kernel, marker, interrupt), five of them for a Greeks request: a round of 32
// requests of up to 64K options, one third with Greeks, submitted, waited for
// and copied out one by one takes 390 us, with those copies 1050.
// Bound by the launch and the link's latency.
//
// us a copy, reply and runtime: price of 1000 options 7.7 and 14.6, of 65,536
// 18.2 and 20.1; all five Greeks outputs of 1000 9.3 and 70, of 65,536 61 and 96,
// price and theta of 65,536 28 and 38.  A reply holds the largest request of the
// small lane with Greeks; past it the gain is less (of 131,072, all five 121 and
// 150, price alone 28 and 29).  Two replies, as one thread's memcpy is the other's
// kernel: 1, 2, 4 and 8 threads copying 16,384 options with Greeks get one every
// 22.2, 12.9, 11.9, 12.0 us (22.2, 13.0, 8.9, 9.5 with four; 61-69 by the runtime).
constexpr int kReplies = 2;                         // replies on their way at once
constexpr size_t kReplyBytes = size_t(3) << 19;     // 1.5 MB: the Greeks of 64K options
constexpr int kReplyBlocks = 64;

// This block's part of `words` 8-byte words; the last block raises the flag.
__device__ __forceinline__ void reply_words(const uint64_t* __restrict__ src,
                                            uint64_t* __restrict__ dst, int words, uint32_t blocks,
                                            uint32_t* count, uint32_t* flag, uint32_t seq) {
    for (int i = blockIdx.x * kThreads + threadIdx.x; i < words; i += gridDim.x * kThreads)
        system_store(dst + i, src[i]);
    stores_done();
    __syncthreads();
    if (threadIdx.x == 0 && arrive_one(count, blocks)) {
        agent_store(count, 0u);   // for the next reply, which the stream orders behind this one
        system_store(flag, seq);
    }
}
__global__ __launch_bounds__(kThreads) void k_reply(const uint64_t* src, uint64_t* dst, int words,
                                                    uint32_t* count, uint32_t* flag,
                                                    uint32_t seq) {
    reply_words(src, dst, words, gridDim.x, count, flag, seq);
}
// Outputs with others between them: row y of the grid takes the output
// (order >> 4 y) & 15 after src, outputs `stride` words apart.  (Its arguments cost
// a reply of one span 0.2 us.)
__global__ __launch_bounds__(kThreads) void k_reply_rows(const uint64_t* src, uint64_t* dst,
                                                         int words, int stride, uint32_t order,
                                                         uint32_t* count, uint32_t* flag,
                                                         uint32_t seq) {
    reply_words(src + (int64_t)((order >> (4 * blockIdx.y)) & 15u) * stride,
                dst + (int64_t)blockIdx.y * words, words, gridDim.x * gridDim.y, count, flag, seq);
}

__global__ void k_zero_word(uint32_t* p) { *p = 0; }

using ServePrice = PriceF32<Ref32, kVW>;
using ServeGreeks = GreeksF32<kVW>;

// A small batch in one launch: its table travels as the kernel's argument, and
// one grid holds the price section's tiles, then the Greeks section's.  The
// stage kernel and a kernel per section cost 14 us of GPU time and two launches
// for requests that price in 3: 32 requests submitted together are done in 19 us
// and 25, one of 1M options in 21 and 25.  Only a batch that finds nothing else in
// flight takes it, or one of at most 4 requests that finds one other.  Where more
// are, a batch's wait is what the dispatcher's next round can be filled with: with
// every small batch in this form, rounds came more often and smaller, and the bulk
// lane's tail grew.  Every small batch / by this rule / only with nothing else in
// flight / none, at a Poisson rate, the middle of four runs in turn:
//   20,000/s     p50 20.0, 21.4, 22.4, 25.0 us
//   200,000/s    p50 21-37, 29-42, 35-43, 33-44 us over the four
//   800,000/s    p99 205, 152, 161, 158 us (of books up to 64K options 139, 129, 135, 128)
//   1,200,000/s  p99 242, 178, 186, 175 us (207, 136, 140, 128)
// Larger batches keep the three kernels (at saturation one kernel for both
// sections, at the Greeks form's registers, ran 1.73e11 options/s against 1.76e11).
constexpr int kSmallDesc = 32;
constexpr int kSmallBeside = 4;   // with one other batch in flight
constexpr int64_t kSmallTiles = 2048;
struct SmallBatch {
    int32_t np, nd;         // price requests, all requests
    int32_t price_tiles, pad;
    Desc d[kSmallDesc];     // price requests first; tile_begin counts through the batch
};
static_assert(sizeof(SmallBatch) <= 4096, "fits a kernel's arguments");

template <int kThr>
__global__ __launch_bounds__(kThr) __attribute__((amdgpu_waves_per_eu(waves_for<ServeGreeks, false>())))
void k_serve_small(const SmallBatch b) {
    const int64_t t = blockIdx.x;
    const int lane = threadIdx.x & 63;
    const uint64_t before = __ballot(lane < b.nd && b.d[lane < kSmallDesc ? lane : 0].tile_begin <= t);
    const Desc& x = b.d[__builtin_amdgcn_readfirstlane(__popcll(before) - 1)];
    const int64_t n = x.n;
    const int64_t g = (t - x.tile_begin) * kThr + threadIdx.x;
    if (t < b.price_tiles) {
        const ServePrice op = op_of<ServePrice>(x);
        if ((g + 1) * kVW <= n) op.template finish<true>(g, op.template load<true>(g));
        else
            for (int64_t i = g * kVW; i < n; ++i) op.scalar(i);
    } else {
        const ServeGreeks op = op_of<ServeGreeks>(x);
        if ((g + 1) * kVW <= n) op.template finish<true>(g, op.template load<true>(g));
        else
            for (int64_t i = g * kVW; i < n; ++i) op.scalar(i);
    }
}

// The fused kernel of section sec with kThr threads per block.
template <int kThr>
const void* serve_fn(int sec) {
    return sec == 0 ? reinterpret_cast<const void*>(&k_serve<ServePrice, 0, kThr>)
                    : reinterpret_cast<const void*>(&k_serve<ServeGreeks, 1, kThr>);
}
const void* serve_fn(int threads, int sec) {
    return threads == 64 ? serve_fn<64>(sec) : threads == 128 ? serve_fn<128>(sec)
                                                                : serve_fn<256>(sec);
}
const void* small_fn(int threads) {
    return threads == 64    ? reinterpret_cast<const void*>(&k_serve_small<64>)
           : threads == 128 ? reinterpret_cast<const void*>(&k_serve_small<128>)
                            : reinterpret_cast<const void*>(&k_serve_small<256>);
}

}  // namespace

// The HIP executor of the serving loop (serve_loop.hpp): descriptor tables,
// the stage and fused kernels, three streams and one event per slot.
struct HipExec {
    // Batches in flight at once: two of the small lane on their own stream,
    // four of the bulk lane alternating over two streams.  While one runs, the
    // next ones are queued behind it, so the GPU stays busy while clients turn
    // finished requests around into new ones; the small lane's batches run
    // beside the bulk lane's instead of behind them.
    static constexpr int kSlots = 6;
    static constexpr int kSmallSlots = 2;

    int device = 0;
    int use_graph = 0;
    int threads = kServeThreads;                // fused kernels' block size
    int64_t tile = kServeThreads * kVW;         // options per tile
    int64_t grid_cap = kMaxGrid;                // blocks per section at most
    char* arena = nullptr;
    hipStream_t stream = nullptr;               // capture stream
    hipStream_t streams[3] = {};                // bulk batches alternate over 0 and 1;
                                                // the small lane's run on 2
    uint8_t* host_slot[kSlots] = {};            // pinned, written by the dispatcher
    uint8_t* host_slot_dev[kSlots] = {};        // the same memory, device address
    uint8_t* dev_slot[kSlots] = {};
    hipGraphExec_t graph[kSlots] = {};
    hipGraph_t graph_src[kSlots] = {};          // kept: its nodes name the exec's nodes
    hipGraphNode_t section_node[kSlots][2] = {};
    unsigned section_grid[kSlots][2] = {};      // grid the exec's section node has now
    void* section_args[kSlots][1] = {};         // kernel arguments: &dev_slot[s]
    hipEvent_t ev[kSlots] = {};
    hipStream_t slot_stream[kSlots] = {};        // the stream slot s was last launched on
    bool in_flight[kSlots] = {};                 // launched and not seen to end (dispatcher only)
    int64_t seq = 0, nlaunch = 0;
    struct Reply {
        std::mutex mu;
        hipStream_t stream = nullptr;
        uint32_t seq = 0;
    } reply[kReplies];
    uint8_t* reply_host = nullptr;              // pinned: kReplies x (kReplyBytes, flag line)
    uint8_t* reply_dev = nullptr;               // the same memory, device address
    uint32_t* reply_count = nullptr;            // device: a counter per reply, zero between uses
    static constexpr size_t kReplySpan = kReplyBytes + 256;

    hipError_t init(int dev, size_t arena_bytes, int graph_on, int grid_blocks, int block_threads) {
        device = dev;
        use_graph = graph_on;
        if (block_threads == 64 || block_threads == 128 || block_threads == 256)
            threads = block_threads;
        tile = (int64_t)threads * kVW;
        hipError_t e = hipSetDevice(device);
        if (e == hipSuccess) e = hipMalloc((void**)&arena, arena_bytes);
        if (e == hipSuccess) e = hipStreamCreateWithFlags(&stream, hipStreamNonBlocking);
        for (int j = 0; j < 3 && e == hipSuccess; ++j)
            e = hipStreamCreateWithFlags(&streams[j], hipStreamNonBlocking);
        for (int s = 0; s < kSlots && e == hipSuccess; ++s) {
            e = hipHostMalloc((void**)&host_slot[s], kSlotBytes, hipHostMallocCoherent);
            if (e == hipSuccess)
                e = hipHostGetDevicePointer((void**)&host_slot_dev[s], host_slot[s], 0);
            if (e == hipSuccess) e = hipMalloc((void**)&dev_slot[s], kSlotBytes);
            if (e == hipSuccess) e = hipEventCreateWithFlags(&ev[s], hipEventDisableTiming);
            if (e == hipSuccess) ::memset(host_slot[s], 0, sizeof(SlotHeader));
        }
        for (int r = 0; r < kReplies && e == hipSuccess; ++r)
            e = hipStreamCreateWithFlags(&reply[r].stream, hipStreamNonBlocking);
        if (e == hipSuccess)
            e = hipHostMalloc((void**)&reply_host, kReplies * kReplySpan, hipHostMallocCoherent);
        if (e == hipSuccess) e = hipHostGetDevicePointer((void**)&reply_dev, reply_host, 0);
        if (e == hipSuccess) e = hipMalloc((void**)&reply_count, kReplies * 256);
        for (int r = 0; r < kReplies && e == hipSuccess; ++r) {
            ::memset(reply_host + r * kReplySpan + kReplyBytes, 0, sizeof(uint32_t));
            // counters 256 bytes apart; a plain store kernel, then done before use
            hipLaunchKernelGGL(k_zero_word, dim3(1), dim3(1), 0, reply[r].stream,
                               reply_count + r * 64);
            e = hipGetLastError();
        }
        if (grid_blocks > 0) grid_cap = std::min<int64_t>(grid_blocks, kMaxGrid);
        for (int s = 0; s < kSlots && e == hipSuccess && use_graph; ++s) e = capture(s);
        return e;
    }
    void release() {
        (void)hipSetDevice(device);
        drain();
        for (int s = 0; s < kSlots; ++s) {
            if (graph[s]) (void)hipGraphExecDestroy(graph[s]);
            if (graph_src[s]) (void)hipGraphDestroy(graph_src[s]);
            if (ev[s]) (void)hipEventDestroy(ev[s]);
            if (host_slot[s]) (void)hipHostFree(host_slot[s]);
            if (dev_slot[s]) (void)hipFree(dev_slot[s]);
        }
        if (stream) (void)hipStreamDestroy(stream);
        for (hipStream_t st : streams)
            if (st) (void)hipStreamDestroy(st);
        for (Reply& r : reply)
            if (r.stream) (void)hipStreamDestroy(r.stream);
        if (reply_host) (void)hipHostFree(reply_host);
        if (reply_count) (void)hipFree(reply_count);
        if (arena) (void)hipFree(arena);
    }

    // Captures slot s as one graph: stage, price section, Greeks section.  The
    // section nodes are found by kernel so each launch can set their grids.
    hipError_t capture(int s) {
        hipGraph_t g = nullptr;
        hipError_t e = hipStreamBeginCapture(stream, hipStreamCaptureModeThreadLocal);
        if (e != hipSuccess) return e;
        hipLaunchKernelGGL(k_stage, dim3(kStageBlocks), dim3(kThreads), 0, stream,
                           reinterpret_cast<const uint4*>(host_slot_dev[s]),
                           reinterpret_cast<uint4*>(dev_slot[s]));
        section_args[s][0] = &dev_slot[s];
        for (int sec = 0; sec < 2; ++sec)
            (void)hipLaunchKernel(serve_fn(threads, sec), dim3(1), dim3(threads), section_args[s],
                                  0, stream);
        e = hipStreamEndCapture(stream, &g);
        if (e != hipSuccess) return e;
        graph_src[s] = g;
        const void* fn[2] = {serve_fn(threads, 0), serve_fn(threads, 1)};
        hipGraphNode_t nodes[3];
        size_t count = 3;
        e = hipGraphGetNodes(g, nodes, &count);
        for (size_t i = 0; i < count && e == hipSuccess; ++i) {
            hipKernelNodeParams p{};
            e = hipGraphKernelNodeGetParams(nodes[i], &p);
            for (int sec = 0; sec < 2 && e == hipSuccess; ++sec)
                if (p.func == fn[sec]) section_node[s][sec] = nodes[i];
        }
        if (e == hipSuccess && (count != 3 || !section_node[s][0] || !section_node[s][1]))
            e = hipErrorInvalidValue;
        if (e == hipSuccess) e = hipGraphInstantiate(&graph[s], g, nullptr, nullptr, 0);
        section_grid[s][0] = section_grid[s][1] = 1;
        return e;
    }

    // Sets section sec of slot s's graph to a grid of `blocks`.
    hipError_t set_section_grid(int s, int sec, unsigned blocks) {
        if (section_grid[s][sec] == blocks) return hipSuccess;
        hipKernelNodeParams p{};
        p.func = const_cast<void*>(serve_fn(threads, sec));
        p.gridDim = dim3(blocks);
        p.blockDim = dim3(threads);
        p.sharedMemBytes = 0;
        p.kernelParams = section_args[s];
        p.extra = nullptr;
        const hipError_t e = hipGraphExecKernelNodeSetParams(graph[s], section_node[s][sec], &p);
        if (e == hipSuccess) section_grid[s][sec] = blocks;
        return e;
    }

    // Fills slot s with the batch's descriptors, price requests first, each
    // section in admission order.  The slot is the dispatcher's own while no
    // batch uses it, so no lock is held.
    void write_slot(int s, const std::vector<serve::Admitted>& reqs) {
        SlotHeader* h = reinterpret_cast<SlotHeader*>(host_slot[s]);
        Desc* d = reinterpret_cast<Desc*>(host_slot[s] + sizeof(SlotHeader));
        int nd[2] = {0, 0};
        for (const serve::Admitted& r : reqs) ++nd[r.kind == serve::kGreeks ? 1 : 0];
        int next[2] = {0, nd[0]};
        int64_t tiles[2] = {0, 0};
        for (const serve::Admitted& r : reqs) {
            const int sec = r.kind == serve::kGreeks ? 1 : 0;
            size_t bo[6], oo[5];
            serve::book_layout(r.book_n, bo);
            serve::output_layout(r.n, r.kind, oo);
            Desc& x = d[next[sec]++];
            for (int j = 0; j < 5; ++j) x.in[j] = reinterpret_cast<const float*>(arena + r.book_off + bo[j]);
            x.type = reinterpret_cast<const uint8_t*>(arena + r.book_off + bo[5]);
            for (int j = 0; j < 5; ++j) x.out[j] = reinterpret_cast<float*>(arena + r.out_off + oo[j]);
            x.n = r.n;
            x.tile_begin = tiles[sec];
            x.kind = r.kind;
            x.pad = 0;
            tiles[sec] += (r.n + tile - 1) / tile;
        }
        h->ndesc[0] = nd[0];
        h->ndesc[1] = nd[1];
        h->tiles[0] = tiles[0];
        h->tiles[1] = tiles[1];
        h->seq = ++seq;
    }

    // ---- the executor interface ----
    void thread_start() { (void)hipSetDevice(device); }

    // Launches slot s on its lane's stream (the bulk lane alternates between
    // two): graph replay, or directly: a small batch with little else in flight
    // as one kernel, any other as the stage kernel and the fused kernel of each
    // non-empty section; each section's grid is one block per tile.  Then
    // records the slot's event.
    int launch(int s, const std::vector<serve::Admitted>& reqs, std::string* err) {
        const int64_t others = std::count(in_flight, in_flight + kSlots, true);
        write_slot(s, reqs);
        hipStream_t st = s < kSmallSlots ? streams[2] : streams[nlaunch++ & 1];
        slot_stream[s] = st;
        const SlotHeader* h = reinterpret_cast<const SlotHeader*>(host_slot[s]);
        const int nd = h->ndesc[0] + h->ndesc[1];
        hipError_t e = hipSuccess;
        if (graph[s]) {
            // an empty section keeps one block, which returns at once
            for (int sec = 0; sec < 2 && e == hipSuccess; ++sec) {
                const int64_t blocks = std::max<int64_t>(1, std::min(h->tiles[sec], grid_cap));
                e = set_section_grid(s, sec, (unsigned)blocks);
            }
            if (e == hipSuccess) e = hipGraphLaunch(graph[s], st);
        } else if (nd <= (others == 0 ? kSmallDesc : others == 1 ? kSmallBeside : 0) &&
                   h->tiles[0] + h->tiles[1] <= std::min(kSmallTiles, grid_cap)) {
            SmallBatch b;
            b.np = h->ndesc[0];
            b.nd = nd;
            b.price_tiles = (int32_t)h->tiles[0];
            b.pad = 0;
            ::memcpy(b.d, host_slot[s] + sizeof(SlotHeader), sizeof(Desc) * (size_t)b.nd);
            for (int i = b.np; i < b.nd; ++i) b.d[i].tile_begin += h->tiles[0];
            void* args[1] = {&b};
            e = hipLaunchKernel(small_fn(threads), dim3((unsigned)(h->tiles[0] + h->tiles[1])),
                                dim3(threads), args, 0, st);
        } else {
            hipLaunchKernelGGL(k_stage, dim3(kStageBlocks), dim3(kThreads), 0, st,
                               reinterpret_cast<const uint4*>(host_slot_dev[s]),
                               reinterpret_cast<uint4*>(dev_slot[s]));
            e = hipGetLastError();
            void* args[1] = {&dev_slot[s]};
            for (int sec = 0; sec < 2 && e == hipSuccess; ++sec)
                if (h->tiles[sec] > 0)
                    e = hipLaunchKernel(serve_fn(threads, sec),
                                        dim3((unsigned)std::min(h->tiles[sec], grid_cap)),
                                        dim3(threads), args, 0, st);
        }
        if (e == hipSuccess) e = hipEventRecord(ev[s], st);
        if (e != hipSuccess) *err = hipGetErrorString(e);
        in_flight[s] = e == hipSuccess;   // a failed launch is quiesced before the next
        return e == hipSuccess ? 0 : -1;
    }
    int query(int s, std::string* err) {
        const hipError_t q = hipEventQuery(ev[s]);
        if (q == hipErrorNotReady) return 0;
        in_flight[s] = false;
        if (q == hipSuccess) return 1;
        *err = hipGetErrorString(q);
        return -1;
    }
    // A launch that failed part-way may have queued the stage kernel or a
    // section on the slot's stream: wait for that stream before the loop frees
    // the batch's outputs and reuses the slot's tables.
    void quiesce(int s) {
        if (slot_stream[s]) (void)hipStreamSynchronize(slot_stream[s]);
    }
    void drain() {
        if (stream) (void)hipStreamSynchronize(stream);
        for (hipStream_t st : streams)
            if (st) (void)hipStreamSynchronize(st);
        for (Reply& r : reply)
            if (r.stream) (void)hipStreamSynchronize(r.stream);
    }

    // Memory the CPU may write directly (what the runtime does not know is the
    // caller's ordinary memory).
    static bool host_memory(const void* p) {
        hipPointerAttribute_t a;
        ::memset(&a, 0, sizeof(a));
        if (hipPointerGetAttributes(&a, p) != hipSuccess) {
            (void)hipGetLastError();
            return true;
        }
        return a.type == hipMemoryTypeHost || a.type == hipMemoryTypeUnregistered;
    }

    // Bytes from one output of a Greeks request to the next.
    static size_t output_stride(size_t bytes) {
        return serve::output_bytes((int64_t)(bytes / 4), serve::kPrice);
    }

    // Copies k of a request's outputs, of `bytes` bytes each, from the arena
    // (src[j], ascending) to dst[j]: through a reply's pinned memory when one is
    // free and they fit it, else by the runtime's copies.
    hipError_t copy_out(void* const* dst, char* const* src, int k, size_t bytes) {
        bool host = k > 0;
        for (int j = 0; j < k; ++j) host = host && host_memory(dst[j]);
        if (host && k * output_stride(bytes) <= kReplyBytes) {
            for (int r = 0; r < kReplies; ++r) {
                std::unique_lock<std::mutex> lk(reply[r].mu, std::try_to_lock);
                if (!lk.owns_lock()) continue;
                return reply_out(r, dst, src, k, bytes);
            }
        }
        hipError_t e = hipSuccess;
        for (int j = 0; j < k && e == hipSuccess; ++j)
            e = hipMemcpy(dst[j], src[j], bytes, hipMemcpyDeviceToHost);
        return e;
    }

    hipError_t reply_out(int r, void* const* dst, char* const* src, int k, size_t bytes) {
        uint8_t* host = reply_host + r * kReplySpan;
        uint8_t* dev = reply_dev + r * kReplySpan;
        const size_t stride = output_stride(bytes);
        const bool joined = (size_t)(src[k - 1] - src[0]) == (size_t)(k - 1) * stride;
        const size_t apart = joined ? stride : (bytes + 7) / 8 * 8;   // in the reply
        const int words = (int)(((joined ? (k - 1) * stride : 0) + bytes + 7) / 8);
        const uint64_t* from = reinterpret_cast<const uint64_t*>(src[0]);
        uint64_t* to = reinterpret_cast<uint64_t*>(dev);
        uint32_t* count = reply_count + r * 64;
        uint32_t* dev_flag = reinterpret_cast<uint32_t*>(dev + kReplyBytes);
        const uint32_t seq = ++reply[r].seq;
        const int blocks = (words + kThreads - 1) / kThreads;
        if (joined) {
            hipLaunchKernelGGL(k_reply, dim3(std::min(blocks, kReplyBlocks)), dim3(kThreads), 0,
                               reply[r].stream, from, to, words, count, dev_flag, seq);
        } else {
            uint32_t order = 0;
            for (int j = 0; j < k; ++j) order |= (uint32_t)((src[j] - src[0]) / stride) << (4 * j);
            hipLaunchKernelGGL(k_reply_rows, dim3(std::min(blocks, kReplyBlocks / k), k),
                               dim3(kThreads), 0, reply[r].stream, from, to, words,
                               (int)(stride / 8), order, count, dev_flag, seq);
        }
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
        const uint32_t* flag = reinterpret_cast<const uint32_t*>(host + kReplyBytes);
        auto arrived = [&] { return __atomic_load_n(flag, __ATOMIC_ACQUIRE) == seq; };
        const int64_t until = serve::steady_ns() + 200000;
        while (!arrived() && serve::steady_ns() < until) __builtin_ia32_pause();
        if (!arrived()) {
            e = hipStreamSynchronize(reply[r].stream);
            if (e != hipSuccess) return e;
            if (!arrived()) return hipErrorUnknown;
        }
        for (int j = 0; j < k; ++j) ::memcpy(dst[j], host + j * apart, bytes);
        return hipSuccess;
    }
};

}  // namespace bs

struct bs_ctx_s {
    bs::HipExec exec;
    bs::serve::Loop<bs::HipExec>* loop = nullptr;
};

using namespace bs;

namespace {

static_assert(serve::kErrBudget == BS_ERR_BUDGET && serve::kErrBusy == BS_ERR_BUSY &&
                  serve::kErrNotFound == BS_ERR_NOT_FOUND && serve::kErrTimeout == BS_ERR_TIMEOUT &&
                  serve::kErrCancelled == BS_ERR_CANCELLED && serve::kErrFailed == BS_ERR_FAILED &&
                  serve::kErrShutdown == BS_ERR_SHUTDOWN && serve::kDone == BS_TICKET_DONE &&
                  serve::kCancelled == BS_TICKET_CANCELLED && serve::kGreeks == BS_REQ_GREEKS,
              "serve_core codes mirror bs_mi355.h");

int status(int rc, const char* what) { return rc == BS_OK ? BS_OK : set_error(rc, what); }

}  // namespace

extern "C" {

int bs_ctx_create(int device, size_t hbm_budget_bytes, const bs_serve_opts* opts, bs_ctx_t* out) {
    return guarded("bs_ctx_create", [&]() -> int {
        if (!out) return set_error(BS_ERR_INVALID, "ctx is NULL");
        *out = nullptr;
        if (hbm_budget_bytes < serve::kAlign * 16)
            return set_error(BS_ERR_INVALID, "hbm_budget_bytes too small");
        int ndev = 0;
        hipError_t e = hipGetDeviceCount(&ndev);
        if (e != hipSuccess || device < 0 || device >= ndev)
            return set_error(BS_ERR_NODEVICE, "device index out of range");
        serve::Limits lim;
        lim.max_batch_requests = kMaxDesc;
        lim.max_batch_options = int64_t(1) << 31;
        lim.small_options = 65536;
        int use_graph = 0, grid_blocks = 0;
        const int block_threads = config().block_threads;
        if (opts) {
            if (opts->small_request_options != 0)
                lim.small_options = opts->small_request_options < 0 ? 0 : opts->small_request_options;
            if (opts->max_batch_requests > 0)
                lim.max_batch_requests = std::min<int64_t>(opts->max_batch_requests, kMaxDesc);
            if (opts->max_batch_options > 0) lim.max_batch_options = opts->max_batch_options;
            use_graph = opts->use_graph;
            grid_blocks = opts->grid_blocks;
        }
        auto* c = new bs_ctx_s();
        e = c->exec.init(device, hbm_budget_bytes, use_graph, grid_blocks, block_threads);
        if (e != hipSuccess) {
            const int rc = hip_error(e, "bs_ctx_create");
            c->exec.release();
            delete c;
            return rc;
        }
        try {
            c->loop = new serve::Loop<HipExec>(&c->exec, hbm_budget_bytes, lim,
                                               opts && opts->completion_queue != 0);
            c->loop->start();
        } catch (...) {   // free the device resources, then report the failure
            delete c->loop;
            c->exec.release();
            delete c;
            throw;
        }
        *out = c;
        return BS_OK;
    });
}

int bs_ctx_destroy(bs_ctx_t ctx) {
    return guarded("bs_ctx_destroy", [&]() -> int {
        bs_ctx_s* c = ctx;
        if (!c) return set_error(BS_ERR_INVALID, "ctx is NULL");
        if (c->loop) c->loop->stop();
        c->exec.release();
        delete c->loop;
        delete c;
        return BS_OK;
    });
}

int bs_book_register(bs_ctx_t ctx, const float* s, const float* k, const float* r, const float* v,
                     const float* t, const uint8_t* otype, int64_t n, bs_book_t* book) {
    return guarded("bs_book_register", [&]() -> int {
        bs_ctx_s* c = ctx;
        if (!c || !book) return set_error(BS_ERR_INVALID, "ctx or book is NULL");
        if (n <= 0) return set_error(BS_ERR_INVALID, "n <= 0");
        if (!s || !k || !r || !v || !t || !otype) return set_error(BS_ERR_INVALID, "NULL array");
        int64_t id;
        size_t off;
        const int rc = c->loop->register_book(n, &id, &off);
        if (rc == BS_ERR_SHUTDOWN) return set_error(rc, "context shutting down");
        if (rc != BS_OK) return set_error(rc, "book does not fit in the arena");
        size_t bo[6];
        serve::book_layout(n, bo);
        const void* src[6] = {s, k, r, v, t, otype};
        hipError_t e = hipSetDevice(c->exec.device);
        for (int j = 0; j < 6 && e == hipSuccess; ++j)
            e = hipMemcpy(c->exec.arena + off + bo[j], src[j], (size_t)n * (j < 5 ? 4 : 1),
                          hipMemcpyHostToDevice);
        // The batches run on non-blocking streams: the book must be in device
        // memory before its id is handed out.
        if (e == hipSuccess) e = hipStreamSynchronize(nullptr);
        if (e != hipSuccess) {
            c->loop->release_book(id);
            return hip_error(e, "bs_book_register");
        }
        *book = id;
        return BS_OK;
    });
}

int bs_book_release(bs_ctx_t ctx, bs_book_t book) {
    return guarded("bs_book_release", [&]() -> int {
        bs_ctx_s* c = ctx;
        if (!c) return set_error(BS_ERR_INVALID, "ctx is NULL");
        return status(c->loop->release_book(book), "bs_book_release");
    });
}

int bs_submit(bs_ctx_t ctx, bs_book_t book, int kind, bs_ticket_t* ticket) {
    return guarded("bs_submit", [&]() -> int {
        bs_ctx_s* c = ctx;
        if (!c || !ticket) return set_error(BS_ERR_INVALID, "ctx or ticket is NULL");
        return status(c->loop->submit(book, kind, ticket), "bs_submit");
    });
}

int bs_submit_many(bs_ctx_t ctx, const bs_book_t* books, const int* kinds, const int64_t* users,
                   int64_t count, bs_ticket_t* tickets) {
    return guarded("bs_submit_many", [&]() -> int {
        bs_ctx_s* c = ctx;
        if (!c) return set_error(BS_ERR_INVALID, "ctx is NULL");
        if (count < 0 || (count > 0 && (!books || !kinds || !tickets)))
            return set_error(BS_ERR_INVALID, "bad request arrays");
        return status(c->loop->submit_many(books, kinds, users, count, tickets), "bs_submit_many");
    });
}

int bs_reap(bs_ctx_t ctx, bs_completion* out, int64_t max, int64_t timeout_us, int64_t* count) {
    return guarded("bs_reap", [&]() -> int {
        static_assert(sizeof(bs_completion) == sizeof(serve::Completion) &&
                          offsetof(bs_completion, user) == offsetof(serve::Completion, user) &&
                          offsetof(bs_completion, state) == offsetof(serve::Completion, state) &&
                          offsetof(bs_completion, done_ns) == offsetof(serve::Completion, t_done),
                      "bs_completion layout");
        bs_ctx_s* c = ctx;
        if (!c || !count) return set_error(BS_ERR_INVALID, "ctx or count is NULL");
        *count = 0;
        if (max < 0 || (max > 0 && !out)) return set_error(BS_ERR_INVALID, "bad output array");
        const int rc = c->loop->reap(reinterpret_cast<serve::Completion*>(out), max, timeout_us, count);
        return rc == BS_OK ? BS_OK : set_error(rc, "context has no completion queue");
    });
}

int bs_result_release_many(bs_ctx_t ctx, const bs_ticket_t* tickets, int64_t count) {
    return guarded("bs_result_release_many", [&]() -> int {
        bs_ctx_s* c = ctx;
        if (!c) return set_error(BS_ERR_INVALID, "ctx is NULL");
        if (count < 0 || (count > 0 && !tickets)) return set_error(BS_ERR_INVALID, "bad ticket array");
        return status(c->loop->release_many(tickets, count), "bs_result_release_many");
    });
}

int bs_poll(bs_ctx_t ctx, bs_ticket_t ticket, int* state) {
    return guarded("bs_poll", [&]() -> int {
        bs_ctx_s* c = ctx;
        if (!c || !state) return set_error(BS_ERR_INVALID, "ctx or state is NULL");
        return status(c->loop->poll(ticket, state), "unknown ticket");
    });
}

int bs_wait(bs_ctx_t ctx, bs_ticket_t ticket, int64_t timeout_us) {
    return guarded("bs_wait", [&]() -> int {
        bs_ctx_s* c = ctx;
        if (!c) return set_error(BS_ERR_INVALID, "ctx is NULL");
        std::string msg;
        const int rc = c->loop->wait(ticket, timeout_us, &msg);
        switch (rc) {
            case BS_OK: return BS_OK;
            case BS_ERR_TIMEOUT: return set_error(rc, "bs_wait timed out");
            case BS_ERR_NOT_FOUND: return set_error(rc, "unknown ticket");
            case BS_ERR_CANCELLED: return set_error(rc, "ticket cancelled");
            default: return set_error(rc, msg);
        }
    });
}

int bs_result_device(bs_ctx_t ctx, bs_ticket_t ticket, const float** price, const float** delta,
                     const float** vega, const float** rho, const float** theta) {
    return guarded("bs_result_device", [&]() -> int {
        bs_ctx_s* c = ctx;
        if (!c) return set_error(BS_ERR_INVALID, "ctx is NULL");
        int64_t n;
        int kind;
        size_t off;
        const int rc = c->loop->result_info(ticket, &n, &kind, &off);
        if (rc == BS_ERR_NOT_FOUND) return set_error(rc, "unknown ticket");
        if (rc != BS_OK) return set_error(rc, "ticket not done");
        size_t oo[5];
        serve::output_layout(n, kind, oo);
        const float** dst[5] = {price, delta, vega, rho, theta};
        for (int j = 0; j < 5; ++j) {
            if (!dst[j]) continue;
            *dst[j] = (j == 0 || kind == serve::kGreeks)
                          ? reinterpret_cast<const float*>(c->exec.arena + off + oo[j])
                          : nullptr;
        }
        return BS_OK;
    });
}

int bs_result_copy(bs_ctx_t ctx, bs_ticket_t ticket, float* price, float* delta, float* vega,
                   float* rho, float* theta) {
    return guarded("bs_result_copy", [&]() -> int {
        bs_ctx_s* c = ctx;
        if (!c) return set_error(BS_ERR_INVALID, "ctx is NULL");
        int64_t n;
        int kind;
        size_t off;
        const int rc = c->loop->result_info(ticket, &n, &kind, &off);
        if (rc == BS_ERR_NOT_FOUND) return set_error(rc, "unknown ticket");
        if (rc != BS_OK) return set_error(rc, "ticket not done");
        size_t oo[5];
        serve::output_layout(n, kind, oo);
        float* want[5] = {price, delta, vega, rho, theta};
        hipError_t e = hipSetDevice(c->exec.device);
        void* dst[5];
        char* src[5];
        int k = 0;
        bool refused = false;   // Greeks asked of a price ticket: after the price is copied
        for (int j = 0; j < 5 && !refused; ++j) {
            if (!want[j]) continue;
            refused = j > 0 && kind != serve::kGreeks;
            if (refused) break;
            dst[k] = want[j];
            src[k++] = c->exec.arena + off + oo[j];
        }
        if (e == hipSuccess) e = c->exec.copy_out(dst, src, k, (size_t)n * 4);
        if (e != hipSuccess) return hip_error(e, "bs_result_copy");
        return refused ? set_error(BS_ERR_INVALID, "not a Greeks ticket") : BS_OK;
    });
}

int bs_result_release(bs_ctx_t ctx, bs_ticket_t ticket) {
    return guarded("bs_result_release", [&]() -> int {
        bs_ctx_s* c = ctx;
        if (!c) return set_error(BS_ERR_INVALID, "ctx is NULL");
        return status(c->loop->release(ticket), "bs_result_release");
    });
}

int bs_cancel(bs_ctx_t ctx, bs_ticket_t ticket) {
    return guarded("bs_cancel", [&]() -> int {
        bs_ctx_s* c = ctx;
        if (!c) return set_error(BS_ERR_INVALID, "ctx is NULL");
        return status(c->loop->cancel(ticket), "bs_cancel: ticket not queued");
    });
}

int bs_ticket_times(bs_ctx_t ctx, bs_ticket_t ticket, int64_t* submit_ns, int64_t* done_ns) {
    return guarded("bs_ticket_times", [&]() -> int {
        bs_ctx_s* c = ctx;
        if (!c) return set_error(BS_ERR_INVALID, "ctx is NULL");
        return status(c->loop->times(ticket, submit_ns, done_ns), "unknown ticket");
    });
}

int bs_ctx_stats(bs_ctx_t ctx, bs_serve_stats* out) {
    return guarded("bs_ctx_stats", [&]() -> int {
        bs_ctx_s* c = ctx;
        if (!c || !out) return set_error(BS_ERR_INVALID, "ctx or stats is NULL");
        serve::Stats st;
        serve::LoopTimes lt;
        size_t cap, used, peak;
        c->loop->stats(&st, &cap, &used, &peak, &lt);
        out->arena_bytes = (int64_t)cap;
        out->arena_used = (int64_t)used;
        out->arena_peak = (int64_t)peak;
        out->books_resident = st.books_resident;
        out->requests_queued = st.requests_queued;
        out->requests_running = st.requests_running;
        out->requests_done = st.requests_done;
        out->requests_failed = st.requests_failed;
        out->requests_cancelled = st.requests_cancelled;
        out->launches = st.launches;
        out->options_priced = st.options_priced;
        out->admission_waits = st.admission_waits;
        out->queue_ns_total = st.queue_ns;
        out->batch_ns_total = lt.batch;
        out->dispatch_admit_ns = lt.admit;
        out->dispatch_launch_ns = lt.launch;
        out->dispatch_retire_ns = lt.retire;
        out->gpu_idle_ns = lt.idle;
        out->idle_launches = lt.idle_launches;
        return BS_OK;
    });
}

}  // extern "C"
