// bs_arrive.hpp -- results handed from many blocks to the last of them, and
// from a kernel to a spinning host thread, without fences.
//
// A block stores its result with relaxed agent-scope (or system-scope) stores,
// which write through to memory past the L2 of the block's die, waits for
// their acknowledgement and counts itself in with a relaxed add at the same
// scope; the block that counts last loads the results at that scope.  A release
// fence in place of the wait would write back the die's whole L2 for every
// block.  Counters of different groups belong on lines of their own: adds from
// all dies to one line take turns, about 25 ns each.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace bs {

template <class T>
__device__ __forceinline__ T agent_load(const T* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <class T>
__device__ __forceinline__ void agent_store(T* p, T v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <class T>
__device__ __forceinline__ void system_store(T* p, T v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// Waits until this wave's stores have been acknowledged.
__device__ __forceinline__ void stores_done() {
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    __builtin_amdgcn_s_waitcnt(0);
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
}

// Counts the caller in; true for the one that makes `full`.
__device__ __forceinline__ bool arrive_one(uint32_t* counter, uint32_t full) {
    const uint32_t before =
        __hip_atomic_fetch_add(counter, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    return before == full - 1;
}

// The same for a whole wave, counted once.
__device__ __forceinline__ bool arrive(uint32_t* counter, uint32_t full) {
    int last = 0;
    if ((threadIdx.x & 63) == 0) last = arrive_one(counter, full);
    return __builtin_amdgcn_readfirstlane(last) != 0;
}

}  // namespace bs
