// tm_last.h -- the last workgroup of a launch takes over.
//
// A launch whose workgroups hand results to a final step (a reduction, a
// decision) needs no second launch for it: every workgroup stores its results
// and counts itself, and the one that counts last does the step.  The
// hand-over uses no fence: on this part a device-scope fence writes back and
// invalidates the whole L2 of the workgroup's XCD.  Results are stored and
// read with relaxed device-scope atomics, which pass by the caches that are not
// coherent between XCDs; each workgroup waits for its own stores to complete
// (s_waitcnt) before it counts, and the last one reads after its count has
// returned.  Nothing waits for another workgroup.
#pragma once

#include <hip/hip_runtime.h>

namespace tmh {

template <class T>
__device__ __forceinline__ void put(T* a, T v)
{
    __hip_atomic_store(a, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <class T>
__device__ __forceinline__ T get(const T* a)
{
    return __hip_atomic_load(a, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// true for every thread of the last of `blocks` workgroups; the counter is
// left at zero for the next launch
__device__ __forceinline__ bool last_block(unsigned* counter, unsigned blocks)
{
    __shared__ int s_last;
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");    // this wave's stores have completed
    __syncthreads();
    if (threadIdx.x == 0) {
        const unsigned c = __hip_atomic_fetch_add(counter, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        s_last = c + 1 == blocks;
        if (s_last) put(counter, 0u);
    }
    __syncthreads();
    return s_last != 0;
}

// The same for launches of many workgroups, in two stages: a counter for each
// eighth of them (consecutive workgroups: an eighth runs on one XCD) and one
// for the eighths, each on a line of its own, so that no more than blocks / 8
// atomics meet on one address.  blocks: a multiple of 8; counters: kLastCounters
// zeros, left at zero.
constexpr int kLastStride = 32;
constexpr int kLastCounters = 9 * kLastStride;
__device__ __forceinline__ bool last_block_of_many(unsigned* counters, int lb, int blocks)
{
    __shared__ int s_last;
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");    // this wave's stores have completed
    __syncthreads();
    if (threadIdx.x == 0) {
        const int part = blocks / 8;
        unsigned* own = counters + kLastStride * (1 + lb / part);
        s_last = 0;
        if (__hip_atomic_fetch_add(own, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1 == (unsigned)part) {
            put(own, 0u);
            if (__hip_atomic_fetch_add(counters, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == 7u) {
                put(counters, 0u);
                s_last = 1;
            }
        }
    }
    __syncthreads();
    return s_last != 0;
}

}    // namespace tmh
