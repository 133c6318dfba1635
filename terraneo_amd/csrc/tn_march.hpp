// Pieces of the atomic-free lateral march over the hex cells of a diamond
// (kernels_eps_march.hip) that other column kernels share.  Device-only header.
#pragma once

#include "tn_cell.hpp"
#include "tn_eps_march.hpp"

namespace tn {
namespace march {

// first column of run `b` when `total` columns are split over `blocks` runs
// (run lengths differ by at most one)
__host__ __device__ inline int run_begin(int total, int b, int blocks)
{
    return (int)((int64_t)total * b / blocks);
}

// Point-to-point hand-off between neighbouring waves through LDS counters
// instead of a block barrier per step: the waves of a SIMD drift apart and hide
// each other's memory latency.  The waves of a workgroup are co-resident and
// every wave posts both counters at every step, so each wait is satisfied
// after at most RING - 1 steps of a neighbour; the bound (g.limit polls, by
// default 2^20, about 40 ms at 2.4 GHz) only guarantees that a wait ends
// whatever happens.  A wait that gives up flags it in the host-visible word
// g.fail (a vector store; the host turns it into an error).
__device__ __forceinline__ void wait_counter(int* c, int target, const MarchGuard& g)
{
    for (int i = 0; i < g.limit; ++i) {
        if (__hip_atomic_load(c, __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_WORKGROUP) >= target) return;
        __builtin_amdgcn_s_sleep(1);
    }
    if (__hip_atomic_load(c, __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_WORKGROUP) >= target) return;
    if (g.fail) __hip_atomic_store(g.fail, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

__device__ __forceinline__ void post_counter(int* c, int value, int lane)
{
    if (lane == 0) __hip_atomic_store(c, value, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_WORKGROUP);
}

}  // namespace march
}  // namespace tn
