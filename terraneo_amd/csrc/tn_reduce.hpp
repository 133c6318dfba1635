// Block reductions shared by the kernel files.  Device-only header.
#pragma once

#include <hip/hip_runtime.h>

namespace tn {

__device__ inline double wave_sum(double v)
{
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    return v;
}

// Block total of `v`, valid in thread 0 (no atomics).
__device__ inline double block_total(double v)
{
    __shared__ double part[16];
    v = wave_sum(v);
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    if (lane == 0) part[wv] = v;
    __syncthreads();
    double s = 0.0;
    if (wv == 0) {
        const int nw = blockDim.x >> 6;
        s = lane < nw ? part[lane] : 0.0;
        s = wave_sum(s);
    }
    __syncthreads();
    return s;
}

// The block's total of `v` into part[blockIdx.x].  Reductions leave one
// partial per block and k_reduce_finalize adds them in a fixed order, so a
// reduction gives the same bits on every run (no floating-point atomics).
__device__ inline void block_partial(double v, double* __restrict__ part)
{
    const double t = block_total(v);
    if (threadIdx.x == 0) part[blockIdx.x] = t;
}

// The sum of nblk partial sums, the same bits in every thread of every block: a
// kernel that needs a preceding reduction's result adds the partials itself
// instead of waiting for one more launch.
__device__ inline double partials_total(const double* __restrict__ part, int nblk)
{
    __shared__ double wsum[16];
    double s = 0.0;
    for (int b = threadIdx.x; b < nblk; b += blockDim.x) s += part[b];
    s = wave_sum(s);
    const int lane = threadIdx.x & 63;
    if (lane == 0) wsum[threadIdx.x >> 6] = s;
    __syncthreads();
    return wave_sum(lane < (int)(blockDim.x >> 6) ? wsum[lane] : 0.0);
}

}  // namespace tn
