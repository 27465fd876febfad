// plx_reduce.hpp -- block reductions of the Krylov kernels (256-thread blocks).
#pragma once
#include <hip/hip_runtime.h>

namespace plx {

// Block sum of 256 threads (every thread gets it; fixed order): shuffles inside the waves, then the four
// wave sums.
__device__ __forceinline__ double block_sum(double v, double *s) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    __syncthreads();
    if ((threadIdx.x & 63) == 0) s[threadIdx.x >> 6] = v;
    __syncthreads();
    return (s[0] + s[1]) + (s[2] + s[3]);
}

// Sum of n partials by the whole block.
__device__ __forceinline__ double total(const double *__restrict__ part, int n, double *s) {
    double acc = 0.0;
    for (int i = threadIdx.x; i < n; i += 256) acc += part[i];
    return block_sum(acc, s);
}

}  // namespace plx
