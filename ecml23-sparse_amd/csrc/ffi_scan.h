// Prefix sum over a workgroup.
#ifndef FFI_SCAN_H
#define FFI_SCAN_H

#include <hip/hip_runtime.h>

namespace ffi {

#if defined(__HIPCC__)
// The sum of `v` over the threads below this one, and over all THREADS of them in *total; THREADS a multiple of 64.  Called by the
// whole workgroup; a barrier comes between two calls of it.
template <int THREADS>
__device__ __forceinline__ unsigned long long block_sum_below(unsigned long long v, unsigned long long* total) {
    __shared__ unsigned long long of_wave[THREADS / 64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    unsigned long long upto = v;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const unsigned long long below = __shfl_up(upto, off, 64);
        if (lane >= off) upto += below;
    }
    if (lane == 63) of_wave[wave] = upto;
    __syncthreads();
    unsigned long long before = 0, all = 0;
#pragma unroll
    for (int i = 0; i < THREADS / 64; ++i) {
        if (i < wave) before += of_wave[i];
        all += of_wave[i];
    }
    *total = all;
    return before + upto - v;
}
#endif

}  // namespace ffi

#endif  // FFI_SCAN_H
