// Work lists of slices (slices.h).
#include "slices.h"

namespace pcvl {

// Exclusive prefix of the slice counts, one block: slice0[b], total at
// slice0[B].  4096 counts per pass, four consecutive ones per thread (their
// loads in flight together); a shuffle scan of the thread sums per wave and
// the 16 wave totals through LDS.
__global__ void __launch_bounds__(1024) slice_scan_kernel(const int32_t *__restrict__ nslices, int64_t B,
                                                        int64_t *__restrict__ slice0)
{
    __shared__ int wsum[16];
    const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
    int64_t carry = 0;
    for (int64_t base = 0; base < B; base += 4096) {
        const int64_t i0 = base + 4 * (int64_t)t;
        int v[4];
#pragma unroll
        for (int q = 0; q < 4; q++) v[q] = i0 + q < B ? nslices[i0 + q] : 0;   // below 2^16 each
        const int own = v[0] + v[1] + v[2] + v[3];
        int x = own;
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
            const int y = __shfl_up(x, off, 64);
            if (lane >= off) x += y;
        }
        if (lane == 63) wsum[wv] = x;
        __syncthreads();
        int before = 0, total = 0;
#pragma unroll
        for (int k = 0; k < 16; k++) {
            const int w = wsum[k];
            if (k < wv) before += w;
            total += w;
        }
        int64_t run = carry + before + x - own;
#pragma unroll
        for (int q = 0; q < 4; q++) {
            if (i0 + q < B) slice0[i0 + q] = run;
            run += v[q];
        }
        carry += total;
        __syncthreads();   // wsum is rewritten by the next pass
    }
    if (t == 0) slice0[B] = carry;
}

// Owner of every slice, packed so that a wave finds its slice's item with one
// load.
__global__ void slice_owner_kernel(const int64_t *__restrict__ slice0, int64_t B, uint64_t *__restrict__ owner)
{
    const int64_t b = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (b >= B) return;
    const int64_t g0 = slice0[b], g1 = slice0[b + 1];
    for (int64_t g = g0; g < g1; g++) owner[g] = ((uint64_t)b << SLICE_BITS) | (uint64_t)(g - g0);
}

int launch_slice_owners(const int32_t *nslices, int64_t B, int64_t *slice0, uint64_t *owner, hipStream_t stream)
{
    hipLaunchKernelGGL(slice_scan_kernel, dim3(1), dim3(1024), 0, stream, nslices, B, slice0);
    PCVL_HIP_CHECK(hipGetLastError());
    hipLaunchKernelGGL(slice_owner_kernel, dim3((unsigned)((B + 255) / 256)), dim3(256), 0, stream, slice0, B, owner);
    PCVL_HIP_CHECK(hipGetLastError());
    return OK;
}

} // namespace pcvl
