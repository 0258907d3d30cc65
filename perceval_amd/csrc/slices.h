// Work lists of slices: every item of a batch is cut into a number of slices,
// and persistent waves pull slices of any item from one cursor.
#pragma once

#include "common.h"

namespace pcvl {

// Owner word of a slice: its item and its index in the item.
constexpr int SLICE_BITS = 16;   // at most 2^16 - 1 slices per item

__device__ __forceinline__ void slice_owner(uint64_t own, int64_t &item, int &slice)
{
    // wave-uniform, said so that addresses derived from it live in SGPRs
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)own);
    const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(own >> 32));
    const uint64_t v = ((uint64_t)hi << 32) | lo;
    item = (int64_t)(v >> SLICE_BITS);
    slice = (int)(v & ((1u << SLICE_BITS) - 1));
}

// slice0[b] = slices before item b (slice0[B]: all of them) and the owner word
// of every slice, from the B slice counts.  Two launches on `stream`.
int launch_slice_owners(const int32_t *nslices, int64_t B, int64_t *slice0, uint64_t *owner, hipStream_t stream);

// The slices of a wave (one-wave workgroups): up to 8 consecutive ones at a
// time, the first without a pull, so that the cursor, one address for the whole
// chip at 12..20 ns a pull, is not what short slices wait for, and a wave that
// stays with one owner keeps its rows in LDS.  Fewer at a time towards the end
// (a wave's 16th part of what is left, down to one): with 8 to the end, the
// last slices of 10^5 permanents of order 20 cost 3% of the 47 ms.  Chains of
// 20,000 proposals, 20 photons in 20 modes 6.46 -> 4.43 ms (18 in 24, 15,119:
// 2.73 -> 2.37; 20 in 60, 10^5: 45.8 -> 45.4), sampling 20,000 of 20 photons in
// 60 modes 34.3 -> 33.0 ms.
// The state is in LDS: in registers it would be live through the slice loops,
// whose scalar registers are full.
struct SliceQueue {
    struct State {
        int64_t total, g, end;
        int64_t first;   // slices that are not pulled
    };
    State &q;

    __device__ __forceinline__ int64_t take(int64_t left) const
    {
        const int64_t fit = left / (16 * (int64_t)gridDim.x);
        return fit < 1 ? 1 : fit > 8 ? 8 : fit;
    }

    __device__ __forceinline__ SliceQueue(State &shared, int64_t slices) : q(shared)
    {
        const int64_t per = take(slices);
        if (threadIdx.x == 0) q = State{slices, (int64_t)blockIdx.x * per, ((int64_t)blockIdx.x + 1) * per, (int64_t)gridDim.x * per};
        __syncthreads();
    }

    // The next slice, or -1 after the last one.
    __device__ __forceinline__ int64_t next(unsigned long long *cursor)
    {
        if (threadIdx.x == 0 && q.g == q.end) {
            const int64_t per = take(q.total - q.g);
            q.g = q.first + (int64_t)atomicAdd(cursor, (unsigned long long)per);
            q.end = q.g + per;
        }
        __syncthreads();
        const uint64_t v = (uint64_t)(q.g < q.total ? q.g : -1);
        const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v), hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
        __syncthreads();
        if (threadIdx.x == 0) q.g++;
        return (int64_t)(((uint64_t)hi << 32) | lo);
    }
};

} // namespace pcvl
