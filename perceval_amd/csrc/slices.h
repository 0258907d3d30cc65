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

} // namespace pcvl
