// Colour leaves on the device: what the resolver and the edit passes share of reading one
// (variable_weight_size_colors.h:343-413).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace hd {

// fields of a block header's low word: the block's first colour within its macro block, and the
// bits per weight (0: one colour without weights)
__device__ __forceinline__ uint32_t hdr_index(uint32_t h) { return h & 16383u; }
__device__ __forceinline__ uint32_t hdr_bpw(uint32_t h) { return (h >> 16) == 0xFFFFu ? 0u : ((h >> 14) & 3u) + 1u; }

// The block of blocks[lo .. hi] that holds colour `local` of its macro block: the last one that
// starts at or before it (block starts ascend and differ; the first starts at 0), and its
// position. Bound by the chain of loads: three probes a step in flight together make it half as
// long as a binary search's.
__device__ __forceinline__ uint64_t block_of(const uint64_t* __restrict__ blocks, uint32_t lo, uint32_t hi,
                                             uint32_t local, uint32_t& at) {
    uint64_t blk = blocks[lo];
    while (lo < hi) {
        const uint32_t len = hi - lo + 1;
        const uint32_t p1 = lo + max(len / 4, 1u), p2 = min(lo + max(len / 2, 1u), hi), p3 = min(p2 + max(len / 4, 1u), hi);
        const uint64_t b1 = blocks[p1], b2 = blocks[p2], b3 = blocks[p3];
        if (hdr_index((uint32_t)b3) <= local) {
            lo = p3;
            blk = b3;
        } else if (hdr_index((uint32_t)b2) <= local) {
            lo = p2;
            blk = b2;
            hi = p3 - 1;
        } else if (hdr_index((uint32_t)b1) <= local) {
            lo = p1;
            blk = b1;
            hi = p2 - 1;
        } else {
            hi = p1 - 1;
        }
    }
    at = lo;
    return blk;
}

}  // namespace hd
