// fragments.hpp -- what an entry leaves for the sort (gfx950): its cell key or sort word, its winding change
// and its bucket's count.  Shared by the curve pass and the chain passes.
#pragma once

#include "device_common.hpp"
#include "kernels.hpp"

namespace spr {

// An entry's fragment outputs; returns its global bucket.  Frames with narrow sort words store the
// bucket (in key) and the narrow word (bucket inside the path, x + 2 or 0 in the off-canvas
// bucket, winding change + 1), which is all their scatter needs; the others store the key, the
// winding change and the path.
__device__ inline uint32_t store_fragment(const FragArgs& A, int64_t i, uint32_t yx, int swn, uint32_t path,
                                          uint32_t bb, int2 pr) {
    const uint32_t loc = bucket_local((int32_t)yx, pr, A.err);
    const uint32_t bucket = bb + loc;
    if (A.nword) {
        const uint32_t xl = loc == (uint32_t)pr.y ? 0u : (yx & 0xFFFFu) - kNarrowX0;
        A.key[i] = (int32_t)bucket;
        A.nword[i] = (loc << 17) | (xl << 2) | (uint32_t)(swn + 1);
    } else {
        A.key[i] = (int32_t)yx;
        A.wn[i] = (int8_t)swn;
        A.epath[i] = path;
    }
    return bucket;
}

// An entry without a segment (counted but not written: the two passes round differently far outside any
// canvas): the off-canvas cell, no winding change.  Every counted entry gets a bucket, since the scatter takes
// whatever is there as an index.
__device__ inline void store_gap(const FragArgs& A, int64_t i, int curve, uint32_t path, uint32_t bb, int2 pr) {
    const uint32_t bucket = store_fragment(A, i, kSentinelKey, 0, path, bb, pr);
    atomicAdd(&A.hist[bucket], 1);
    if (A.inter) A.inter[i] = make_int2(curve, 0);
    if (A.chord) A.chord[i] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
}

}  // namespace spr
