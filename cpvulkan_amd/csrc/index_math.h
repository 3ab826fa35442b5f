// Index arithmetic of the kernels at the ends of its ranges: plain integer
// functions that the host can run too (tests/test_index_math.py does).
#pragma once

#include "cpv_types.h"

#if defined(__HIP__) || defined(__HIPCC_RTC__)
#define CPV_INDEX __host__ __device__ __forceinline__
#else
#define CPV_INDEX inline
#endif

namespace cpv {

// The radix sort cuts n items into kSortSegments contiguous segments, one
// per workgroup, which walks its segment in tiles of kSortTile items.
constexpr int kSortSegments = 1024;
constexpr int kSortTile = 2048;

// Segment seg of n items is [b, e).  The segments' common length is taken in
// 64 bits: in 32 a total near 2^32 - 1, which launches may have, wraps it or
// the last segment's end, and that segment's items were neither counted nor
// scattered.
CPV_INDEX void segment_range(uint32_t n, uint32_t seg, uint32_t& b, uint32_t& e)
{
    const uint64_t per = (((uint64_t)n + kSortSegments - 1) / kSortSegments + 63u) & ~63ull;
    const uint64_t first = seg * per, last = first + per;
    b = first < n ? (uint32_t)first : n;
    e = last < n ? (uint32_t)last : n;
}

// Items of the tile that starts at t0 < e of a segment that ends at e.  The
// walk adds this, not kSortTile, which would wrap past a segment's end near
// 2^32; items are told from what lies beyond by their offset in the tile.
CPV_INDEX uint32_t tile_items(uint32_t t0, uint32_t e) { return e - t0 < (uint32_t)kSortTile ? e - t0 : (uint32_t)kSortTile; }

}  // namespace cpv
