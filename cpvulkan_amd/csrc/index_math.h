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

// Whether a texture level's texels may be read without a bounds test: its
// wrapped coordinates lie inside whatever the coordinate, and every texel's
// offset fits 32 bits.  MIRRORED_REPEAT sums two remainders by twice the
// extent, which pass 2^31 for extents above 2^29, so wider levels keep the
// test; so does an empty one.
CPV_INDEX bool plain_extent(uint32_t w, uint32_t h)
{
    return (uint64_t)w * h - 1ull < (1ull << 30) && w <= (1u << 29) && h <= (1u << 29);
}

// wrap (CPVulkan/ImageSampler.cpp:12-38)
CPV_INDEX int32_t wrap_coord(int32_t v, int32_t size, int32_t mode)
{
    if (mode == 0) {                                                       // REPEAT: (v % size + size) % size
        if ((size & (size - 1)) == 0) return v & (size - 1);               // no division for sizes 2^k
        const int32_t m = v % size;
        return m < 0 ? m + size : m;
    }
    if (mode == 1) {                                                       // MIRRORED_REPEAT
        const int32_t two = 2 * size;
        const int32_t n = (v % two + two) % two - size;
        return size - 1 - (n >= 0 ? n : -(1 + n));
    }
    if (mode == 2) return v < 0 ? 0 : (v > size - 1 ? size - 1 : v);       // CLAMP_TO_EDGE
    if (mode == 3) return v < -1 ? -1 : (v > size ? size : v);             // CLAMP_TO_BORDER
    const int32_t m = v >= 0 ? v : -(1 + v);                               // MIRROR_CLAMP_TO_EDGE
    return m < 0 ? 0 : (m > size - 1 ? size - 1 : m);
}

// Whether a tile with a list of n pairs is split among waves that take one of
// its blocks each, in a launch whose tiles have `waves` waves each.
//
// A wave that holds many blocks walks a long tile's list once for all of them,
// one after the other: a serial chain that the launch may end up waiting for.
// But each block's own walk reads the list again, so tiles are split only
// where such a chain would be longer than the rest: with lists much alike
// (none beyond twice the mean of the tiles that have any) a launch of enough
// waves to fill the chip (kEvenWaves, one and a half for each SIMD) splits
// none, and one of fewer waves every tile that is long at all.
// us a frame, all split against none, for soups of 80 to 120 triangles a 16x16
// tile: one wave for 16x16 tiles 329 against 385 with 1,200 waves (640x480),
// 727 against 478 with 3,600 (1280x720); one wave for 32x32 tiles 631 against
// 1,806 with 300 waves, 1,485 against 1,923 with 920, 4,160 against 2,869 with
// 2,040 (1920x1080); four waves for 32x32 tiles 276 against 471 with 1,200,
// 1,598 against 1,460 with 8,160.  Clustered soups, whose lists differ: 1M
// triangles at 1080p 2,260 against 4,189 (16x16, one wave) and 4,836 against
// 17,331 (32x32, one wave).
constexpr uint32_t kEvenWaves = 1536u;
CPV_INDEX bool splits_tile(const LongTiles& l, uint32_t n, uint32_t waves)
{
    return n >= l.from && ((uint64_t)l.filled * waves < kEvenWaves || (uint64_t)n * l.filled >= 2ull * l.pairs);
}

}  // namespace cpv
