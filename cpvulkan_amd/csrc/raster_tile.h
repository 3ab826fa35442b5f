// Fine raster / fragment kernel.
//
// Work unit: one wavefront owns BPW 8x8 pixel blocks of one tile and walks
// that tile's primitive list in submission order.  Wavefronts never
// synchronise with each other: the framebuffer pixels live in registers for
// the whole tile (loaded or cleared at the start, stored at the end), the
// primitive records are read with scalar loads (one record serves all 64
// lanes), and the per-chunk filter reads bounding boxes with vector gathers.
//
// Per primitive and pixel the reference's order of operations is kept
// (CPVulkan/CommandBuffer.Draw.cpp:874-954, 1300-1313 and
// LLVMRuntime/PipelineCompiler.cpp:1020-1085); the shortcuts taken are
// exact: hierarchical depth culling and the per-fragment early depth
// rejection use proven error bounds, and the colour work of passing
// fragments is queued and drained in order per pixel.
#pragma once
#pragma clang fp contract(off)

namespace cpv {

// A wave-uniform record through the constant address space, which lets the
// compiler use scalar loads (the records are read-only during the kernel).
__device__ __forceinline__ void load_record_uniform(const TriSetup* recs, uint32_t gp, TriSetup& r)
{
    uint32_t* dst = (uint32_t*)&r;
#if defined(__HIP_DEVICE_COMPILE__)
    typedef const __attribute__((address_space(4))) uint32_t* ScalarU32Ptr;
    ScalarU32Ptr p = (ScalarU32Ptr)(recs + gp);
#else
    const uint32_t* p = (const uint32_t*)(recs + gp);
#endif
#pragma unroll
    for (int q = 0; q < 32; q++) dst[q] = p[q];
}

__device__ __forceinline__ void load_pixel(const uint8_t* p, int bytes, uint32_t w[4])
{
    w[0] = w[1] = w[2] = w[3] = 0u;
    if (bytes == 4) {
        w[0] = *(const uint32_t*)p;
    } else if (bytes == 2) {
        w[0] = *(const uint16_t*)p;
    } else if (bytes == 8) {
        const uint2 v = *(const uint2*)p;
        w[0] = v.x; w[1] = v.y;
    } else if (bytes == 16) {
        const uint4 v = *(const uint4*)p;
        w[0] = v.x; w[1] = v.y; w[2] = v.z; w[3] = v.w;
    } else {
        // unrolled over the largest pixel so w[] keeps constant indices (registers)
#pragma unroll
        for (int b = 0; b < 16; b++)
            if (b < bytes) w[b >> 2] |= (uint32_t)p[b] << ((b & 3) * 8);
    }
}

__device__ __forceinline__ void store_pixel(uint8_t* p, int bytes, const uint32_t w[4])
{
    if (bytes == 4) {
        *(uint32_t*)p = w[0];
    } else if (bytes == 2) {
        *(uint16_t*)p = (uint16_t)w[0];
    } else if (bytes == 8) {
        *(uint2*)p = make_uint2(w[0], w[1]);
    } else if (bytes == 16) {
        *(uint4*)p = make_uint4(w[0], w[1], w[2], w[3]);
    } else {
#pragma unroll
        for (int b = 0; b < 16; b++)
            if (b < bytes) p[b] = (uint8_t)(w[b >> 2] >> ((b & 3) * 8));
    }
}

// Resident wavefronts per SIMD the raster kernel is compiled for: the
// kernel is latency bound, and more resident waves hide more of it until
// the register budget (512 / waves VGPRs) forces spills.  A fragment shader
// may set kWavesPerEU; measured on MI355X: 6 for the colour shaders, 5 for
// the textured Lambert shader (the default).
template <class FS, class = void>
struct RasterWavesPerEU {
    static constexpr int value = 5;
};
template <class FS>
struct RasterWavesPerEU<FS, decltype((void)FS::kWavesPerEU)> {
    static constexpr int value = FS::kWavesPerEU;
};

// The target applies when a lane holds one 8x8 block's pixel (8x8 tiles,
// or 16x16 tiles with four waves); a lane holding several blocks' pixels
// needs the registers of the compiler's default budget.
template <class FS, int TILE, int WAVES>
constexpr int raster_waves_per_eu()
{
    return (TILE / 8) * (TILE / 8) / WAVES == 1 ? RasterWavesPerEU<FS>::value : 1;
}


// Orders one wave's LDS writes before its lanes read each other's words.
__device__ __forceinline__ void wave_lds_fence()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// The lanes (all of the wave active) that hold a true predicate, as a scalar
// mask, and back.  The primitive walk keeps its lane tests in such masks:
// a comparison writes one directly, they combine by scalar instructions, and
// an empty one is a scalar branch.
__device__ __forceinline__ uint64_t lanes(bool p)
{
#if defined(__HIP_DEVICE_COMPILE__)
    return __builtin_amdgcn_ballot_w64(p);
#else
    return p ? 1u : 0u;
#endif
}
__device__ __forceinline__ bool in_lanes(uint64_t m)
{
#if defined(__HIP_DEVICE_COMPILE__)
    // programs are also compiled at run time, by the hiprtc that the process
    // has loaded: an older one (PyTorch's wheels bring ROCm 7.0's) does not
    // know the builtin
#if __has_builtin(__builtin_amdgcn_inverse_ballot_w64)
    return __builtin_amdgcn_inverse_ballot_w64(m);
#else
    uint32_t bit;
    __asm__("v_cndmask_b32_e64 %0, 0, 1, %1" : "=v"(bit) : "s"(m));
    return bit != 0u;
#endif
#else
    return m != 0;
#endif
}

// An upper bound of the values of a wave's 64 lanes (all active) from row
// shifts and row broadcasts by DPP on the floats' ordered integer images:
// their largest, or a NaN (which no comparison below takes for a rejection)
// when a lane holds a positive one.  Six vector instructions, where a tree
// of __shfl_xor is six dependent trips through the LDS pipe for every chunk
// of the primitive walk, and fmaxf adds a canonicalising instruction to each.
__device__ __forceinline__ float wave_max(float f)
{
#if defined(__HIP_DEVICE_COMPILE__)
    int32_t v = __builtin_bit_cast(int32_t, f);
    v ^= (v >> 31) & 0x7FFFFFFF;
#define CPV_DPP_MAX(ctrl) v = max(v, __builtin_amdgcn_update_dpp((int32_t)0x80000000, v, ctrl, 0xF, 0xF, false))
    CPV_DPP_MAX(0x111);   // row_shr:1
    CPV_DPP_MAX(0x112);   // row_shr:2
    CPV_DPP_MAX(0x114);   // row_shr:4
    CPV_DPP_MAX(0x118);   // row_shr:8
    CPV_DPP_MAX(0x142);   // row_bcast:15
    CPV_DPP_MAX(0x143);   // row_bcast:31
#undef CPV_DPP_MAX
    v = __builtin_amdgcn_readlane(v, 63);
    v ^= (v >> 31) & 0x7FFFFFFF;
    return __builtin_bit_cast(float, v);
#else
    return f;
#endif
}

// LDS of a workgroup: the lanes' queues of shading work and each wave's ring
// of candidate pairs.
template <class FS, int TILE, int WAVES>
struct RasterStage {
    static constexpr int kQueue = FS::kMayDiscard ? 1 : 4;   // a power of two
    static constexpr int kRing = TILE == 8 ? 1 : 512;        // a power of two, at least 63 + 256
    float4 q[FS::kMayDiscard ? 1 : WAVES][kQueue][64];
    uint32_t ring[WAVES][kRing];
};

// True when a triangle's depth (weights q_i = e_i / area to within 2 ulps,
// z_i >= 0, kPrimFast) surely fails LESS and LESS_OR_EQUAL against `cur`.
// The reference's depth is the rounded sum of z_i * w_i, w_i = e_i / area
// correctly rounded; it lies within 4.1u S of the real sum D of z_i e_i / area,
// S = sum |z_i e_i / area| (e_i >= 0 on covered pixels, so S = D), u = 2^-24,
// and the fused sum below, whose weights err by 2u and which rounds three
// times, within 5.1u S, both to 2^-122 where products are subnormal (z_i <=
// 2^20).  So the depth is at least da (1 - 2^-19) - 2^-120, with a factor of
// three to spare for the roundings of that expression.  With kPrimFast's
// ranges nothing overflows; a NaN edge makes the comparison false.
__device__ __forceinline__ bool depth_surely_not_less(float cur, float q0, float q1, float q2, const TriSetup& r)
{
    const float da = fmaf(r.z[2], q2, fmaf(r.z[1], q1, r.z[0] * q0));
    return fmaf(da, 1.0f - 0x1p-19f, -0x1p-120f) > cur;
}

// e / area correctly rounded, from q = fl(e * rinv), rinv = fl(1 / area):
// two Newton steps with exact fma residuals (Markstein, "Computation of
// elementary functions on the IBM RISC System/6000 processor", 1990: when q
// is within an ulp of the quotient and rinv is the rounded reciprocal, the
// fma q + rinv * (e - area q) rounds correctly; q = fl(e rinv) is within 1.5
// ulps, one step brings it within an ulp).  For area in [2^-60, 2^60] and e
// in [2^-60, 2^43] no step leaves the normal range and the residual is exact.
// Four instructions beside the product that the depth test shares, where a
// division takes ten, one of them a quarter-rate reciprocal.
__device__ __forceinline__ float divide_exact(float e, float area, float rinv, float q)
{
    q = fmaf(fmaf(-area, q, e), rinv, q);
    return fmaf(fmaf(-area, q, e), rinv, q);
}

// The kernel body.  Launches whose every draw tests depth with LESS or
// LESS_OR_EQUAL alone (less_depth) take short depth tests: one comparison
// each for the intervals and the estimate, two for the fragment.  The branch
// is wave-uniform, and one body serves every launch: a second copy for the
// op as a template constant raised the register demand past the budget
// (24 bytes per lane spilled) and doubled the code.
template <class FS, int TILE, int WAVES, bool ANYPRIM, bool FIXED>
__device__ __forceinline__ void raster_body(const RasterArgs& a, RasterStage<FS, TILE, WAVES>& stage_area)
{
    constexpr int BW = TILE / 8;               // 8x8 blocks per tile row
    constexpr int BLOCKS = BW * BW;
    constexpr int BPW = BLOCKS / WAVES;        // blocks (pixels) per lane
    static_assert(BLOCKS % WAVES == 0, "tile blocks must divide among the waves");

    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    const uint32_t home = blockIdx.x % kRasterQueues;
    // Pairs that outgrew their arrays were dropped: the launch draws nothing
    // and leaves the attachments as they were, so that it can be run again
    // with larger arrays.
    if (*a.overflow) return;

    // Each survivor's record is read with scalar loads.  Staging the visit
    // fields of a chunk's candidates through LDS (global_load_lds) where a wave
    // holds several blocks, as this kernel did, took 6 KB a wave, which with
    // one block's ring and queue left a CU 13 waves: without it the 48-job
    // batch went from 1,764 to 1,373 us a submit with 16x16 tiles and two
    // waves, from 2,040 to 1,776 with one, and with 32x32 tiles and four waves
    // from 2,359 to 1,873.
    // candidates between two depth tests of a chunk's remaining ones, and the
    // fewest whose depths are bounded over the wave's block
    constexpr int kCullLanes = 16, kCullVisits = 5, kRefineCandidates = 2;
    // block-local depth bounds of triangles, where a lane holds one pixel
    // of an 8x8 block (lane = row * 8 + column)
    constexpr bool BLOCK_DEPTH = !ANYPRIM && BPW == 1;
    // the hierarchical depth op (-1: no hierarchical culling)
    const int32_t hiz_op = a.hiz_op;
    const bool less = a.less_depth != 0;
    // Chunk culling compares the lower end of a candidate's depth interval with
    // the largest stored depth.  Launches with GREATER or GREATER_OR_EQUAL hold
    // the intervals of the negated depths in their records (setup_kernel), and
    // the stored depths are compared negated: the op then fails in the same
    // direction.  (Choosing the interval's end here made every frame 0.8%
    // slower.)  For EQUAL the lower end alone is compared: the upper one's test
    // in the walk raised the scalar spills from 67 to 92.
    const uint32_t cull_mode = a.cull_mode;
    auto toward = [&](float v) { return __uint_as_float(__float_as_uint(v) ^ (cull_mode & kCullGreater)); };
    uint32_t tried = 0;   // queues found empty, starting at home
    // Split tiles (splits_tile) are units of work, one per block of each of the
    // workgroup's waves, and start first.  Waves that hold two blocks gain
    // nothing from it (48-job batch, 16x16 tiles: 1,354 us unsplit, 1,373).
    constexpr bool SPLIT = BPW >= kSplitBlocks;
    const bool units = SPLIT && blockIdx.x < a.long_groups;
    uint32_t unit = blockIdx.x;

    for (;;) {
        uint32_t item = SPLIT ? blockIdx.x - a.long_groups : blockIdx.x;
        uint32_t kmask = ~0u;   // the blocks k of a lane that this pass takes
        int slot = wave;
        if (a.persistent) {
            // Unit u of queue q is wave slot u % WAVES of the queue's
            // (u / WAVES)-th tile, queue item (u / WAVES) * kRasterQueues + q.
            // Every wave ends after at most one failed take per queue.
            for (; tried < kRasterQueues; tried++) {
                const uint32_t q = (home + tried) % kRasterQueues;
                const uint32_t per_q = a.tiles > q ? (a.tiles - q + kRasterQueues - 1) / kRasterQueues : 0u;
                uint32_t u = 0;
                if (lane == 0) u = atomicAdd(a.queue + q * kRasterQueueStride, 1u);
                u = __builtin_amdgcn_readfirstlane(u);
                if (u < per_q * (uint32_t)WAVES) {
                    item = (u / WAVES) * kRasterQueues + q;
                    slot = (int)(u % WAVES);
                    break;
                }
            }
            if (tried == kRasterQueues) break;
        }
        if (units) {
            // units u, u + 8, ... of eight tiles are the eight's blocks 0, 1, ...:
            // a tile's are taken by workgroups of one XCD
            const uint32_t t = unit / (kRasterQueues * BPW) * kRasterQueues + unit % kRasterQueues;
            if (unit / (kRasterQueues * BPW) * kRasterQueues >= uniform_ptr(a.longs)->count) break;
            kmask = 1u << unit / kRasterQueues % BPW;
            unit += a.long_groups;
            if (t >= uniform_ptr(a.longs)->count) continue;
            item = uniform_ptr(a.long_tiles)[t];
        } else if (item >= a.tiles) {
            break;
        }
        const uint32_t tile = units ? item : __builtin_amdgcn_readfirstlane(a.order ? a.order[item] : item);
        const uint2 range = uniform_ptr(a.tile_range)[tile];
        const uint32_t lbeg = range.x, lend = range.y;
        if (SPLIT && a.long_groups) {
            const bool split = lend > lbeg && splits_tile(*uniform_ptr(a.longs), lend - lbeg, WAVES);
            if (units && !split) continue;
            if (!units && split) break;
        }
        const uint64_t t_begin = clock64();

        const uint32_t ti = find_target(uniform_ptr(a.targets), a.target_count, tile);
        const TargetParams& tp = *uniform_ptr(&a.targets[ti]);
        const uint32_t local = tile - tp.tile_base;
        const int tile_x0 = __builtin_amdgcn_readfirstlane((int)(local % tp.tiles_x) * TILE);
        const int tile_y0 = __builtin_amdgcn_readfirstlane((int)(local / tp.tiles_x) * TILE);
        const bool has_color = FIXED || tp.has_color, has_ds = FIXED || tp.has_ds;
        const int color_bytes = FIXED ? 4 : tp.color_bytes, ds_bytes = FIXED ? 4 : tp.ds_bytes;

        // ---- pixel state: loadOp CLEAR sets the packed clear value;
        // LOAD / DONT_CARE read the attachment.
        PixelState px[BPW];
        // the stored depth as a float, beside its packed code (a D32 code is
        // its bits)
        float zc[BPW];
        int pxx[BPW], pxy[BPW];
        bool inside[BPW];
        const int32_t tile_depth = FIXED ? 32 : has_ds ? tp.ds_fmt.depth_kind : 0;
#pragma unroll
        for (int k = 0; k < BPW; k++) {
            const int blk = slot + k * WAVES;
            const int bx0 = tile_x0 + (blk % BW) * 8, by0 = tile_y0 + (blk / BW) * 8;
            pxx[k] = bx0 + (lane & 7);
            pxy[k] = by0 + (lane >> 3);
            inside[k] = pxx[k] < (int)tp.width && pxy[k] < (int)tp.height && (!SPLIT || (kmask >> k & 1u));
#pragma unroll
            for (int w = 0; w < 4; w++) px[k].color[w] = tp.clear_color[w];
            px[k].ds0 = tp.clear_ds[0];
            px[k].ds1 = tp.clear_ds[1];
            const uint64_t pix = (uint64_t)pxy[k] * tp.width + (uint64_t)pxx[k];
            if (inside[k] && has_color && tp.color_load != 1)
                load_pixel(global_ptr<const uint8_t>(tp.color_addr) + pix * color_bytes, color_bytes, px[k].color);
            if (inside[k] && has_ds && tp.ds_load != 1) {
                uint32_t w4[4];
                load_pixel(global_ptr<const uint8_t>(tp.ds_addr) + pix * ds_bytes, ds_bytes, w4);
                px[k].ds0 = w4[0];
                px[k].ds1 = w4[1];
            } else if (inside[k] && has_ds && ds_bytes == 8) {
                // D32_SFLOAT_S8_UINT cleared: SetPixelDepthStencil writes the
                // depth and the stencil byte and keeps the three padding bytes
                // (ImageCompiler.cpp:895-945)
                uint32_t w4[4];
                load_pixel(global_ptr<const uint8_t>(tp.ds_addr) + pix * ds_bytes, ds_bytes, w4);
                px[k].ds1 = (w4[1] & 0xFFFFFF00u) | (tp.clear_ds[1] & 0xFFu);
            }
            zc[k] = stored_depth(tile_depth, px[k].ds0);
        }
        auto cur_depth = [&](int k) { return FIXED ? __uint_as_float(px[k].ds0) : zc[k]; };

        // ---- per-draw state, refreshed when the draw changes
        uint32_t cur_draw = 0xFFFFFFFFu;
        float xf[BPW], yf[BPW];
        float vp_min = 0.0f, vp_max = 1.0f;
        bool vp_identity = true, depth_write = false;
        uint64_t or_equal = 0;   // every lane for LESS_OR_EQUAL, none for LESS
        const FragmentState* fst = nullptr;
        const DrawEnv* env = nullptr;
        // conservative depth rejection allowed for this draw, and its op
        // (launches without less_depth)
        bool early = false;
        int32_t depth_op = 7;
        unsigned long long nfrag = 0;

        // Deferred colour work: a fragment that passed the depth/stencil
        // tests has its depth/stencil written at once, and its colour
        // (interpolation, fragment shader, blend, pack) queued.  Queues drain
        // in order, so every pixel still sees its colour writes in primitive
        // order; draining for all lanes at once keeps the shading path from
        // running once per primitive whenever any lane passes.  A lane's
        // queue is a ring of Q 16-byte entries in LDS (primitive and block,
        // three weights): a push is one store, where entries in registers
        // took 20 vector selects per push, a shift per drain and 16 registers.
        constexpr int Q = RasterStage<FS, TILE, WAVES>::kQueue;
        int qn = 0, qhead = 0;
        auto& queue = stage_area.q[FS::kMayDiscard ? 0 : wave];

        auto shade = [&](uint32_t gprim, int k, float w0, float w1, float w2) {
            PixelState ps = px[0];
            int sx = pxx[0], sy = pxy[0];
#pragma unroll
            for (int kk = 1; kk < BPW; kk++)
                if (kk == k) { ps = px[kk]; sx = pxx[kk]; sy = pxy[kk]; }
            ps = shade_fragment<FS, ANYPRIM, FIXED>(a.recs, a.draws, a.fstates, a.uniform_fstate, a.vout, a.vout_stride, gprim, w0, w1,
                                                    w2, sx, sy, ps);
#pragma unroll
            for (int kk = 0; kk < BPW; kk++)
                if (kk == k) px[kk] = ps;
        };
        // Shades the oldest queued entry of every lane that has one: called
        // when some lane's queue is full, this keeps the other lanes' queues
        // filled, so each shading pass runs with as many lanes as possible.
        auto drain_one = [&]() {
            if (qn > 0) {
                const float4 e = queue[qhead & (Q - 1)][lane];
                const uint32_t tag = __float_as_uint(e.x);
                shade(tag & kPairPrim, (int)(tag >> 28), e.y, e.z, e.w);
                qhead++;
                qn--;
            }
        };

        // ---- walk the tile's primitives in submission order
        // The pairs that name one of this wave's blocks (the emit kernels pack
        // a primitive's blocks, or for 32x32 tiles 16x16 quadrants, into the
        // pair) are its candidates: fetch() gives the next up to 64 of them,
        // a candidate per lane in order.  Lists of more than 64 pairs are
        // read 256 at a time and their candidates packed through a ring in
        // LDS, so that every chunk but the last is full: a wave's 8x8 block
        // is named by about 40% of the 1M soup's pairs, and the clustered 4K
        // frame's heaviest tile, a serial chain of 950 chunks of 64 pairs,
        // is one of about 330.
        uint32_t mine = 0u;
        if (TILE == 16) {
#pragma unroll
            for (int k = 0; k < BPW; k++)
                if (!SPLIT || (kmask >> k & 1u)) mine |= 1u << (kPairBlockShift + slot + k * WAVES);
        } else if (TILE == 32) {
#pragma unroll
            for (int k = 0; k < BPW; k++) {
                const int blk = slot + k * WAVES;
                if (!SPLIT || (kmask >> k & 1u)) mine |= 1u << (kPairBlockShift + (blk / BW) / 2 * 2 + (blk % BW) / 2);
            }
        }
        const bool deep = lend > lbeg && lend - lbeg > 64u;   // wave-uniform
        const bool packed = TILE != 8 && deep;   // every pair of an 8x8 tile names its block
        auto& ring = stage_area.ring[wave];
        constexpr uint32_t R = RasterStage<FS, TILE, WAVES>::kRing;
        uint32_t pos = packed ? lbeg & ~3u : lbeg, head = 0, tail = 0;
        auto group = [&](uint32_t at) {   // pairs at + 4 * lane .. + 3 of the list (16-byte aligned)
            const uint32_t i = at + 4u * (uint32_t)lane;
            return i >= at && i < lend ? *(const uint4*)(a.tile_prims + i) : make_uint4(0u, 0u, 0u, 0u);
        };
        uint4 g_next = packed ? group(pos) : make_uint4(0u, 0u, 0u, 0u);   // loaded a step ahead
        auto fetch = [&](uint32_t& e, bool& ok) {
            if (packed) {
                while (tail - head < 64u && pos < lend) {
                    const uint32_t v[4] = {g_next.x, g_next.y, g_next.z, g_next.w};
                    const uint32_t i = pos + 4u * (uint32_t)lane;
                    pos += min(256u, lend - pos);
                    g_next = group(pos);
                    uint32_t at = tail;
                    bool hit[4];
#pragma unroll
                    for (int j = 0; j < 4; j++) {
                        hit[j] = (v[j] & mine) != 0u && i + j >= lbeg && i + j < lend;
                        const uint64_t m = lanes(hit[j]);
                        at = __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, at));
                        tail += (uint32_t)__popcll(m);
                    }
#pragma unroll
                    for (int j = 0; j < 4; j++)
                        if (hit[j]) { ring[at & (R - 1)] = v[j]; at++; }
                }
                wave_lds_fence();
                const uint32_t n = min(64u, tail - head);
                e = ring[(head + (uint32_t)lane) & (R - 1)];
                ok = (uint32_t)lane < n;
                head += n;
                wave_lds_fence();
            } else {
                const uint32_t i = pos + (uint32_t)lane;
                ok = i >= pos && i < lend;
                e = ok ? a.tile_prims[i] : 0u;
                if (TILE != 8) ok = ok && (e & mine) != 0u;
                pos += min(64u, lend - min(pos, lend));
            }
        };
        auto more = [&]() { return packed ? tail != head || pos < lend : pos < lend; };
        // The next chunk's candidates are fetched, and the lower end of their
        // depth interval loaded, before this chunk is worked on; with it their
        // records come into the XCD's L2.
        uint32_t e_next = 0u;
        bool ok_next = false;
        float lo_next = 0.0f;
        auto prefetch = [&]() {
            ok_next = false;
            if (more()) {
                fetch(e_next, ok_next);
                if (ok_next) lo_next = a.recs[e_next & kPairPrim].dt_lo;
            }
        };
        bool chunk = more();
        prefetch();
        while (chunk) {
            const uint32_t e = e_next, gp_l = e & kPairPrim, blocks_l = e >> kPairBlockShift;
            float lo_l = lo_next;
            bool ov = ok_next;
            chunk = more();
            prefetch();
            // Hierarchical culling: a primitive whose depth interval fails
            // the test against every depth stored in the wave's pixels
            // cannot change any of them.  `lo_l` holds the lower end of a
            // candidate's interval, and the stored depths only fall (negated
            // ones too), so it is tested again every few visits against their
            // current maximum (a dozen vector instructions, a third of a
            // visit).  Testing once per chunk left the soup 27 us
            // slower once the chunks were full.
            bool refined = !BLOCK_DEPTH || !deep;   // short lists: not worth the records' loads
            auto cull = [&](uint64_t m) {
                float bmax = -__builtin_inff();
#pragma unroll
                for (int k = 0; k < BPW; k++)
                    if (inside[k]) bmax = fmaxf(bmax, toward(cur_depth(k)));
                bmax = wave_max(bmax);
                m &= ~lanes(lo_l > bmax);
                if (BLOCK_DEPTH && !refined && __popcll(m) >= kRefineCandidates) {
                    if (cur_draw != 0xFFFFFFFFu && vp_identity) {
                        // A triangle's depth bounded over the pixels it may
                        // cover in this wave's block (block_depth_range): its
                        // box clipped to the block, far tighter than its
                        // bounds over all its pixels.  For the candidates of
                        // the draw last visited, whose pixel centres the lanes
                        // hold, when that draw's depth range is [0, 1] (the
                        // depth then is the tested value).
                        refined = true;
                        const bool mine_l = in_lanes(m);
                        uint4 p0 = make_uint4(0u, 0u, 0u, 0u), p1 = p0, p2 = p0, p3 = p0, p4 = p0, p5 = p0;
                        if (mine_l) {
                            const uint4* src = (const uint4*)&a.recs[gp_l];
                            p0 = src[0]; p1 = src[1]; p2 = src[2]; p3 = src[3]; p4 = src[4]; p5 = src[5];
                        }
                        // lane c holds column bx0 + c, lane 8 r row by0 + r
                        const int bx0 = __builtin_amdgcn_readfirstlane(pxx[0]), by0 = __builtin_amdgcn_readfirstlane(pxy[0]);
                        const int cl = min(max((int)p3.x - bx0, 0), 7), ch = min(max((int)p3.z - 1 - bx0, 0), 7);
                        const int rl = min(max((int)p3.y - by0, 0), 7), rh = min(max((int)p3.w - 1 - by0, 0), 7);
                        const float xa = __shfl(xf[0], cl, 64), xb = __shfl(xf[0], ch, 64);
                        const float ya = __shfl(yf[0], rl * 8, 64), yb = __shfl(yf[0], rh * 8, 64);
                        if (mine_l && (p4.w & kPrimDraw) == cur_draw) {
                            const float ax[3] = {__uint_as_float(p0.x), __uint_as_float(p0.y), __uint_as_float(p0.z)};
                            const float ay[3] = {__uint_as_float(p0.w), __uint_as_float(p1.x), __uint_as_float(p1.y)};
                            const float dy[3] = {__uint_as_float(p1.z), __uint_as_float(p1.w), __uint_as_float(p2.x)};
                            const float dx[3] = {__uint_as_float(p2.y), __uint_as_float(p2.z), __uint_as_float(p2.w)};
                            const float z[3] = {__uint_as_float(p5.x), __uint_as_float(p5.y), __uint_as_float(p5.z)};
                            float lo, hi;
                            if (block_depth_range(ax, ay, dy, dx, __uint_as_float(p4.z), __uint_as_float(p5.w), z, fminf(xa, xb),
                                                  fmaxf(xa, xb), fminf(ya, yb), fmaxf(ya, yb), lo, hi))
                                lo_l = fmaxf(lo_l, toward((cull_mode & kCullGreater) ? hi : lo));
                        }
                        m &= ~lanes(lo_l > bmax);
                    }
                }
                return m;
            };
            uint64_t mask = lanes(ov);
            int since = kCullVisits;   // candidates visited since the last cull
            const int step = deep ? kCullLanes : 64;
            for (int first = 0; first < 64; first += step) {
              uint64_t window = mask & ((~0ull >> (64 - step)) << first);
              if ((cull_mode & kCullOn) && window && since >= kCullVisits) {
                  mask = cull(mask & (~0ull << first));
                  window &= mask;
                  since = 0;
              }
              since += __popcll(window);
              while (window) {
                const int j = (int)__builtin_ctzll(window);
                window &= window - 1;
                const uint32_t gprim = __builtin_amdgcn_readlane(gp_l, j);
                const uint32_t blocks = (TILE >= 16 && BPW > 1) ? __builtin_amdgcn_readlane(blocks_l, j) : 0u;
                TriSetup r;
                load_record_uniform(a.recs, gprim, r);
                // the loads of all visit fields issued before the first of
                // them is used: one memory latency per survivor, not one
                // for the draw index and another for the rest
                __asm__ volatile("" ::"s"(r.ax[0]), "s"(r.y1), "s"(r.dt_lo), "s"(r.draw_flags), "s"(r.z[0]), "s"(r.rinv));
                const uint32_t flags = r.draw_flags >> kPrimFlagShift;
                if ((r.draw_flags & kPrimDraw) != cur_draw) {
                    cur_draw = r.draw_flags & kPrimDraw;
                    const DrawDesc& d = *uniform_ptr(&a.draws[cur_draw]);
                    // pixel centres (ProcessTriangles :1571-1580)
#pragma unroll
                    for (int k = 0; k < BPW; k++) {
                        xf[k] = ((float)pxx[k] / d.vp_w + d.half_x) * 2.0f - 1.0f;
                        yf[k] = ((float)pxy[k] / d.vp_h + d.half_y) * 2.0f - 1.0f;
                    }
                    vp_min = d.vp_min_depth;
                    vp_max = d.vp_max_depth;
                    vp_identity = vp_min == 0.0f && vp_max == 1.0f;
                    fst = uniform_ptr(&a.fstates[d.fstate]);
                    env = uniform_ptr<DrawEnv>(d.env);
                    or_equal = fst->depth_compare == 3 ? ~0ull : 0ull;   // LESS_OR_EQUAL
                    depth_write = fst->depth_write != 0;
                    // Rejecting on the depth test alone is exact when nothing
                    // else observes the fragment: no depth-bounds or stencil
                    // test (and so no stencil write).
                    early = !less && fst->depth_test && (FIXED || (fst->has_ds && fst->ds.depth_off >= 0 && fst->ds.vk_format != 127u)) &&
                            !fst->depth_bounds_test && !fst->stencil_test;
                    depth_op = fst->depth_compare;
                }
                const bool has_fcolor = FIXED || fst->has_color;
#pragma unroll
                for (int k = 0; k < BPW; k++) {
                    const int blk = slot + k * WAVES;
                    const int bx0 = tile_x0 + (blk % BW) * 8, by0 = tile_y0 + (blk / BW) * 8;
                    if (SPLIT && !(kmask >> k & 1u)) continue;   // wave-uniform
                    if (TILE == 16 && BPW > 1) {
                        if (!((blocks >> blk) & 1u)) continue;   // wave-uniform
                    } else if (BPW > 1) {
                        // wave-uniform: the block's quadrant may be covered
                        // and the block meets the primitive's box
                        if (TILE == 32 && !((blocks >> ((blk / BW) / 2 * 2 + (blk % BW) / 2)) & 1u)) continue;
                        if (r.x1 <= bx0 || r.x0 >= bx0 + 8 || r.y1 <= by0 || r.y0 >= by0 + 8) continue;
                    }
                    // The tests narrow `m`, the lanes still in, with every lane
                    // evaluating them; the visit ends when it is empty, and no
                    // lane branches until the fragments that are left.
                    const int x = pxx[k], y = pxy[k];
                    uint64_t m = lanes(x >= r.x0) & lanes(x < r.x1) & lanes(y >= r.y0) & lanes(y < r.y1);
                    if (hiz_op >= 0) {
                        const float cd = cur_depth(k);
                        if (less) m &= ~lanes(r.dt_lo > cd);
                        else if (cull_mode & kCullGreater) m &= ~lanes(r.dt_lo > -cd);
                        else m &= ~lanes(hiz_rejects(hiz_op, r.dt_lo, r.dt_hi, cd, cd));
                    }
                    if (!m) continue;
                    float w0, w1, w2, depth;
                    if (ANYPRIM && (flags & kPrimPoint)) {
                        // ProcessPoints (:1358-1378): s, t of the pixel in the
                        // point's square, the vertex's outputs and depth as they are
                        const float size = r.dx[0];
                        const float s = 0.5f + (float)(int32_t)((uint32_t)x - (uint32_t)__float_as_int(r.ax[0])) / size;
                        const float t = 0.5f + (float)(int32_t)((uint32_t)y - (uint32_t)__float_as_int(r.ay[0])) / size;
                        m &= lanes(s >= 0.0f) & lanes(t >= 0.0f) & lanes(s <= 1.0f) & lanes(t <= 1.0f);
                        nfrag += (uint32_t)__popcll(m);
                        w0 = 1.0f; w1 = 0.0f; w2 = 0.0f;
                        depth = r.z[0];
                    } else if (ANYPRIM && (flags & kPrimLine)) {
                        // ProcessLines (:1420-1497): all four quad edges >= 0
                        // (NaN fails), t = dot(p - p0, p1 - p0) / |p1 - p0|^2
                        const LineExt L = load_line_ext(a.line_ext, gprim);
                        const float e0 = (xf[k] - r.ax[0]) * r.dy[0] - (yf[k] - r.ay[0]) * r.dx[0];
                        const float e1 = (xf[k] - r.ax[1]) * r.dy[1] - (yf[k] - r.ay[1]) * r.dx[1];
                        const float e2 = (xf[k] - r.ax[2]) * r.dy[2] - (yf[k] - r.ay[2]) * r.dx[2];
                        const float e3 = (xf[k] - L.ax3) * L.dy3 - (yf[k] - L.ay3) * L.dx3;
                        m &= lanes(e0 >= 0.0f) & lanes(e1 >= 0.0f) & lanes(e2 >= 0.0f) & lanes(e3 >= 0.0f);
                        nfrag += (uint32_t)__popcll(m);
                        if (!m) continue;
                        const float t = ((xf[k] - L.p0x) * L.ddx + (yf[k] - L.p0y) * L.ddy) / r.area;
                        w0 = 1.0f - t; w1 = t; w2 = 0.0f;
                        depth = r.z[0] * t + r.z[1] * (1.0f - t);
                    } else {
                        // GetFragmentInput (:874-903); NaN edge values are not
                        // < 0 and pass, and fminf passes over them
                        const float e0 = (xf[k] - r.ax[0]) * r.dy[0] - (yf[k] - r.ay[0]) * r.dx[0];
                        const float e1 = (xf[k] - r.ax[1]) * r.dy[1] - (yf[k] - r.ay[1]) * r.dx[1];
                        const float e2 = (xf[k] - r.ax[2]) * r.dy[2] - (yf[k] - r.ay[2]) * r.dx[2];
                        const float emin = fminf(fminf(e0, e1), e2);
                        m &= ~lanes(emin < 0.0f);
                        nfrag += (uint32_t)__popcll(m);
                        const bool fast = (flags & kPrimFast) != 0;   // wave-uniform
                        const float q0 = e0 * r.rinv, q1 = e1 * r.rinv, q2 = e2 * r.rinv;
                        if (less) {
                            if (fast && vp_identity) m &= ~lanes(depth_surely_not_less(cur_depth(k), q0, q1, q2, r));
                        } else if (early) {
                            if (vp_identity)
                                m &= ~lanes(depth_surely_fails_unit(depth_op, cur_depth(k), e0, e1, e2, r.area, r.z[0], r.z[1], r.z[2]));
                            else
                                m &= ~lanes(depth_surely_fails(depth_op, cur_depth(k), e0, e1, e2, r.area, r.z[0], r.z[1], r.z[2],
                                                               vp_min, vp_max));
                        }
                        if (!m) continue;
                        // a tiny edge value (or an exact zero, whose sign the
                        // quotient keeps) takes the divisions
                        if (fast && !(m & ~lanes(emin >= 0x1p-60f))) {
                            w0 = divide_exact(e0, r.area, r.rinv, q0);
                            w1 = divide_exact(e1, r.area, r.rinv, q1);
                            w2 = divide_exact(e2, r.area, r.rinv, q2);
                        } else {
                            w0 = e0 / r.area; w1 = e1 / r.area; w2 = e2 / r.area;
                        }
                        depth = r.z[0] * w0 + r.z[1] * w1 + r.z[2] * w2;
                    }
                    // DrawPixel (:1300-1313)
                    const float dt = (vp_max - vp_min) * depth + vp_min;
                    const bool front = (flags & kPrimFront) != 0;
                    if (FS::kMayDiscard) {
                        if (!in_lanes(m)) continue;
                        // the shader decides first whether anything is written
                        float in_v[FS::kInputs > 0 ? FS::kInputs : 1];
                        fragment_inputs<FS, ANYPRIM>(r, a.vout, a.vout_stride, w0, w1, w2, in_v);
                        const float fc[4] = {fst->origin_upper_left ? (float)x : uniform_ptr(&a.draws[cur_draw])->vp_w - (float)x - 1.0f,
                                             (float)y, depth, 1.0f};
                        float colour[4];
                        if (FS::run(*env, in_v, fc, front, colour)) continue;
                        const DepthStencilResult dr = depth_stencil_call<FIXED>(*fst, px[k], dt, front ? 1u : 0u);
                        px[k] = dr.px;
                        if (!FIXED) zc[k] = stored_depth(tile_depth, px[k].ds0);
                        if (dr.write && has_fcolor) color_write_state<FIXED>(*fst, px[k], colour);
                    } else {
                        if (less) {
                            const float cd = cur_depth(k);
                            m &= lanes(dt < cd) | (lanes(dt == cd) & or_equal);
                            if (!m) continue;
                            if (depth_write && in_lanes(m)) {
                                if (FIXED) {
                                    px[k].ds0 = __float_as_uint(dt);
                                } else {
                                    pack_depth_stencil(fst->ds, dt, unpack_stencil(fst->ds, px[k].ds0, px[k].ds1), px[k].ds0, px[k].ds1);
                                    zc[k] = stored_depth(tile_depth, px[k].ds0);
                                }
                            }
                        } else {
                            bool write = false;
                            if (in_lanes(m)) {
                                const DepthStencilResult dr = depth_stencil_call<FIXED>(*fst, px[k], dt, front ? 1u : 0u);
                                px[k] = dr.px;
                                if (!FIXED) zc[k] = stored_depth(tile_depth, px[k].ds0);
                                write = dr.write != 0;
                            }
                            m = lanes(write);
                        }
                        if (!m || !has_fcolor) continue;
                        // every lane is active here; a lane queues at most one
                        // entry per visit, so a free slot always exists
                        if (lanes(qn == Q)) drain_one();
                        if (in_lanes(m)) {
                            queue[(qhead + qn) & (Q - 1)][lane] = make_float4(__uint_as_float(gprim | ((uint32_t)k << 28)), w0, w1, w2);
                            qn++;
                        }
                    }
                }
              }
            }
        }
        if (!FS::kMayDiscard) {
            while (lanes(qn > 0)) drain_one();
        }
        (void)env;

        // ---- write back
#pragma unroll
        for (int k = 0; k < BPW; k++) {
            if (!inside[k]) continue;
            const uint64_t pix = (uint64_t)pxy[k] * tp.width + (uint64_t)pxx[k];
            if (has_color) store_pixel(global_ptr<uint8_t>(tp.color_addr) + pix * color_bytes, color_bytes, px[k].color);
            if (has_ds) {
                const uint32_t w4[4] = {px[k].ds0, px[k].ds1, 0u, 0u};
                store_pixel(global_ptr<uint8_t>(tp.ds_addr) + pix * ds_bytes, ds_bytes, w4);
            }
        }

        // ---- statistics (nfrag is wave-uniform)
        if (a.count && lane == 0 && nfrag) atomicAdd(a.fragments, nfrag);
        if (a.trace_cycles && lane == 0) a.trace_cycles[(uint64_t)tile * WAVES + slot] = (float)(clock64() - t_begin);

        if (!a.persistent && !units) break;
    }
}

// ANYPRIM: the launch may hold point and line records besides triangles
// (one 16x16 / four-wave instantiation per fragment shader carries it).
// FIXED: every pipeline and target of the launch has the fixed formats
// (fold_fixed_formats).
template <class FS, int TILE, int WAVES, bool ANYPRIM = false, bool FIXED = false>
__global__ __launch_bounds__(64 * WAVES) __attribute__((amdgpu_waves_per_eu(raster_waves_per_eu<FS, TILE, WAVES>()))) void
raster_kernel(RasterArgs a)
{
    __shared__ RasterStage<FS, TILE, WAVES> stage;
    raster_body<FS, TILE, WAVES, ANYPRIM, FIXED>(a, stage);
}

}  // namespace cpv
