// Transfer and clear commands on the context stream: region copies
// (vkCmdCopyBuffer / CopyImage / CopyBufferToImage / CopyImageToBuffer
// after the front end has turned their regions into byte rows), buffer
// fills and updates, rectangle clears (vkCmdClearColorImage,
// vkCmdClearDepthStencilImage, vkCmdClearAttachments) and blits.
//
// Each is enqueued on the same stream as the render passes, so a replayed
// command buffer keeps its order without host synchronisation.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>

#include "cpv_internal.h"
#include "raster_kernels.h"

using namespace cpv;
using namespace cpvrt;

namespace {

// Rows of one repeated pixel.
struct FillArgs {
    uint8_t* dst;           // first byte of the first row
    uint64_t row_bytes;
    uint64_t pitch;         // from row to row
    uint64_t chunks;        // 16-byte chunks of memory that a row can meet
    uint32_t rows;
    uint32_t size;          // bytes of a pixel: 1, 2, 4, 8 or 16, dividing every row's address
    uint32_t pattern[4];    // the pixel repeated over 16 bytes
};

// Each thread takes 16-byte aligned chunks: a chunk inside its row is one
// store, at a row's ends the pixels inside are stored one by one.  A pixel's
// size divides 16 and its address, so every chunk holds the same pattern.
// Bound by HBM writes: 64 MiB in 11.1 us (6.0 TB/s; as whole words 11.4),
// 1 GiB in 154 us (7.0 TB/s; 203), a clear of 3840x2160 RGBA8 in 6.6 us (5.0
// TB/s; one 4-byte store a thread, with the packing on the device, took 28).
__global__ __launch_bounds__(256) void fill_rows_kernel(FillArgs a)
{
    const uint4 v = make_uint4(a.pattern[0], a.pattern[1], a.pattern[2], a.pattern[3]);
    for (uint32_t row = blockIdx.y * blockDim.y + threadIdx.y; row < a.rows; row += gridDim.y * blockDim.y) {
        const uint64_t beg = (uint64_t)a.dst + row * a.pitch, end = beg + a.row_bytes, first = beg & ~15ull;
        for (uint64_t k = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; k < a.chunks; k += (uint64_t)gridDim.x * blockDim.x) {
            const uint64_t p = first + k * 16u;
            if (p >= beg && p + 16 <= end) {
                *global_ptr<uint4>(p) = v;
            } else {
                // words inside the row whole (pixels of 8 and 16 bytes are
                // words inside it too), the rest by pixels of 1 and 2 bytes
#pragma unroll
                for (uint32_t w = 0; w < 4u; w++) {
                    const uint64_t q = p + 4u * w;
                    if (q >= beg && q + 4u <= end) {
                        *global_ptr<uint32_t>(q) = a.pattern[w];
                    } else if (q + 4u > beg && q < end) {
                        for (uint32_t o = 0; o < 4u; o += a.size)
                            if (q + o >= beg && q + o < end) store_pixel(global_ptr<uint8_t>(q + o), (int)a.size, a.pattern);
                    }
                }
            }
        }
    }
}

// FillBufferCommand::Process (CPVulkan/CommandBuffer.cpp:307-326): the word
// fills every whole 4-byte unit (fill_rows_kernel); the bytes of a size % 4
// tail go to byte size / 4 + i, as the reference indexes them.
__global__ void fill_tail_kernel(uint8_t* dst, uint64_t size, uint32_t data)
{
    const uint32_t i = threadIdx.x;
    if (i < (uint32_t)(size % 4)) dst[size / 4 + i] = (uint8_t)(data >> (8 * i));
}

struct ClearArgs {
    uint8_t* base;          // first byte of the image level
    uint32_t total, stored; // bytes of a pixel, and of those that are written
    uint32_t width;         // pixels per row
    int32_t x0, y0;
    uint32_t w, h;
    uint32_t words[4];      // the packed pixel
};

// Bytes a pixel store writes: the reference's SetPixelDepthStencil stores
// the depth and the stencil byte of D32_SFLOAT_S8_UINT and leaves its three
// padding bytes (ImageCompiler.cpp:895-945); every other format is written whole.
CPV_HOST_DEV int stored_bytes(const FormatDesc& f)
{
    return (f.total == 8 && f.depth_off == 0 && f.stencil_off == 4) ? 5 : f.total;
}

// The packed pixel of a clear value (SetPixel overloads for
// VkClearColorValue and VkClearDepthStencilValue, ImageSampler.cpp:723-800).
void pack_clear(const FormatDesc& f, const uint32_t value[4], uint32_t words[4])
{
    words[0] = words[1] = words[2] = words[3] = 0u;
    if (f.depth_off >= 0 || f.stencil_off >= 0) {
        float depth;
        std::memcpy(&depth, &value[0], 4);
        pack_depth_stencil(f, depth, value[1], words[0], words[1]);
    } else if (f.base == kBaseUInt) {
        pack_color_u32(f, value, words);
    } else if (f.base == kBaseSInt) {
        int32_t v[4];
        std::memcpy(v, value, 16);
        pack_color_i32(f, v, words);
    } else {
        float v[4];
        std::memcpy(v, value, 16);
        pack_color_f32(f, v, words);
    }
}

// SetPixel of the packed clear value over a rectangle (ClearImage,
// CommandBuffer.Draw.cpp:117-149; ClearAttachmentsCommand :2176-2220), for
// the pixels that fill_rows_kernel does not take: 3 and 12 bytes, and
// D32_SFLOAT_S8_UINT's 5 of 8.
__global__ void clear_rect_kernel(ClearArgs a)
{
    // rectangle pixels in row-major order, grid-strided; the stride's row
    // and column steps are divided out once
    const uint64_t n = (uint64_t)a.w * a.h;
    const uint64_t step = (uint64_t)gridDim.x * blockDim.x;
    uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    uint32_t rx = (uint32_t)(i % a.w), ry = (uint32_t)(i / a.w);
    const uint32_t sx = (uint32_t)(step % a.w), sy = (uint32_t)(step / a.w);
    for (; i < n; i += step) {
        const uint32_t x = (uint32_t)a.x0 + rx, y = (uint32_t)a.y0 + ry;
        store_pixel(a.base + ((uint64_t)y * a.width + x) * a.total, (int)a.stored, a.words);
        rx += sx;
        ry += sy;
        if (rx >= a.w) { rx -= a.w; ry++; }
    }
}

struct BlitArgs {
    TextureDesc src;        // the source level as level 0, CLAMP_TO_EDGE
    uint8_t* dst;
    FormatDesc dfmt;
    uint32_t dst_width;
    int32_t s0x, s0y, s1x, s1y, d0x, d0y, d1x, d1y;
    uint32_t w, h;          // |d1 - d0|
    uint32_t filter;
    uint32_t aspect;        // VkImageAspectFlags of the region
    uint32_t src_kind;      // 0 float, 1 uint, 2 sint, 3 depth/stencil
};

CPV_DEV uint32_t raw_channel(const FormatDesc& f, const uint32_t px[4], int c)
{
    return f.off[c] < 0 ? 0u : get_field(px, f.off[c], f.element);
}

CPV_DEV void read_pixel(const uint8_t* p, int bytes, uint32_t w[4])
{
    w[0] = w[1] = w[2] = w[3] = 0u;
    // unrolled over the largest pixel so w[] keeps constant indices (registers)
#pragma unroll
    for (int b = 0; b < 16; b++)
        if (b < bytes) w[b >> 2] |= (uint32_t)p[b] << ((b & 3) * 8);
}

// BlitImageCommand::Process (CPVulkan/CommandBuffer.cpp:57-238): per
// destination pixel, u = (dstX + 0.5 - dst0.x) * ((float)(src1.x - src0.x) /
// (dst1.x - dst0.x)) + src0.x (likewise v); colour formats are sampled at
// (u / W, v / H) with the blit filter and CLAMP_TO_EDGE (SampleImage,
// ImageSampler.cpp:676-681) and written with SetPixel; depth/stencil
// formats read the texel at the truncated (u, v).
// KIND is a.src_kind and FILTER a.filter, fixed per instantiation so each
// carries only its own path; KIND 4 is a float source whose texels
// sample_level_as<true> reads (with both in one kernel, 2048x2048 of R8 to half
// the size took 24.1 us against 21.8).
template <int KIND, int FILTER>
__global__ void blit_kernel(BlitArgs a)
{
    const TextureDesc& src = a.src;
    const FormatDesc& dfmt = a.dfmt;
    const bool negx = a.d1x < a.d0x, negy = a.d1y < a.d0y;
    const float rx = (float)(a.s1x - a.s0x) / (float)(a.d1x - a.d0x);
    const float ry = (float)(a.s1y - a.s0y) / (float)(a.d1y - a.d0y);
    // destination pixels in row-major order, grid-strided as clear_rect_kernel
    const uint64_t n = (uint64_t)a.w * a.h;
    const uint64_t step = (uint64_t)gridDim.x * blockDim.x;
    uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    uint32_t ux = (uint32_t)(i % a.w), uy = (uint32_t)(i / a.w);
    const uint32_t sx = (uint32_t)(step % a.w), sy = (uint32_t)(step / a.w);
    for (; i < n; i += step, ux += sx, uy += sy) {
        if (ux >= a.w) { ux -= a.w; uy++; }
        const int32_t x = (int32_t)ux, y = (int32_t)uy;
        const int32_t dx = negx ? x + a.d1x : x + a.d0x;
        const int32_t dy = negy ? y + a.d1y : y + a.d0y;
        const float u = ((float)dx + 0.5f - (float)a.d0x) * rx + (float)a.s0x;
        const float v = ((float)dy + 0.5f - (float)a.d0y) * ry + (float)a.s0y;
        uint8_t* out = a.dst + ((uint64_t)dy * a.dst_width + (uint64_t)dx) * dfmt.total;
        uint32_t px[4] = {0u, 0u, 0u, 0u};
        if (KIND == 3) {
            const TextureDesc& t = a.src;
            // (uint32_t)u as GetDepthPixel receives it; held inside the level
            const uint32_t sx = min((uint32_t)fmaxf(u, 0.0f), t.level_w[0] - 1u), sy = min((uint32_t)fmaxf(v, 0.0f), t.level_h[0] - 1u);
            uint32_t sw[4];
            read_pixel((const uint8_t*)t.address + t.level_offset[0] + ((uint64_t)sy * t.level_w[0] + sx) * t.fmt.total, t.fmt.total, sw);
            uint32_t dw[4];
            read_pixel(out, a.dfmt.total, dw);
            float depth = a.dfmt.depth_off >= 0 ? unpack_depth(a.dfmt, dw[0]) : 0.0f;
            uint32_t stencil = a.dfmt.stencil_off >= 0 ? get_field(dw, a.dfmt.stencil_off, 1) : 0u;
            if (a.aspect & 2u) depth = unpack_depth(t.fmt, sw[0]);                        // DEPTH
            if (a.aspect & 4u) stencil = t.fmt.stencil_off >= 0 ? get_field(sw, t.fmt.stencil_off, 1) : 0u;   // STENCIL
            if ((a.aspect & 2u) && !(a.aspect & 4u) && a.dfmt.stencil_off < 0) stencil = 0u;
            if ((a.aspect & 4u) && !(a.aspect & 2u) && a.dfmt.depth_off < 0) depth = 0.0f;
            uint32_t d0 = 0u, d1 = 0u;
            pack_depth_stencil(a.dfmt, depth, stencil, d0, d1);
            px[0] = d0;
            px[1] = d1;
        } else if (KIND == 0 || KIND == 4) {
            float c[4];
            sample_level_as<KIND == 4>(src, 0, u / (float)src.level_w[0], v / (float)src.level_h[0], FILTER, c);
            if (src.fmt.off[0] < 0) c[0] = 0.0f;
            if (src.fmt.off[1] < 0) c[1] = 0.0f;
            if (src.fmt.off[2] < 0) c[2] = 0.0f;
            if (src.fmt.off[3] < 0) c[3] = 1.0f;
            pack_color_f32(dfmt, c, px);
        } else {
            // integer formats: the nearest texel's channel values
            const TextureDesc& t = a.src;
            int32_t cx = (int32_t)floorf(u / (float)t.level_w[0] * (float)t.level_w[0]);
            int32_t cy = (int32_t)floorf(v / (float)t.level_h[0] * (float)t.level_h[0]);
            cx = wrap_coord(cx, (int32_t)t.level_w[0], 2);
            cy = wrap_coord(cy, (int32_t)t.level_h[0], 2);
            uint32_t sw[4];
            read_pixel((const uint8_t*)t.address + t.level_offset[0] + ((uint64_t)cy * t.level_w[0] + (uint64_t)cx) * t.fmt.total, t.fmt.total, sw);
            uint32_t ch[4];
            for (int k = 0; k < 4; k++) ch[k] = raw_channel(t.fmt, sw, k);
            if (t.fmt.off[3] < 0) ch[3] = 1u;
            if (KIND == 1) {
                pack_color_u32(a.dfmt, ch, px);
            } else {
                int32_t si[4];
                for (int k = 0; k < 4; k++) {
                    const int sh = 32 - 8 * t.fmt.element;
                    si[k] = (t.fmt.off[k] < 0 || sh <= 0) ? (int32_t)ch[k] : ((int32_t)(ch[k] << sh) >> sh);
                }
                pack_color_i32(a.dfmt, si, px);
            }
        }
        store_pixel(out, stored_bytes(dfmt), px);
    }
}

// A colour blit whose source and destination formats both hold four 8-bit
// UNORM channels in 4 bytes (the common one: mip chains), the same arithmetic
// with the formats and the wrapping folded; a wave takes 64 pixels of a row
// (or of several, when the region is narrower).
// Bound by its vector instructions (two exact divisions, sixteen channels
// unpacked and twelve lerps a pixel): 4096x4096 to 2048x2048 takes 26.4 us,
// 3.2 TB/s (in blit_kernel, with a grid-strided pixel index, 40 us), and the
// levels below 512x512 are 2.4 to 3 us of launch.  Four pixels of a row per
// thread took 41 us: the texel loads of a wave then lie 32 bytes apart.
template <int FILTER>
__global__ __launch_bounds__(256) void blit_unorm8_kernel(BlitArgs a)
{
    TextureDesc& src = a.src;
    src.sampler.address_u = src.sampler.address_v = 2;
    const bool negx = a.d1x < a.d0x, negy = a.d1y < a.d0y;
    const float rx = (float)(a.s1x - a.s0x) / (float)(a.d1x - a.d0x);
    const float ry = (float)(a.s1y - a.s0y) / (float)(a.d1y - a.d0y);
    const uint32_t x = blockIdx.x * blockDim.x + threadIdx.x;
    if (x >= a.w) return;
    const int32_t dx = negx ? (int32_t)x + a.d1x : (int32_t)x + a.d0x;
    const float u = ((float)dx + 0.5f - (float)a.d0x) * rx + (float)a.s0x;
    const float tu = u / (float)src.level_w[0];
    for (uint32_t y = blockIdx.y * blockDim.y + threadIdx.y; y < a.h; y += gridDim.y * blockDim.y) {
        const int32_t dy = negy ? (int32_t)y + a.d1y : (int32_t)y + a.d0y;
        const float v = ((float)dy + 0.5f - (float)a.d0y) * ry + (float)a.s0y;
        float c[4];
        sample_level_as<true>(src, 0, tu, v / (float)src.level_h[0], FILTER, c);
        uint32_t px = 0;
#pragma unroll
        for (int i = 0; i < 4; i++) px |= round_to_u32(minnum(maxnum(c[i], 0.0f), 1.0f) * 255.0f) << (a.dfmt.off[i] * 8);
        global_ptr<uint32_t>((uint64_t)a.dst)[(uint64_t)dy * a.dst_width + (uint64_t)dx] = px;
    }
}

uint32_t grid_for(uint64_t n)
{
    return (uint32_t)std::max<uint64_t>(1, std::min<uint64_t>((n + 255) / 256, 16384));
}

// Threads of a workgroup of 256 that lie along a row of n items: the power of
// two that holds them, at most 64.
uint32_t threads_across(uint64_t n)
{
    uint32_t t = 1;
    while (t < 64u && t < n) t *= 2;
    return t;
}

constexpr uint64_t kFillCached = (128u << 20) / 16;   // 16-byte chunks

// Enqueues rows of a repeated pixel of `size` bytes (dividing 16 and every
// row's address).
int fill_rows(cpv_context* c, uint64_t dst, uint64_t row_bytes, uint64_t pitch, uint32_t rows, uint32_t size, const uint32_t* pixel)
{
    FillArgs a{};
    a.dst = (uint8_t*)(uintptr_t)dst;
    a.row_bytes = row_bytes;
    a.pitch = pitch;
    a.rows = rows;
    a.size = size;
    // the chunks from a row's first aligned address to its end, at most
    a.chunks = rows == 1 ? ((dst & 15u) + row_bytes + 15) / 16 : (15 + row_bytes + 15) / 16;
    for (uint32_t o = 0; o < 16; o += size) std::memcpy((uint8_t*)a.pattern + o, pixel, size);
    void* args[] = {&a};
    // a row's chunks by one to 64 threads, so that narrow rows leave few idle
    // (20 of 16,384 bytes: 16,384 rows in 20 us with 64)
    const uint32_t across = rows == 1 ? 256u : threads_across(a.chunks);
    const dim3 block(across, 256u / across);
    // One run of up to 128 MiB by 1,024 workgroups (64 MiB in 11.1 us, with a
    // chunk per thread 12.1), a longer one, past what the caches take, by a
    // chunk per thread (1 GiB in 154 us, by 1,024 workgroups 224).
    const uint64_t most = rows > 1 ? 64 : a.chunks > kFillCached ? 1u << 23 : 1024;
    const uint64_t gx = std::min<uint64_t>((a.chunks + block.x - 1) / block.x, most);
    const uint32_t gy = std::min<uint32_t>((rows + block.y - 1) / block.y, 16384);
    HIP_TRY(hipLaunchKernel((const void*)fill_rows_kernel, dim3((uint32_t)gx, gy), block, args, 0, c->stream));
    return CPV_OK;
}

}  // namespace

extern "C" int cpv_copy_regions(cpv_context* c, const cpv_copy_region* r, uint32_t count)
{
    if (!c || (!r && count)) return fail(CPV_ERROR_INVALID, "null argument");
    std::lock_guard<std::mutex> g(c->lock);
    note_enqueue(c);
    if (int rc = resolve_pending(c)) return rc;
    HIP_TRY(hipSetDevice(c->device));
    for (uint32_t i = 0; i < count; i++) {
        if (!r[i].rows || !r[i].row_bytes) continue;
        if (r[i].rows > 1 && (r[i].src_pitch < r[i].row_bytes || r[i].dst_pitch < r[i].row_bytes))
            return fail(CPV_ERROR_INVALID, "copy pitch below the row size");
        if (r[i].rows == 1 || (r[i].src_pitch == r[i].row_bytes && r[i].dst_pitch == r[i].row_bytes)) {
            HIP_TRY(hipMemcpyAsync((void*)(uintptr_t)r[i].dst, (const void*)(uintptr_t)r[i].src, r[i].row_bytes * r[i].rows,
                                   hipMemcpyDefault, c->stream));
        } else {
            HIP_TRY(hipMemcpy2DAsync((void*)(uintptr_t)r[i].dst, r[i].dst_pitch, (const void*)(uintptr_t)r[i].src, r[i].src_pitch,
                                     r[i].row_bytes, r[i].rows, hipMemcpyDefault, c->stream));
        }
    }
    return CPV_OK;
}

extern "C" int cpv_fill_buffer(cpv_context* c, uint64_t dst, uint64_t size, uint32_t data)
{
    if (!c || (!dst && size)) return fail(CPV_ERROR_INVALID, "null argument");
    std::lock_guard<std::mutex> g(c->lock);
    note_enqueue(c);
    if (int rc = resolve_pending(c)) return rc;
    HIP_TRY(hipSetDevice(c->device));
    if (size / 4 && (dst & 3u) == 0) {
        if (int rc = fill_rows(c, dst, size / 4 * 4, 0, 1, 4, &data)) return rc;
    } else if (size / 4) {
        return fail(CPV_ERROR_INVALID, "fill destination must be 4-byte aligned");
    }
    if (size % 4) {
        uint8_t* p = (uint8_t*)(uintptr_t)dst;
        void* args[] = {&p, &size, &data};
        HIP_TRY(hipLaunchKernel((const void*)fill_tail_kernel, dim3(1), dim3(64), args, 0, c->stream));
    }
    return CPV_OK;
}

extern "C" int cpv_update_buffer(cpv_context* c, uint64_t dst, const void* data, uint64_t size)
{
    if (!c || ((!dst || !data) && size)) return fail(CPV_ERROR_INVALID, "null argument");
    std::lock_guard<std::mutex> g(c->lock);
    note_enqueue(c);
    if (int rc = resolve_pending(c)) return rc;
    HIP_TRY(hipSetDevice(c->device));
    // through the pinned staging ring, so the caller's memory is free on return
    return stage_upload(c, (void*)(uintptr_t)dst, data, size);
}

extern "C" int cpv_clear_rects(cpv_context* c, const cpv_image_level* image, const uint32_t value[4], const cpv_rect* rects,
                               uint32_t count)
{
    if (!c || !image || !value || (!rects && count)) return fail(CPV_ERROR_INVALID, "null argument");
    FormatDesc f;
    if (!format_desc(image->format, &f)) return fail(CPV_ERROR_UNSUPPORTED, "clear of an unsupported format");
    std::lock_guard<std::mutex> g(c->lock);
    note_enqueue(c);
    if (int rc = resolve_pending(c)) return rc;
    HIP_TRY(hipSetDevice(c->device));
    ClearArgs a{};
    a.base = (uint8_t*)(uintptr_t)image->address;
    a.total = (uint32_t)f.total;
    a.stored = (uint32_t)stored_bytes(f);
    a.width = image->width;
    pack_clear(f, value, a.words);
    // sizes that divide 16, written whole, at addresses they divide
    const bool rows_fill = a.total == a.stored && 16 % a.total == 0 && image->address % a.total == 0;
    for (uint32_t i = 0; i < count; i++) {
        const cpv_rect& r = rects[i];
        if (r.x < 0 || r.y < 0 || (uint64_t)r.x + r.width > image->width || (uint64_t)r.y + r.height > image->height)
            return fail(CPV_ERROR_INVALID, "clear rectangle outside the image");
        if (!r.width || !r.height) continue;
        if (rows_fill) {
            const uint64_t at = image->address + ((uint64_t)r.y * image->width + (uint32_t)r.x) * a.total;
            const uint64_t row = (uint64_t)r.width * a.total;
            // rows without a gap are one
            const bool whole = r.width == image->width;
            if (int rc = fill_rows(c, at, whole ? row * r.height : row, (uint64_t)image->width * a.total, whole ? 1 : r.height, a.total, a.words))
                return rc;
            continue;
        }
        a.x0 = r.x;
        a.y0 = r.y;
        a.w = r.width;
        a.h = r.height;
        void* args[] = {&a};
        HIP_TRY(hipLaunchKernel((const void*)clear_rect_kernel, dim3(grid_for((uint64_t)r.width * r.height)), dim3(256), args, 0, c->stream));
    }
    return CPV_OK;
}

extern "C" int cpv_blit_image(cpv_context* c, const cpv_image_level* src, const cpv_image_level* dst, const cpv_blit_region* regions,
                              uint32_t count, uint32_t filter)
{
    if (!c || !src || !dst || (!regions && count)) return fail(CPV_ERROR_INVALID, "null argument");
    FormatDesc sf, df;
    if (!format_desc(src->format, &sf) || !format_desc(dst->format, &df)) return fail(CPV_ERROR_UNSUPPORTED, "blit of an unsupported format");
    const bool sds = sf.depth_off >= 0 || sf.stencil_off >= 0, dds = df.depth_off >= 0 || df.stencil_off >= 0;
    if (sds != dds) return fail(CPV_ERROR_INVALID, "blit between colour and depth/stencil formats");
    if (sf.total > 16 || df.total > 16 || (!sds && sf.element > 4)) return fail(CPV_ERROR_UNSUPPORTED, "blit of a format wider than 4 bytes per channel");
    const bool integer = sf.base == kBaseUInt || sf.base == kBaseSInt;
    if ((sds || integer) && filter != 0) return fail(CPV_ERROR_INVALID, "depth/stencil and integer blits use VK_FILTER_NEAREST");
    std::lock_guard<std::mutex> g(c->lock);
    note_enqueue(c);
    if (int rc = resolve_pending(c)) return rc;
    HIP_TRY(hipSetDevice(c->device));
    BlitArgs a;
    std::memset(&a, 0, sizeof(a));
    a.src.address = src->address;
    a.src.fmt = sf;
    a.src.level_count = 1;
    a.src.level_offset[0] = 0;
    a.src.level_w[0] = src->width;
    a.src.level_h[0] = src->height;
    a.src.sampler.address_u = a.src.sampler.address_v = 2;   // CLAMP_TO_EDGE
    a.src.sampler.mag_filter = a.src.sampler.min_filter = (int32_t)filter;
    a.dst = (uint8_t*)(uintptr_t)dst->address;
    a.dfmt = df;
    a.dst_width = dst->width;
    a.filter = filter;
    a.src_kind = sds ? 3u : sf.base == kBaseUInt ? 1u : sf.base == kBaseSInt ? 2u : 0u;
    auto unorm8x4 = [](const FormatDesc& f) {
        return f.base == kBaseUNorm && f.element == 1 && f.total == 4 && f.depth_off < 0 && f.stencil_off < 0 &&
               f.off[0] >= 0 && f.off[1] >= 0 && f.off[2] >= 0 && f.off[3] >= 0;
    };
    // sources that sample_level_as<true> reads, and of those to the same kind of format
    const bool plain_src = a.src_kind == 0 && unorm8x4(sf) && plain_extent(src->width, src->height) && src->address % 4 == 0;
    const bool plain = plain_src && unorm8x4(df) && dst->address % 4 == 0;
    for (uint32_t i = 0; i < count; i++) {
        const cpv_blit_region& r = regions[i];
        const int32_t w = std::abs(r.dst[2] - r.dst[0]), h = std::abs(r.dst[3] - r.dst[1]);
        if (!w || !h) continue;
        const int32_t dx0 = std::min(r.dst[0], r.dst[2]), dy0 = std::min(r.dst[1], r.dst[3]);
        if (dx0 < 0 || dy0 < 0 || dx0 + w > (int32_t)dst->width || dy0 + h > (int32_t)dst->height)
            return fail(CPV_ERROR_INVALID, "blit destination outside the image");
        const int32_t sx0 = std::min(r.src[0], r.src[2]), sy0 = std::min(r.src[1], r.src[3]);
        const int32_t sx1 = std::max(r.src[0], r.src[2]), sy1 = std::max(r.src[1], r.src[3]);
        if (sx0 < 0 || sy0 < 0 || sx1 > (int32_t)src->width || sy1 > (int32_t)src->height)
            return fail(CPV_ERROR_INVALID, "blit source outside the image");
        a.s0x = r.src[0]; a.s0y = r.src[1]; a.s1x = r.src[2]; a.s1y = r.src[3];
        a.d0x = r.dst[0]; a.d0y = r.dst[1]; a.d1x = r.dst[2]; a.d1y = r.dst[3];
        a.w = (uint32_t)w;
        a.h = (uint32_t)h;
        a.aspect = r.aspect;
        void* args[] = {&a};
        if (plain) {
            const uint32_t across = threads_across((uint64_t)w);
            const dim3 block(across, 256u / across);
            const uint32_t gx = ((uint32_t)w + block.x - 1) / block.x;
            const uint32_t gy = std::min<uint32_t>(((uint32_t)h + block.y - 1) / block.y, 65535);
            HIP_TRY(hipLaunchKernel(filter ? (const void*)blit_unorm8_kernel<1> : (const void*)blit_unorm8_kernel<0>, dim3(gx, gy), block,
                                    args, 0, c->stream));
            continue;
        }
        const void* fn = a.src_kind == 3 ? (const void*)blit_kernel<3, 0>
                         : a.src_kind == 2 ? (const void*)blit_kernel<2, 0>
                         : a.src_kind == 1 ? (const void*)blit_kernel<1, 0>
                         : plain_src ? (filter ? (const void*)blit_kernel<4, 1> : (const void*)blit_kernel<4, 0>)
                         : filter ? (const void*)blit_kernel<0, 1> : (const void*)blit_kernel<0, 0>;
        HIP_TRY(hipLaunchKernel(fn, dim3(grid_for((uint64_t)w * h)), dim3(256), args, 0, c->stream));
    }
    return CPV_OK;
}
