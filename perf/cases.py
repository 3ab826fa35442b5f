"""Timed cases of the draw path, through the Python binding of its C-ABI.

A case is one piece of work that a program using this driver hands over: a
render pass, a recorded batch replayed, or the transfer commands around them.
Inputs (vertices, indices, uniforms, textures, attachments) are resident in
device memory, as a Vulkan application's are once it has recorded its command
buffers; `run` hands the descriptors over and returns the attachments.

Kinds of case (`kind`) and what of a real program each stands for:
  cube      the 15-draw_cube sample: 12 triangles, MVP, B8G8R8A8 + D16
  replay    a recorded command buffer (cpv_batch) of a few small render passes,
            what the ICD submits for a reusable command buffer
  soup      triangles of log-normal size in any order, uniform or clustered
            centres, opaque or alpha blended (particles, foliage, UI)
  grid      an indexed, textured, lit heightfield (terrain)
  scene     a pass of many indexed draws with their own transforms, opaque and
            then transparent, with a stencil attachment (a forward renderer)
  overlay   points and lines drawn over what the attachment holds (LOAD)
  jobs      many independent targets of uneven size recorded as one batch
  transfer  a mip chain made by blits, a clear, a fill and padded row copies

The attachments are packed pixels and depths whose every bit the reference's
operation order fixes, so the tolerance of every case is "exact".  `exact`
gives the stored depths of the D32_SFLOAT cases in 64 bits; packed pixels have
no 64-bit counterpart.
"""
from __future__ import annotations

import ctypes as C
import math

import numpy as np
import torch

import cpvulkan_amd
from cpvulkan_amd import abi
from cpvulkan_amd import spirv as S
from cpvulkan_amd import workloads as W

F = abi.FORMAT
DEV = "cuda"

# edge length of a soup triangle in pixels, L ~ LogNormal(log(8), 1): its mean
# covered area is about sqrt(3) / 4 * 64 * e^2 pixels, less the jitter
SOUP_MU, SOUP_SIGMA = math.log(8.0), 1.0
SOUP_AREA = 193.6
# operations a covered pixel cannot do without: three edge functions (5 each),
# three weights, the depth (5) and the depth test
COVER_OPS = 24
# a shaded pixel's four interpolated channels, blend and pack
SHADE_OPS = 60


def listed():
    return [
        # the smallest call: latency and launches count.  The sample's own size, shaders translated from SPIR-V
        dict(name="cube_500", kind="cube", width=500, height=500, program="spirv", count=0),
        # a reusable command buffer of three small passes, replayed; the context's default options (fragments counted)
        dict(name="replay_3x640", kind="replay", passes=3, width=640, height=480, program="builtin", count=1),
        # a small ordinary frame with shaders translated from SPIR-V
        dict(name="soup_3k_600p", kind="soup", tris=3001, width=800, height=600, clusters=0, blend=1, compare="LESS",
             ds="D32_SFLOAT", program="spirv", count=0),
        # the benchmark's frame: a million alpha-blended triangles at 1080p
        dict(name="soup_1m_1080p", kind="soup", tris=1_000_000, width=1920, height=1080, clusters=0, blend=1, compare="LESS",
             ds="D32_SFLOAT", program="builtin", count=0),
        # opaque geometry on a ragged target, the samples' compare op, 16-bit depth, the context's default options
        dict(name="soup_opaque_150k", kind="soup", tris=150_001, width=1366, height=767, clusters=0, blend=0,
             compare="LESS_OR_EQUAL", ds="D16_UNORM", program="builtin", count=1),
        # the largest frame: four million triangles in clusters at 4K
        dict(name="skewed_4m_4k", kind="soup", tris=4_000_000, width=3840, height=2160, clusters=8, blend=1, compare="LESS",
             ds="D32_SFLOAT", program="builtin", count=0),
        # terrain at 4K
        dict(name="grid_512_4k", kind="grid", n=512, width=3840, height=2160, tex=1024, program="builtin", count=0),
        # terrain at 720p with shaders translated from SPIR-V
        dict(name="grid_257_720p", kind="grid", n=257, width=1280, height=720, tex=256, program="spirv", count=0),
        # a forward renderer's pass
        dict(name="scene_192_1080p", kind="scene", draws=192, rings=16, sectors=24, width=1920, height=1080, count=0),
        # points and lines over an existing image
        dict(name="overlay_1080p", kind="overlay", points=20_000, lines=6_001, line_width=1.5, width=1920, height=1080, count=0),
        # many targets of uneven size in one recorded batch, in the tile configuration the autotuner picks for such batches
        dict(name="jobs_48", kind="jobs", jobs=48, lo=12, hi=200_000, max_side=2048, count=0),
        # transfers: mips of a 4096 x 4096 texture, a 4K clear, a fill and a padded copy
        dict(name="transfer_4096", kind="transfer", tex=4096, width=3840, height=2160, fill=64 << 20, rows=2048, row_bytes=6000),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["cube", "replay", "soup", "soup", "soup", "grid", "scene", "overlay", "jobs", "transfer"])
    w, h = _log(rng, 200, 3840), _log(rng, 150, 2160)
    count = rng.choice([0, 0, 1])
    program = rng.choice(["builtin", "spirv"])
    if kind == "cube":
        return dict(kind=kind, width=w, height=h, program=program, count=count)
    if kind == "replay":
        return dict(kind=kind, passes=rng.randint(1, 6), width=min(w, 1920), height=min(h, 1080), program=program, count=count)
    if kind == "soup":
        tris = _log(rng, 100, 2_000_000)
        tris = min(tris, w * h // 2)   # at most about a hundred layers
        blend = rng.randint(0, 1)
        return dict(kind=kind, tris=tris, width=w, height=h, clusters=rng.choice([0, 0, 8]) if tris > 1000 else 0, blend=blend,
                    compare=rng.choice(["LESS", "LESS", "LESS_OR_EQUAL"]),
                    ds=rng.choice(["D32_SFLOAT", "D32_SFLOAT", "D16_UNORM"]), program=program, count=count)
    if kind == "grid":
        return dict(kind=kind, n=_log(rng, 24, 512), width=w, height=h, tex=2 ** rng.randint(5, 10), program=program, count=0)
    if kind == "scene":
        return dict(kind=kind, draws=_log(rng, 8, 256), rings=rng.randint(6, 24), sectors=rng.randint(8, 40), width=w, height=h,
                    count=count)
    if kind == "overlay":
        return dict(kind=kind, points=_log(rng, 100, 40_000), lines=_log(rng, 50, 10_000), line_width=rng.choice([1.0, 1.5, 3.0]),
                    width=w, height=h, count=count)
    if kind == "jobs":
        return dict(kind=kind, jobs=rng.randint(4, 48), lo=12, hi=_log(rng, 1000, 100_000), max_side=rng.choice([512, 1024, 2048]),
                    count=0)
    return dict(kind=kind, tex=_log(rng, 63, 4096), width=w, height=h, fill=_log(rng, 1000, 64 << 20), rows=_log(rng, 10, 2048),
                row_bytes=_log(rng, 64, 6000))


# ------------------------------------------------------------- what a program keeps

_contexts: dict = {}
_programs: dict = {}


def _context(count: int, tile: int = 16, waves: int = 4):
    """One context of the program for each set of options it renders with."""
    key = (count, tile, waves)
    if key not in _contexts:
        ctx = cpvulkan_amd.Context(0)
        ctx.set_config(tile_size=tile, waves_per_tile=waves, count_fragments=count)
        _contexts[key] = ctx
    return _contexts[key]


def _program(ctx, vs: str, fs: str):
    key = (id(ctx), vs, fs)   # contexts live as long as the process
    if key not in _programs:
        _programs[key] = cpvulkan_amd.Program(ctx, S.SHADERS[vs](), S.SHADERS[fs]())
    return _programs[key]


class _Replay:
    """A recorded batch, given back with the state that holds it."""

    def __init__(self, batch):
        self.batch = batch

    def __del__(self):
        self.batch.close()


def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed) & 0x7FFFFFFF)
    return g


def _uniform(g, shape, lo=0.0, hi=1.0):
    return torch.rand(shape, generator=g, device=DEV, dtype=torch.float64) * (hi - lo) + lo


# ------------------------------------------------------------- descriptors

ALPHA = W.ALPHA_BLEND
VEC4 = F["R32G32B32A32_SFLOAT"]
COLOR_LAYOUT = dict(bindings=[(0, 32, 0)], attributes=[(0, 0, VEC4, 0), (1, 0, VEC4, 16)])


def _pipeline(ctx, program, vs, fs, spirv=None, **state):
    p = dict(state)
    if program == "spirv":
        p["program"] = _program(ctx, *spirv).handle
    else:
        p["vs"], p["fs"] = abi.VS[vs], abi.FS[fs]
    return p


DS_DTYPE = {"D32_SFLOAT": torch.float32, "D16_UNORM": torch.int16, "D24_UNORM_S8_UINT": torch.int32}


def _target(width, height, color, ds, clear=(0.0, 0.0, 0.0, 0.0), load="CLEAR", into=None):
    """Attachments of one pass and its descriptor; `into` holds (colour, depth) tensors to use."""
    if into is None:
        c = torch.zeros((height, width), dtype=torch.int32, device=DEV)
        d = torch.zeros((height, width), dtype=DS_DTYPE[ds], device=DEV)
    else:
        c, d = into
    ps = abi.PassDesc()
    ps.width, ps.height, ps.color_count, ps.has_depth_stencil = width, height, 1, 1
    a = ps.color[0]
    a.address, a.format, a.load_op = c.data_ptr(), F[color], abi.LOAD_OP[load]
    for i, v in enumerate(clear):
        a.clear.f32[i] = v
    z = ps.depth_stencil
    z.address, z.format, z.load_op = d.data_ptr(), F[ds], abi.LOAD_OP[load]
    z.clear.ds.depth, z.clear.ds.stencil = 1.0, 0
    return ps, c, d


def _draw(width, height, vertices, count, indices=None, uniforms=(), textures=(), index_size=4):
    d = abi.DrawDesc()
    d.count, d.instance_count = count, 1
    if indices is not None:
        d.indexed, d.index_size, d.index_address = 1, index_size, indices.data_ptr()
    d.vertex_address[0] = vertices.data_ptr()
    d.vertex_bytes[0] = vertices.numel() * vertices.element_size()
    for i, v in enumerate((0.0, 0.0, float(width), float(height), 0.0, 1.0)):
        d.viewport[i] = v
    for b, t in uniforms:
        d.uniform_address[b] = t.data_ptr()
    for b, t, size, levels in textures:
        td = d.textures[b]
        td.address, td.format, td.width, td.height = t.data_ptr(), F["R8G8B8A8_UNORM"], size, size
        td.levels, td.base_level, td.level_count = levels, 0, levels
        s = td.sampler
        s.mag_filter = s.min_filter = abi.FILTER["LINEAR"]
        s.mipmap_mode = 1
        s.address_u = s.address_v = s.address_w = abi.ADDRESS["REPEAT"]
        s.max_lod = float(levels)
    return d


# ------------------------------------------------------------- geometry

def _soup_vertices(g, n, width, height, clusters=0):
    """n triangles as the benchmark's generator draws them (workloads.soup_triangles), on the GPU."""
    if clusters:
        means, sig = _uniform(g, (clusters, 2), -0.8, 0.8), _uniform(g, (clusters,), 0.02, 0.2)
        k = torch.randint(0, clusters, (n,), generator=g, device=DEV)
        c = means[k] + torch.randn((n, 2), generator=g, device=DEV, dtype=torch.float64) * sig[k][:, None]
    else:
        c = _uniform(g, (n, 2), -1.0, 1.0)
    L = torch.exp(torch.randn((n, 1), generator=g, device=DEV, dtype=torch.float64) * SOUP_SIGMA + SOUP_MU)
    ang = _uniform(g, (n, 1), 0.0, 2.0 * math.pi) + torch.arange(3, device=DEV, dtype=torch.float64) * (2.0 * math.pi / 3.0) + \
        _uniform(g, (n, 3), -0.3, 0.3)
    flip = torch.rand((n, 1), generator=g, device=DEV) < 0.5
    ang = torch.where(flip, ang[:, [0, 2, 1]], ang)
    r = L / math.sqrt(3.0)
    v = torch.empty((n, 3, 8), dtype=torch.float32, device=DEV)
    v[:, :, 0] = c[:, 0:1] + r * torch.cos(ang) * (2.0 / width)
    v[:, :, 1] = c[:, 1:2] + r * torch.sin(ang) * (2.0 / height)
    v[:, :, 2] = _uniform(g, (n, 3))
    v[:, :, 3] = 1.0
    v[:, :, 4:7] = _uniform(g, (n, 3, 3))
    v[:, :, 7] = _uniform(g, (n, 3), 0.2, 1.0)
    return v


def _perlin(g, x, y):
    """2-D gradient noise with a lattice drawn from g."""
    ang = _uniform(g, (256 * 256,), 0.0, 2.0 * math.pi)
    gx, gy = torch.cos(ang), torch.sin(ang)

    def at(px, py):
        xi, yi = torch.floor(px).long(), torch.floor(py).long()
        xf, yf = px - xi, py - yi

        def corner(dx, dy):
            k = ((xi + dx) & 255) * 256 + ((yi + dy) & 255)
            return gx[k] * (xf - dx) + gy[k] * (yf - dy)

        u = xf * xf * xf * (xf * (xf * 6.0 - 15.0) + 10.0)
        t = yf * yf * yf * (yf * (yf * 6.0 - 15.0) + 10.0)
        a = corner(0, 0) * (1 - u) + corner(1, 0) * u
        b = corner(0, 1) * (1 - u) + corner(1, 1) * u
        return a * (1 - t) + b * t

    return at


def _grid_geometry(g, n):
    lin = torch.linspace(-1.0, 1.0, n, device=DEV, dtype=torch.float64)
    Z, X = torch.meshgrid(lin, lin, indexing="ij")
    noise, f, eps = _perlin(g, X, Z), 3.0, 1e-3

    def height(x, z):
        return 0.2 * noise((x + 1.0) * f, (z + 1.0) * f)

    dx = (height(X + eps, Z) - height(X - eps, Z)) / (2 * eps)
    dz = (height(X, Z + eps) - height(X, Z - eps)) / (2 * eps)
    N = torch.stack([-dx, torch.ones_like(dx), -dz], dim=-1)
    N = N / N.norm(dim=-1, keepdim=True)
    v = torch.empty((n, n, 8), dtype=torch.float32, device=DEV)
    v[..., 0], v[..., 1], v[..., 2] = X, height(X, Z), Z
    v[..., 3:6] = N
    v[..., 6], v[..., 7] = (X + 1.0) * 2.0, (Z + 1.0) * 2.0
    i = torch.arange(n - 1, device=DEV)
    a = (i[:, None] * n + i[None, :]).reshape(-1)
    b, c, d = a + 1, a + n, a + n + 1
    idx = torch.stack([a, b, c, c, b, d], dim=1).reshape(-1).to(torch.int32)
    return v.reshape(-1, 8).contiguous(), idx.contiguous()


def _noise_mips(g, size):
    """size^2 RGBA8 noise with its box-filtered mip chain, level after level."""
    lv = torch.randint(0, 256, (size, size, 4), generator=g, device=DEV, dtype=torch.int32)
    out = [lv]
    while lv.shape[0] > 1:
        lv = (lv[0::2, 0::2] + lv[1::2, 0::2] + lv[0::2, 1::2] + lv[1::2, 1::2] + 2) // 4
        out.append(lv)
    return torch.cat([x.reshape(-1).to(torch.uint8) for x in out]), len(out)


def _f32(a):
    return torch.from_numpy(np.ascontiguousarray(a, dtype=np.float32).reshape(-1)).to(DEV)


def _sphere(rings, sectors):
    """Indexed sphere: (pos vec4, colour vec4) vertices and 16-bit indices."""
    t = np.linspace(0.0, math.pi, rings + 1)[:, None]
    p = np.linspace(0.0, 2.0 * math.pi, sectors + 1)[None, :]
    x, y, z = np.sin(t) * np.cos(p), np.cos(t) + 0.0 * p, np.sin(t) * np.sin(p)
    v = np.stack([x, y, z, np.ones_like(x), 0.5 + 0.5 * x, 0.5 + 0.5 * y, 0.5 + 0.5 * z, 0.6 + 0.0 * x], axis=-1)
    i, j = np.meshgrid(np.arange(rings), np.arange(sectors), indexing="ij")
    a = (i * (sectors + 1) + j).reshape(-1)
    b, c = a + 1, a + sectors + 1
    return v.reshape(-1, 8).astype(np.float32), np.stack([a, c, b, b, c, c + 1], axis=1).reshape(-1).astype(np.int16)


# ------------------------------------------------------------- prepare

def _cube_mvp(rng, width, height):
    fov = math.radians(45.0) * (height / width if width > height else 1.0)
    eye = np.array([-5.0, 3.0, -10.0]) + rng.uniform(-2.0, 2.0, 3)
    m = W.mat4_mul(W.vulkan_clip(), W.perspective(fov, width / height, 0.1, 100.0))
    return W.mat4_mul(m, W.look_at(eye, (0, 0, 0), (0, -1, 0)))


def _cube_pass(ctx, case, rng):
    w, h = case["width"], case["height"]
    ps, c, d = _target(w, h, "B8G8R8A8_UNORM", "D16_UNORM", clear=(0.2, 0.2, 0.2, 0.2))
    verts, mvp = _f32(W.cube_vertices()), _f32(_cube_mvp(rng, w, h))
    pipe = _pipeline(ctx, case["program"], "MVP_COLOR", "COLOR", ("vs_mvp_color", "fs_color"), front_face=abi.FRONT_FACE["CW"],
                     depth_compare=abi.COMPARE["LESS_OR_EQUAL"], color_format=F["B8G8R8A8_UNORM"], ds_format=F["D16_UNORM"],
                     **COLOR_LAYOUT)
    return (ps, [W.pipeline_desc(pipe)], [_draw(w, h, verts, 36, uniforms=[(0, mvp)])], None), (c, d), (verts, mvp)


def _prep_cube(case, seed):
    ctx = _context(case["count"])
    args, out, keep = _cube_pass(ctx, case, np.random.default_rng(seed))
    return dict(ctx=ctx, args=args, out=dict(color=out[0], depth=out[1]), keep=keep)


def _prep_replay(case, seed):
    ctx = _context(case["count"])
    rng = np.random.default_rng(seed)
    parts = [_cube_pass(ctx, case, rng) for _ in range(case["passes"])]
    torch.cuda.synchronize()
    batch = _Replay(ctx.batch_passes([p[0] for p in parts]))
    return dict(batch=batch, out=dict(color=[p[1][0] for p in parts], depth=[p[1][1] for p in parts]), keep=parts)


def _prep_soup(case, seed):
    ctx = _context(case["count"])
    w, h, n = case["width"], case["height"], case["tris"]
    verts = _soup_vertices(_gen(seed), n, w, h, case["clusters"])
    ps, c, d = _target(w, h, "R8G8B8A8_UNORM", case["ds"])
    pipe = _pipeline(ctx, case["program"], "PASSTHROUGH", "COLOR", ("vs_passthrough", "fs_color"),
                     depth_compare=abi.COMPARE[case["compare"]], blend=ALPHA if case["blend"] else None,
                     color_format=F["R8G8B8A8_UNORM"], ds_format=F[case["ds"]], **COLOR_LAYOUT)
    return dict(ctx=ctx, args=(ps, [W.pipeline_desc(pipe)], [_draw(w, h, verts, 3 * n)], None), out=dict(color=c, depth=d),
                keep=verts)


def _grid_orbit(seed):
    return float(np.random.default_rng(seed).uniform(0.0, 360.0))


def _prep_grid(case, seed):
    ctx = _context(case["count"])
    w, h = case["width"], case["height"]
    g = _gen(seed)
    verts, idx = _grid_geometry(g, case["n"])
    tex, levels = _noise_mips(g, case["tex"])
    mvp = _f32(W.grid_mvp(w, h, _grid_orbit(seed)))
    light = np.array([0.3, 0.9, -0.2]) / np.linalg.norm([0.3, 0.9, -0.2])
    light = _f32(np.concatenate([light, [0.0]]))
    ps, c, d = _target(w, h, "R8G8B8A8_UNORM", "D32_SFLOAT")
    pipe = _pipeline(ctx, case["program"], "MVP_LAMBERT", "TEX_LAMBERT", ("vs_mvp_lambert", "fs_tex_lambert"),
                     bindings=[(0, 32, 0)], attributes=[(0, 0, F["R32G32B32_SFLOAT"], 0), (1, 0, F["R32G32B32_SFLOAT"], 12),
                                                        (2, 0, F["R32G32_SFLOAT"], 24)],
                     color_format=F["R8G8B8A8_UNORM"], ds_format=F["D32_SFLOAT"])
    dr = _draw(w, h, verts, idx.numel(), indices=idx, uniforms=[(0, mvp), (2, light)], textures=[(1, tex, case["tex"], levels)])
    return dict(ctx=ctx, args=(ps, [W.pipeline_desc(pipe)], [dr], None), out=dict(color=c, depth=d),
                keep=(verts, idx, tex, mvp, light))


def _prep_scene(case, seed):
    ctx = _context(case["count"])
    rng = np.random.default_rng(seed)
    w, h, n = case["width"], case["height"], case["draws"]
    v, i = _sphere(case["rings"], case["sectors"])
    verts, idx = _f32(v), torch.from_numpy(i).to(DEV)
    proj = W.mat4_mul(W.vulkan_clip(), W.perspective(math.radians(60.0), w / h, 0.1, 100.0))
    view = W.mat4_mul(proj, W.look_at((0.0, 2.0, -9.0), (0, 0, 0), (0, 1, 0)))
    mvps = np.zeros((n, 64), np.float32)   # one 256-byte uniform slot for each draw
    for k in range(n):
        m = np.zeros((4, 4), np.float32)
        s = rng.uniform(0.15, 0.9, 3)
        m[0][0], m[1][1], m[2][2], m[3][3] = s[0], s[1], s[2], 1.0
        m[3][:3] = rng.uniform(-1.0, 1.0, 3) * (6.0, 3.0, 4.0)
        mvps[k, :16] = W.mat4_mul(view, m).reshape(-1)
    uni = _f32(mvps).reshape(n, 64)
    ps, c, d = _target(w, h, "R8G8B8A8_UNORM", "D24_UNORM_S8_UINT", clear=(0.1, 0.2, 0.3, 1.0))
    common = dict(cull=abi.CULL["BACK"], depth_compare=abi.COMPARE["LESS_OR_EQUAL"], color_format=F["R8G8B8A8_UNORM"],
                  ds_format=F["D24_UNORM_S8_UINT"], vs=abi.VS["MVP_COLOR"], fs=abi.FS["COLOR"], **COLOR_LAYOUT)
    st = abi.STENCIL
    mark = (st["KEEP"], st["REPLACE"], st["KEEP"], abi.COMPARE["ALWAYS"], 255, 255, 1)
    seen = (st["KEEP"], st["KEEP"], st["KEEP"], abi.COMPARE["ALWAYS"], 255, 255, 1)
    opaque = dict(common, stencil_test=1, front=mark, back=mark)
    clear = dict(common, stencil_test=1, front=seen, back=seen, depth_write=0, blend=ALPHA)
    draws = [_draw(w, h, verts, idx.numel(), indices=idx, index_size=2, uniforms=[(0, uni[k])]) for k in range(n)]
    which = [0 if k < n - n // 4 else 1 for k in range(n)]   # the last quarter is transparent
    return dict(ctx=ctx, args=(ps, [W.pipeline_desc(opaque), W.pipeline_desc(clear)], draws, which),
                out=dict(color=c, depth_stencil=d), keep=(verts, idx, uni))


def _prep_overlay(case, seed):
    ctx = _context(case["count"])
    w, h, g = case["width"], case["height"], _gen(seed)
    color0 = torch.randint(-2**31, 2**31 - 1, (h, w), generator=g, device=DEV, dtype=torch.int32)
    depth0 = torch.rand((h, w), generator=g, device=DEV) * 0.5 + 0.5
    n, m = case["points"], case["lines"]

    def clip(ndc):
        k = ndc.shape[0]
        cw = _uniform(g, (k, 1), 0.5, 2.0)
        z = _uniform(g, (k, 1))
        return torch.cat([ndc * cw, z * cw, cw, _uniform(g, (k, 3)), _uniform(g, (k, 1), 0.2, 1.0)], dim=1)

    pts = torch.cat([clip(_uniform(g, (n, 2), -1.1, 1.1)), _uniform(g, (n, 1), 0.5, 14.0)], dim=1).float().contiguous()
    a = _uniform(g, (m, 2), -1.1, 1.1)
    length = torch.exp(torch.randn((m, 1), generator=g, device=DEV, dtype=torch.float64) * 0.8 + math.log(40.0))
    ang = _uniform(g, (m, 1), 0.0, 2.0 * math.pi)
    b = a + torch.cat([length * torch.cos(ang) * 2.0 / w, length * torch.sin(ang) * 2.0 / h], dim=1)
    lns = clip(torch.stack([a, b], dim=1).reshape(-1, 2)).float().contiguous()
    ps, c, d = _target(w, h, "R8G8B8A8_UNORM", "D32_SFLOAT", load="LOAD", into=(color0.clone(), depth0.clone()))
    common = dict(fs=abi.FS["COLOR"], blend=ALPHA, color_format=F["R8G8B8A8_UNORM"], ds_format=F["D32_SFLOAT"])
    points = dict(common, vs=abi.VS["PASSTHROUGH_POINT"], topology=abi.TOPOLOGY["POINT_LIST"], bindings=[(0, 36, 0)],
                  attributes=[(0, 0, VEC4, 0), (1, 0, VEC4, 16), (2, 0, F["R32_SFLOAT"], 32)])
    lines = dict(common, vs=abi.VS["PASSTHROUGH"], topology=abi.TOPOLOGY["LINE_LIST"], line_width=case["line_width"], **COLOR_LAYOUT)
    # the image under the overlay is put back first, as a program does that draws it over its last frame's base
    copies = [abi.CopyRegion(color0.data_ptr(), c.data_ptr(), 0, 0, 4 * w * h, 1, 0),
              abi.CopyRegion(depth0.data_ptr(), d.data_ptr(), 0, 0, 4 * w * h, 1, 0)]
    return dict(ctx=ctx, copies=copies, args=(ps, [W.pipeline_desc(points), W.pipeline_desc(lines)],
                                              [_draw(w, h, pts, n), _draw(w, h, lns, 2 * m)], [0, 1]),
                out=dict(color=c, depth=d), keep=(color0, depth0, pts, lns))


def _job_sizes(case):
    rng = np.random.default_rng(case["jobs"] * 1000 + case["max_side"])   # the sizes are the case's, the triangles the seed's
    counts = W.zipf_counts(case["jobs"], rng, lo=case["lo"], hi=case["hi"])
    sides = [s for s in (256, 512, 1024, 2048, 4096) if s <= case["max_side"]]
    return counts, rng.choice(np.asarray(sides), size=case["jobs"])


def _prep_jobs(case, seed):
    ctx = _context(case["count"], 16, 1)
    counts, sides = _job_sizes(case)
    g = _gen(seed)
    px = int((sides.astype(np.int64) ** 2).sum())
    color = torch.zeros(px, dtype=torch.int32, device=DEV)   # the targets end to end
    depth = torch.zeros(px, dtype=torch.float32, device=DEV)
    jobs, keep, at = [], [], 0
    pipe = _pipeline(ctx, "builtin", "PASSTHROUGH", "COLOR", depth_compare=abi.COMPARE["LESS"], blend=ALPHA,
                     color_format=F["R8G8B8A8_UNORM"], ds_format=F["D32_SFLOAT"], **COLOR_LAYOUT)
    pd = W.pipeline_desc(pipe)
    for n, side in zip(counts.tolist(), sides.tolist()):
        verts = _soup_vertices(g, n, side, side)
        into = (color[at:at + side * side], depth[at:at + side * side])
        at += side * side
        j = abi.JobDesc()
        j.pass_, j.pipeline, j.draw = _target(side, side, "R8G8B8A8_UNORM", "D32_SFLOAT", into=into)[0], pd, _draw(side, side, verts, 3 * n)
        jobs.append(j)
        keep.append(verts)
    torch.cuda.synchronize()
    return dict(batch=_Replay(ctx.batch(jobs)), out=dict(color=color, depth=depth), keep=keep)


def _levels(size):
    out = [size]
    while out[-1] > 1:
        out.append(out[-1] // 2)
    return out


def _prep_transfer(case, seed):
    ctx = _context(1)
    g = _gen(seed)
    rgba = F["R8G8B8A8_UNORM"]
    sizes = _levels(case["tex"])
    offs = np.concatenate([[0], np.cumsum([4 * s * s for s in sizes])])
    chain = torch.zeros(int(offs[-1]), dtype=torch.uint8, device=DEV)
    chain[: int(offs[1])] = torch.randint(0, 256, (int(offs[1]),), generator=g, device=DEV, dtype=torch.uint8)
    levels = [abi.ImageLevel(chain.data_ptr() + int(o), rgba, s, s, 0) for o, s in zip(offs, sizes)]
    blits = [(levels[k], levels[k + 1],
              [abi.BlitRegion((C.c_int32 * 4)(0, 0, sizes[k], sizes[k]), (C.c_int32 * 4)(0, 0, sizes[k + 1], sizes[k + 1]), 1, 0)])
             for k in range(len(sizes) - 1)]
    w, h = case["width"], case["height"]
    image = torch.zeros((h, w), dtype=torch.int32, device=DEV)
    value = np.random.default_rng(seed).uniform(0.0, 1.0, 4).astype(np.float32)
    word = int(np.random.default_rng(seed + 1).integers(0, 2**32))
    nfill = case["fill"] // 4 * 4
    fill = torch.zeros(nfill // 4, dtype=torch.int32, device=DEV)
    rows, rb = case["rows"], case["row_bytes"]
    src = torch.randint(0, 256, (rows, rb), generator=g, device=DEV, dtype=torch.uint8)
    dst = torch.zeros((rows, rb + 72), dtype=torch.uint8, device=DEV)   # a padded destination, as buffer rows are
    copy = [abi.CopyRegion(src.data_ptr(), dst.data_ptr(), rb, rb + 72, rb, rows, 0)]
    return dict(ctx=ctx, blits=blits, image=abi.ImageLevel(image.data_ptr(), rgba, w, h, 0), value=[int(v) for v in value.view(np.uint32)],
                rect=[abi.Rect(0, 0, w, h)], fill=(fill.data_ptr(), nfill, word), copy=copy,
                out=dict(mips=chain, image=image, fill=fill, rows=dst), keep=src)


def prepare(case, seed):
    state = globals()["_prep_" + case["kind"]](case, seed)
    torch.cuda.synchronize()   # the uploads are done before the first frame
    return state


# ------------------------------------------------------------- run

def run(state):
    if "batch" in state:
        state["batch"].batch.submit()
        return state["out"]
    ctx = state["ctx"]
    if "blits" in state:
        for src, dst, regions in state["blits"]:
            ctx.blit_image(src, dst, regions, abi.FILTER["LINEAR"])
        ctx.clear_rects(state["image"], state["value"], state["rect"])
        ctx.fill_buffer(*state["fill"])
        ctx.copy_regions(state["copy"])
        return state["out"]
    if "copies" in state:
        ctx.copy_regions(state["copies"])
    ctx.render_pass(*state["args"])
    return state["out"]


# ------------------------------------------------------------- what it comes to

def work(case):
    """Attachments written once (and read once where loaded), geometry, indices and textures read once; operations of every covered
    pixel, and of the shading of about one layer (expected values, from the distributions)."""
    kind = case["kind"]
    if kind == "transfer":
        tex = 4 * sum(s * s for s in _levels(case["tex"]))
        b = 2 * tex + 4 * case["width"] * case["height"] + case["fill"] + 2 * case["rows"] * case["row_bytes"]
        return dict(bytes=b, flops=tex * 8)
    if kind == "jobs":
        counts, sides = _job_sizes(case)
        px, tris = int((sides.astype(np.int64) ** 2).sum()), int(counts.sum())
        return dict(bytes=8 * px + 96 * tris, flops=tris * SOUP_AREA * COVER_OPS + px * SHADE_OPS)
    px = case["width"] * case["height"]
    if kind in ("cube", "replay"):
        n = case.get("passes", 1)
        return dict(bytes=n * (6 * px + 36 * 32), flops=n * 0.15 * px * (COVER_OPS + SHADE_OPS))
    if kind == "soup":
        ds = 2 if case["ds"] == "D16_UNORM" else 4
        return dict(bytes=(4 + ds) * px + 96 * case["tris"], flops=case["tris"] * SOUP_AREA * COVER_OPS + px * SHADE_OPS)
    if kind == "grid":
        n = case["n"]
        return dict(bytes=8 * px + 32 * n * n + 24 * (n - 1) ** 2 + 4 * case["tex"] ** 2, flops=px * (COVER_OPS + 250))
    if kind == "scene":
        verts, tris = (case["rings"] + 1) * (case["sectors"] + 1), 2 * case["rings"] * case["sectors"]
        return dict(bytes=8 * px + 32 * verts + 6 * tris + 64 * case["draws"],
                    flops=case["draws"] * (0.004 * px * (COVER_OPS + SHADE_OPS) + verts * 28))
    return dict(bytes=4 * 8 * px + 36 * case["points"] + 64 * case["lines"],
                flops=(case["points"] * 70 + case["lines"] * 60 * case["line_width"]) * (COVER_OPS + SHADE_OPS))


def tolerance(case):
    # packed pixels, depths and copied bytes: every bit is fixed by the order of operations
    return "exact"


def _min_depth(clip, tris, width, height):
    """Smallest depth of the triangles over every pixel centre they cover (1 where none does), in 64 bits: what a LESS or
    LESS_OR_EQUAL test over a cleared attachment leaves.  clip [n, 4], tris [m, 3]."""
    ndc = clip[:, :3] / clip[:, 3:4]
    size = torch.tensor([width, height], device=clip.device, dtype=torch.float64)
    out = torch.full((height * width,), 1.0, device=clip.device, dtype=torch.float64)
    px = torch.trunc((ndc[:, :2] + 1.0) * 0.5 * size).clamp(-1e9, 1e9)
    lo = px[tris].amin(1).clamp_min(0).long()
    hi = torch.minimum(px[tris].amax(1) + 1, size).long()
    ext = (hi - lo).clamp_min(0)
    n = ext[:, 0] * ext[:, 1]
    first = torch.cat([torch.zeros(1, device=clip.device, dtype=torch.long), torch.cumsum(n, 0)])
    at, end = 0, tris.shape[0]
    while at < end:
        stop = int(torch.searchsorted(first, first[at] + (1 << 24), right=True)) - 1
        stop = min(max(stop, at + 1), end)
        k = torch.repeat_interleave(torch.arange(at, stop, device=clip.device), n[at:stop])
        off = torch.arange(k.numel(), device=clip.device) - (first[k] - first[at])
        x, y = lo[k, 0] + off % ext[k, 0].clamp_min(1), lo[k, 1] + off // ext[k, 0].clamp_min(1)
        cx, cy = (x + 0.5) / width * 2.0 - 1.0, (y + 0.5) / height * 2.0 - 1.0
        P = ndc[tris[k]]

        def edge(a, b):
            return (cx - P[:, a, 0]) * (P[:, b, 1] - P[:, a, 1]) - (cy - P[:, a, 1]) * (P[:, b, 0] - P[:, a, 0])

        e = torch.stack([edge(1, 2), edge(2, 0), edge(0, 1)], dim=1)
        area = e.sum(1)
        e = e * torch.sign(area)[:, None]
        inside = (e >= 0).all(1) & (area != 0)
        z = (e * P[:, :, 2]).sum(1) / area.abs().clamp_min(1e-300)
        out.scatter_reduce_(0, (y * width + x)[inside], z[inside], "amin")
        at = stop
    return out.reshape(height, width)


def exact(case, seed):
    if case["kind"] == "soup" and case["ds"] == "D32_SFLOAT":
        v = _soup_vertices(_gen(seed), case["tris"], case["width"], case["height"], case["clusters"]).reshape(-1, 8)
        tris = torch.arange(3 * case["tris"], device=DEV).reshape(-1, 3)
        return dict(color=None, depth=_min_depth(v[:, :4].double(), tris, case["width"], case["height"]))
    if case["kind"] == "grid":
        v, idx = _grid_geometry(_gen(seed), case["n"])
        m = _f32(W.grid_mvp(case["width"], case["height"], _grid_orbit(seed))).reshape(4, 4).double()
        pos = torch.cat([v[:, :3].double(), torch.ones((v.shape[0], 1), device=DEV, dtype=torch.float64)], dim=1)
        return dict(color=None, depth=_min_depth(pos @ m, idx.long().reshape(-1, 3), case["width"], case["height"]))
    if case["kind"] == "jobs":
        counts, sides = _job_sizes(case)
        g, parts = _gen(seed), []
        for n, side in zip(counts.tolist(), sides.tolist()):
            v = _soup_vertices(g, n, side, side).reshape(-1, 8)
            parts.append(_min_depth(v[:, :4].double(), torch.arange(3 * n, device=DEV).reshape(-1, 3), side, side).reshape(-1))
        return dict(color=None, depth=torch.cat(parts))
    return None
