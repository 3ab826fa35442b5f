"""Points and lines on the GPU against the CPU oracle (ProcessPoints /
ProcessLines, CommandBuffer.Draw.cpp:1315-1508), bit for bit: point lists
with per-vertex gl_PointSize, line lists and strips of several widths,
perspective and affine w, flat / noperspective inputs, indexed lines, a
launch that mixes triangles and lines, lines whose quads defeat the tight
pixel box (zero width, zero length, far-off ends: the whole viewport is
scanned, as the reference does), the recorded batch path, a tile
configuration other than the one points and lines raster with, and the
same scenes through programs translated from SPIR-V."""
from __future__ import annotations

import copy

import numpy as np
import pytest

import oracle_lib
import cpvulkan_amd
from cpvulkan_amd import abi
from cpvulkan_amd import spirv as S
from cpvulkan_amd import workloads as W
from gpu_util import compare, materialize_jobs, oracle_jobs, compare_jobs, render_gpu

pytestmark = pytest.mark.gpu


def _check(ctx, scene, label, count=True):
    print(f"[points/lines] {label}: {scene.width}x{scene.height} prims={scene.primitive_count}", flush=True)
    ref = oracle_lib.render_scene(scene)
    compare(scene, render_gpu(ctx, scene, count=count), ref if count else ref[:2] + (None,), label)


@pytest.mark.parametrize("perspective", [True, False])
@pytest.mark.parametrize("count", [True, False])
def test_points(gpu_ctx, perspective, count):
    _check(gpu_ctx, W.points_scene(600, 256, 160, seed=21, perspective=perspective), f"points persp={perspective}", count)


def test_points_extreme_sizes(gpu_ctx):
    sizes = np.array([0.0, -3.0, 0.25, 1.0, 63.96875, 200.0, 1e9, 1e10, np.inf, np.nan] * 4)
    _check(gpu_ctx, W.points_scene(sizes.size, 200, 120, seed=22, sizes=sizes), "point sizes")


@pytest.mark.parametrize("width", [1.0, 2.5, 4.0, 7.96875])
def test_line_list(gpu_ctx, width):
    _check(gpu_ctx, W.lines_scene(400, 256, 160, seed=23, line_width=width), f"line list w={width}")


@pytest.mark.parametrize("Wd,Ht", [(640, 360), (97, 401)])
@pytest.mark.parametrize("spread", [0.05, 20.0])
def test_thin_lines(gpu_ctx, Wd, Ht, spread):
    """Quads far thinner than a pixel: clip w (and with it the length that normalize divides by) varies by `spread`."""
    s = W.lines_scene(500, Wd, Ht, seed=37, line_width=1.25)
    v = s.draws[0].vertices[0].view(np.float32).reshape(-1, 8)
    w = 0.5 + spread * np.random.default_rng(5).random((v.shape[0], 1), dtype=np.float32)
    v[:, :3] *= w / v[:, 3:4]
    v[:, 3:4] = w
    _check(gpu_ctx, s, f"thin lines {Wd}x{Ht} spread {spread}")


@pytest.mark.parametrize("width", [1.0, 3.0])
@pytest.mark.parametrize("perspective", [True, False])
def test_line_strip(gpu_ctx, width, perspective):
    _check(gpu_ctx, W.lines_scene(300, 240, 136, seed=24, strip=True, line_width=width, perspective=perspective),
           f"line strip w={width} persp={perspective}")


@pytest.mark.parametrize("fs", ["COLOR_FLAT", "COLOR_NOPERSPECTIVE"])
def test_interpolation_modes(gpu_ctx, fs):
    lines = W.lines_scene(300, 200, 120, seed=25, line_width=2.0)
    lines.pipeline["fs"] = abi.FS[fs]
    _check(gpu_ctx, lines, f"lines {fs}")
    tris = W.soup_scene(4000, 200, 120, seed=26)
    tris.pipeline["fs"] = abi.FS[fs]
    v = tris.draws[0].vertices[0].view(np.float32).reshape(-1, 8).copy()
    w = np.random.Generator(np.random.PCG64(5)).uniform(0.5, 2.0, size=v.shape[0]).astype(np.float32)
    v[:, :4] *= w[:, None]
    tris.draws[0].vertices[0] = v.view(np.uint8).reshape(-1)
    _check(gpu_ctx, tris, f"triangles {fs}")


def test_indexed_lines(gpu_ctx):
    s = W.lines_scene(200, 200, 120, seed=27, line_width=1.5)
    rng = np.random.Generator(np.random.PCG64(6))
    d = s.draws[0]
    d.indices = rng.integers(0, d.count, size=3 * d.count).astype(np.uint16)
    d.count = d.indices.size
    _check(gpu_ctx, s, "indexed line list")


def test_triangles_and_lines_in_one_launch(gpu_ctx):
    tri = W.soup_scene(3000, 256, 160, seed=28)
    lin = W.lines_scene(300, 256, 160, seed=29, line_width=2.0)
    s = copy.deepcopy(tri)
    s.pipelines = [tri.pipeline, lin.pipeline]
    s.draws = [tri.draws[0], lin.draws[0], copy.deepcopy(tri.draws[0])]
    s.draw_pipeline = [0, 1, 0]
    _check(gpu_ctx, s, "triangles + lines")


def _explicit_lines(verts: np.ndarray, width: float, Wd=96, Ht=64, depth_compare="LESS") -> W.Scene:
    s = W.lines_scene(1, Wd, Ht, seed=1, line_width=width)
    s.pipeline["depth_compare"] = abi.COMPARE[depth_compare]
    v = np.ascontiguousarray(verts, np.float32)
    s.draws[0].vertices[0] = v.view(np.uint8).reshape(-1)
    s.draws[0].count = v.shape[0]
    return s


def test_degenerate_lines_scan_the_viewport(gpu_ctx):
    F = np.float32
    Wd, Ht = 96, 64
    yf = (F(9) / F(Ht) + (F(1) / F(Ht)) * F(0.5)) * F(2) - F(1)
    c = [0.8, 0.6, 0.4, 1.0]
    v = np.array([
        [-0.5, yf, 0.5, 1.0, *c], [0.1, yf, 0.5, 1.0, *c],            # zero width: the whole row 9
        [0.2, 0.2, 0.3, 1.0, *c], [0.2, 0.2, 0.7, 1.0, *c],           # no extent in x, y: every pixel, NaN depth
        [-30.0, -20.0, 0.4, 1.0, *c], [25.0, 18.0, 0.4, 1.0, *c],     # ends far outside the viewport
        [-0.9, -0.9, 0.2, 1.0, *c], [0.9, 0.9, 0.2, 1.0, *c],         # an ordinary diagonal on top
    ])
    for width in (0.0, 1.0, 3.0):
        _check(gpu_ctx, _explicit_lines(v, width, Wd, Ht), f"degenerate lines w={width}")
    # without the NaN-depth line (NaN encodings are the platform's), every test passes
    keep = np.r_[0:2, 4:8]
    _check(gpu_ctx, _explicit_lines(v[keep], 2.0, Wd, Ht, depth_compare="ALWAYS"), "degenerate lines ALWAYS")


def test_lines_with_another_tile_configuration(gpu_ctx):
    saved = gpu_ctx.config()
    try:
        for tile, waves in ((8, 1), (32, 2)):
            cfg = gpu_ctx.config()
            cfg.tile_size, cfg.waves_per_tile = tile, waves
            gpu_ctx.apply_config(cfg)
            _check(gpu_ctx, W.lines_scene(200, 200, 120, seed=30, line_width=2.0), f"lines with config {tile}x{waves}")
            _check(gpu_ctx, W.points_scene(200, 200, 120, seed=31), f"points with config {tile}x{waves}")
    finally:
        gpu_ctx.apply_config(saved)


def test_batch_with_points_and_lines(gpu_ctx):
    scenes = [W.lines_scene(150, 128, 96, seed=32, line_width=2.0), W.points_scene(150, 96, 64, seed=33),
              W.soup_scene(2000, 128, 128, seed=34)]
    refs = oracle_jobs(scenes)
    mem, ms, jobs = materialize_jobs(gpu_ctx, scenes)
    try:
        with gpu_ctx.batch(jobs) as b:
            for rep in range(2):
                for m in ms:
                    m.reset_attachments()
                b.submit()
                n = b.wait(count=True)
                print(f"[points/lines] batch replay {rep}: {n} fragments", flush=True)
                assert n == sum(r[2] for r in refs)
                compare_jobs(scenes, ms, refs, f"batch replay {rep}")
    finally:
        mem.release()


@pytest.fixture(scope="module")
def programs(gpu_ctx):
    progs = {}
    for vs, fs in [("vs_point_size", "fs_color"), ("vs_passthrough", "fs_color"), ("vs_passthrough", "fs_color_flat"),
                   ("vs_passthrough", "fs_color_noperspective")]:
        print(f"[points/lines] creating program {vs} + {fs}", flush=True)
        progs[(vs, fs)] = cpvulkan_amd.Program(gpu_ctx, S.SHADERS[vs](), S.SHADERS[fs]())
    yield progs
    for p in progs.values():
        p.close()


def _translated(ctx, scene, prog, label):
    s = copy.deepcopy(scene)
    s.pipeline["program"] = prog.handle.value
    print(f"[points/lines] translated {label}", flush=True)
    compare(s, render_gpu(ctx, s), oracle_lib.render_scene(scene), f"translated {label}")


def test_translated_programs(gpu_ctx, programs):
    _translated(gpu_ctx, W.points_scene(400, 200, 120, seed=35), programs[("vs_point_size", "fs_color")], "points")
    lines = W.lines_scene(300, 200, 120, seed=36, line_width=2.5)
    _translated(gpu_ctx, lines, programs[("vs_passthrough", "fs_color")], "lines")
    for fs, kind in (("fs_color_flat", "COLOR_FLAT"), ("fs_color_noperspective", "COLOR_NOPERSPECTIVE")):
        s = copy.deepcopy(lines)
        s.pipeline["fs"] = abi.FS[kind]
        _translated(gpu_ctx, s, programs[("vs_passthrough", fs)], f"lines {kind}")
