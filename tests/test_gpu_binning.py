"""Binning paths against the oracle at the sizes where they change (GPU
only): small launches, whose tile lists one kernel writes (one wavefront per
tile up to 256 primitives per target, a workgroup above; at most 4,096
primitives and 2^23 (tile, primitive) tests), and the scan, emit and sort
kernels beyond (one pass of the sort per 8 bits of the tile count; a scan
round per 4,096 workgroups of 256 primitives)."""
import copy

import numpy as np
import pytest

import oracle_lib
import scenes as S
from gpu_util import compare, compare_jobs, materialize_jobs, oracle_jobs, render_gpu
from cpvulkan_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.fixture
def ctx():
    import cpvulkan_amd
    c = cpvulkan_amd.Context(0)
    yield c
    c.close()


def _check(ctx, scene, label, tile=16, waves=4, count=True):
    print(f"[binning] {label}", flush=True)
    ctx.set_config(tile_size=tile, waves_per_tile=waves)
    ref = oracle_lib.render_scene(scene, threads=oracle_lib.default_threads())
    for k in range(2):   # a second call uses the other buffer set
        compare(scene, render_gpu(ctx, scene, count=count), ref if count else (ref[0], ref[1], None), f"{label} call {k}")


@pytest.mark.parametrize("n", [0, 1, 63, 64, 65, 255, 256, 257, 511, 513, 4095, 4096, 4097, 9000])
@pytest.mark.parametrize("tile,waves", [(16, 4), (8, 1), (32, 2)])
def test_primitive_counts(ctx, n, tile, waves):
    s = S.soup(max(n, 1), 150, 101, seed=n)
    s.draws[0].count = 3 * n
    _check(ctx, s, f"{n} triangles {tile}x{waves}", tile, waves)


@pytest.mark.parametrize("n", [1027, 1028, 1029])   # 8,160 tiles: 2^23 tests lie between 1,028 and 1,029
def test_list_limit(ctx, n):
    _check(ctx, S.soup(n, 1920, 1080, seed=n), f"{n} triangles at 1080p")


@pytest.mark.parametrize("w,h,tile", [(16, 16, 16), (17, 16, 16), (256, 256, 16), (257, 256, 16), (4096, 16, 16), (2056, 2048, 8)])
def test_tile_counts(ctx, w, h, tile):
    """1, 2, 256, 272, 256 and 65,792 tiles: one, two and three sort passes, and a sort of one key."""
    _check(ctx, S.soup(6000, w, h, seed=w + h), f"{w}x{h} in {tile}x{tile} tiles", tile, {16: 4, 8: 1}[tile], count=False)


@pytest.mark.parametrize("n", [40, 3000])
def test_several_draws_and_kinds(ctx, n):
    """Draws that end inside a workgroup's 256 primitives; large primitives among small ones; dropped ones (culled)."""
    s = S.soup(n, 333, 211, seed=4)
    parts = [s, S.soup(n + 257, 333, 211, seed=5, size_px=np.log(300.0)), S.soup(n + 1, 333, 211, seed=6)]
    s = copy.deepcopy(s)
    s.draws = [p.draws[0] for p in parts]
    s.pipeline["cull"] = 2
    _check(ctx, s, f"three draws of about {n}")


@pytest.mark.parametrize("counts", [(1, 300, 12), (5000, 3, 700, 1), (4096, 4096)])
def test_targets_of_uneven_size(ctx, counts):
    scenes = [W.soup_scene(n, 64 + 50 * k, 90 - 20 * k, seed=20 + k) for k, n in enumerate(counts)]
    refs = oracle_jobs(scenes)
    mem, ms, jobs = materialize_jobs(ctx, scenes)
    try:
        ctx.render_jobs(jobs)
        ctx.synchronize()
        assert ctx.fragment_count() == sum(r[2] for r in refs)
        compare_jobs(scenes, ms, refs, "jobs")
        for m in ms:
            m.reset_attachments()
        with ctx.batch(jobs) as b:
            for _ in range(3):
                b.submit()
            assert b.wait(count=True) == sum(r[2] for r in refs)
        compare_jobs(scenes, ms, refs, "batch")
    finally:
        mem.release()


@pytest.mark.parametrize("n", [200, 3000, 20_000])
def test_allocation_free_call(ctx, n):
    from cpvulkan_amd.workloads import DeviceMemory, materialize
    s = S.soup(n, 640, 360, seed=n)
    ref = oracle_lib.render_scene(s, threads=oracle_lib.default_threads())
    mem = DeviceMemory(ctx)
    try:
        m = materialize(s, mem)
        for _ in range(2):
            m.reset_attachments()
            ctx.render_pass_noalloc(m.pass_desc, m.pipelines, m.draws)
            ctx.synchronize()
            compare(s, (m.read_color(), m.read_ds(), ctx.fragment_count()), ref, f"noalloc {n}")
    finally:
        mem.release()


def test_more_setup_workgroups_than_a_scan_round(ctx):
    """4,200 workgroups of setup: the scan of their sums takes a second round."""
    s = S.soup(4200 * 256 - 5, 320, 200, seed=8, size_px=np.log(2.0))
    _check(ctx, s, "1.07M small triangles", count=False)


@pytest.mark.parametrize("op", ["LESS", "LESS_OR_EQUAL", "GREATER"])
@pytest.mark.parametrize("tile,waves", [(16, 4), (16, 1), (32, 4), (8, 1)])
def test_list_lengths(ctx, tile, waves, op):
    """Lists around the sizes at which the raster kernel packs their candidates (64) and reads them (256 at a time), and
    chunks of candidates around 16 and 64, at list starts that are no multiple of four."""
    for n in (1, 15, 17, 63, 64, 65, 66, 127, 200, 255, 257, 320, 519, 1025):
        s = S.soup(n, 40, 33, seed=n, size_px=np.log(24.0))
        s.pipeline["depth_compare"] = {"LESS": 1, "LESS_OR_EQUAL": 3, "GREATER": 4}[op]
        s.clear_depth = 0.0 if op == "GREATER" else 1.0
        _check(ctx, s, f"lists of up to {n} {op} {tile}x{waves}", tile, waves, count=False)
    _check(ctx, s, f"lists of up to {n} {op} {tile}x{waves} counting", tile, waves)


@pytest.mark.parametrize("tile,waves", [(16, 1), (32, 1), (32, 2), (32, 4)])
@pytest.mark.parametrize("n,w,h,size", [(4200, 333, 211, 40.0), (4200, 40, 33, 16.0), (250_000, 640, 360, 6.0)])
def test_long_tiles(ctx, tile, waves, n, w, h, size):
    """Waves that hold four blocks or more take long tiles (256 pairs) block by block: tiles on both sides of the rule, all
    tiles long, and more units of work than the 2,048 workgroups that take them; recorded batches and allocation-free
    calls."""
    s = S.soup(n, w, h, seed=n + w, size_px=np.log(size))
    _check(ctx, s, f"{n} triangles {w}x{h} {tile}x{waves}", tile, waves)
    ref = oracle_lib.render_scene(s, threads=oracle_lib.default_threads())
    mem, ms, jobs = materialize_jobs(ctx, [s])
    try:
        with ctx.batch(jobs) as b:
            for _ in range(3):
                b.submit()
            assert b.wait(count=True) == ref[2]
        compare_jobs([s], ms, [ref], "batch")
        if n < 10_000:
            for m in ms:
                m.reset_attachments()
            ctx.render_pass_noalloc(ms[0].pass_desc, ms[0].pipelines, ms[0].draws)
            ctx.synchronize()
            compare_jobs([s], ms, [ref], "noalloc")
    finally:
        mem.release()


@pytest.mark.parametrize("tile,waves,side", [(16, 1, 640), (32, 1, 1280), (32, 4, 640)])
def test_some_tiles_split(ctx, tile, waves, side):
    """A launch that fills the chip: of lists on both sides of the least length only those far beyond the mean are split."""
    s = S.soup(250_000, side, side, seed=tile + waves, size_px=np.log(5.0))
    rng = np.random.default_rng(9)
    centres = rng.normal(0.3, 0.01, (20_000, 2))
    v = W.soup_triangles(20_000, side, side, 5, centres=centres, mu_px=np.log(5.0))
    s = copy.deepcopy(s)
    d = copy.deepcopy(s.draws[0])
    d.vertices = {0: v.view(np.uint8).reshape(-1)}
    d.count = v.shape[0]
    s.draws.append(d)
    _check(ctx, s, f"{side}x{side} {tile}x{waves}", tile, waves)


@pytest.mark.parametrize("sizes", [(255, 1, 256, 257), (0, 3, 0, 600, 0), (2,) * 2600, (1, 0, 5000, 0, 0, 1, 300, 2)])
@pytest.mark.parametrize("tile,waves", [(16, 4), (8, 1)])
def test_draws_that_share_setup_workgroups(ctx, sizes, tile, waves):
    """Workgroups of 256 primitives over draws that begin anywhere in them, empty ones and several viewports among them; small
    launches and, by a fourth of the draws again, ones that bin pairs."""
    s = S.soup(4, 150, 101, seed=1)
    full = S.soup(max(sum(sizes), 1), 150, 101, seed=5, size_px=np.log(6.0)).draws[0].vertices[0].view(np.float32).reshape(-1, 3, 8)
    s.draws, at = [], 0
    for k, n in enumerate(sizes):
        d = copy.deepcopy(S.soup(1, 150, 101, seed=1).draws[0])
        d.vertices = {0: np.ascontiguousarray(full[at:at + max(n, 1)]).view(np.uint8).reshape(-1)}
        d.count, at = 3 * n, min(at + n, full.shape[0] - 1)
        if k % 3 == 1:
            d.viewport = (3.0, 2.0, 120.0, 90.0, 0.0, 1.0)
        s.draws.append(d)
    _check(ctx, s, f"{len(sizes)} draws {tile}x{waves}", tile, waves)


def test_targets_that_share_setup_workgroups(ctx):
    """Jobs of a few triangles to targets of different widths: a workgroup's primitives are of many targets."""
    scenes = [W.soup_scene(1 + k % 7, 40 + 16 * (k % 5), 30 + 8 * (k % 3), seed=100 + k) for k in range(300)]
    scenes.append(W.soup_scene(5000, 320, 200, seed=99))   # beyond what the small launches' lists take
    refs = oracle_jobs(scenes)
    mem, ms, jobs = materialize_jobs(ctx, scenes)
    try:
        print("[binning] 301 jobs", flush=True)
        ctx.render_jobs(jobs)
        ctx.synchronize()
        assert ctx.fragment_count() == sum(r[2] for r in refs)
        compare_jobs(scenes, ms, refs, "jobs")
    finally:
        mem.release()
