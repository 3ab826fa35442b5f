"""One shading pass of a wave holds fragments of different draws: each must
be shaded with its own draw's texture, sampler, uniforms and blend state
(bit-exact with the oracle; GPU only).  Overlapping textured grids a few
pixels per triangle, every draw with a texture of its own size (powers of two
and not), filter, address mode and light, under two pipelines."""
import numpy as np
import pytest

import oracle_lib
import scenes as S
from gpu_util import compare, render_gpu
from cpvulkan_amd import abi
from cpvulkan_amd import workloads as W

pytestmark = pytest.mark.gpu

MODES = ["REPEAT", "MIRRORED_REPEAT", "CLAMP_TO_EDGE", "CLAMP_TO_BORDER", "MIRROR_CLAMP_TO_EDGE"]


def _scene(draws, op):
    rng = np.random.default_rng(draws)
    scenes = [W.grid_scene(n=12, width=112, height=72, seed=3 + k, tex_size=4, orbit_deg=30.0 * k) for k in range(draws)]
    s, own = scenes[0], [g.draws[0] for g in scenes]
    s.draws = []
    for k, d in enumerate(own):
        w, h = [(5, 12), (16, 3), (1, 1), (32, 32), (7, 64)][k % 5]
        d.textures[1] = W.TextureData(
            data=rng.integers(0, 256, w * h * 4, dtype=np.uint8), width=w, height=h, levels=1,
            format=abi.FORMAT["R8G8B8A8_UNORM" if k % 3 else "B8G8R8A8_UNORM"],
            sampler=dict(mag=k % 2, min=0, address_u=abi.ADDRESS[MODES[k % 5]], address_v=abi.ADDRESS[MODES[(k // 2) % 5]], border=k % 6))
        light = rng.normal(size=4).astype(np.float32)
        d.uniforms[2] = light.view(np.uint8)
        s.draws.append(d)
    plain = dict(s.pipeline, depth_compare=abi.COMPARE[op])
    s.pipelines = [plain, dict(plain, blend=W.ALPHA_BLEND, depth_write=0)]
    s.draw_pipeline = [(k // 2) % 2 for k in range(draws)]
    return s


@pytest.mark.parametrize("tile,waves", [(16, 4), (32, 4), (8, 1)])
@pytest.mark.parametrize("op,ds", [("LESS", "D32_SFLOAT"), ("LESS_OR_EQUAL", "D16_UNORM"), ("LESS", "D24_UNORM_S8_UINT"),
                                   ("GREATER_OR_EQUAL", "D32_SFLOAT_S8_UINT")])
def test_fragments_of_many_draws(gpu_ctx, op, ds, tile, waves):
    s = _scene(14, op)
    s.ds_format = abi.FORMAT[ds]
    s.clear_depth = 0.0 if op.startswith("GREATER") else 1.0
    ref = oracle_lib.render_scene(s)
    gpu_ctx.set_config(tile_size=tile, waves_per_tile=waves)
    try:
        print(f"[groups] {op} {ds} {tile}x{waves}", flush=True)
        compare(s, render_gpu(gpu_ctx, s), ref, "counting")
        compare(s, render_gpu(gpu_ctx, s, count=False), (ref[0], ref[1], None), "culling on")
    finally:
        gpu_ctx.set_config()


@pytest.mark.parametrize("blend", ["opaque", "both"])
def test_small_draws_of_few_states(gpu_ctx, blend):
    """Hundreds of draws of a few pixels under pipelines that differ in blend state, two of them equal: the fragments of one
    shading pass are of many draws and few states.  Every other draw has a viewport of its own."""
    s = S.soup(4, 96, 64, seed=2, size_px=np.log(6.0))
    s.draws = [S.soup(4, 96, 64, seed=10 + k, size_px=np.log(6.0)).draws[0] for k in range(400)]
    for k, d in enumerate(s.draws[::2]):
        d.viewport = (float(k % 3), float(k % 5), 96.0 - k % 7, 64.0 - k % 4, 0.0, 1.0)
    plain = dict(s.pipeline, blend=None)
    s.pipelines = [plain, dict(plain), dict(plain, depth_write=0)] if blend == "opaque" else \
        [plain, dict(plain), dict(plain, blend=W.ALPHA_BLEND), dict(plain, blend=W.ALPHA_BLEND, depth_write=0)]
    s.draw_pipeline = [k % len(s.pipelines) for k in range(len(s.draws))]
    ref = oracle_lib.render_scene(s)
    print(f"[groups] {blend}", flush=True)
    compare(s, render_gpu(gpu_ctx, s), ref, "counting")
    compare(s, render_gpu(gpu_ctx, s, count=False), (ref[0], ref[1], None), "culling on")
