"""The pixel box of a line's quad (bin_kernels.h, line_box), checked by brute
force in float32 on the CPU: every pixel whose four rounded edge values are
>= 0 (ProcessLines, CPVulkan/CommandBuffer.Draw.cpp:1420-1497) lies in the
box, for quads from full width down to a thousandth of a pixel, and quads
that the bound does not cover get none."""
import numpy as np
import pytest

f32 = np.float32


def quad(p0, p1, width, W, H):
    """Corners p00, p01, p10, p11 as setup_line computes them (float32)."""
    v = (p1 - p0).astype(f32)
    inv = f32(1.0) / np.sqrt(((v[0] * v[0] + v[1] * v[1]) + v[2] * v[2]) + v[3] * v[3])
    px, py = v[1] * inv, -(v[0] * inv)
    lx, ly = f32(width) / f32(W), f32(width) / f32(H)
    out = []
    for p in (p0, p1):
        out += [(p[0] + px * lx, p[1] + py * ly), (p[0] - px * lx, p[1] - py * ly)]
    return [np.array(c, f32) for c in out]


def line_box(c, W, H):
    """Restatement of line_box: (x0, y0, x1, y1) clipped to the viewport, or None."""
    if any(not abs(x) <= 4.0 for p in c for x in p):
        return None
    s = np.array([0.5 * W, 0.5 * H])
    q = [p.astype(np.float64) for p in (c[0], c[1], c[3], c[2])]
    for k in range(4):
        u, v = (q[(k + 1) % 4] - q[k]) * s, (q[(k + 2) % 4] - q[(k + 1) % 4]) * s
        e = v[0] * u[1] - v[1] * u[0]
        if not (u @ u >= 2.0 ** -20 and e > 0 and e * e >= 0.01 * (u @ u) * (v @ v)):
            return None
    px = np.array([(p + 1.0) * s for p in q])
    lo, hi = np.floor(px.min(0)).astype(int) - 4, np.floor(px.max(0)).astype(int) + 5
    return max(lo[0], 0), max(lo[1], 0), min(hi[0], W), min(hi[1], H)


def covered(c, W, H):
    x = ((np.arange(W, dtype=f32) / f32(W) + f32(f32(1) / f32(W)) * f32(0.5)) * f32(2) - f32(1))[None, :]
    y = ((np.arange(H, dtype=f32) / f32(H) + f32(f32(1) / f32(H)) * f32(0.5)) * f32(2) - f32(1))[:, None]
    m = np.ones((H, W), bool)
    for a, b in ((0, 1), (3, 2), (2, 0), (1, 3)):
        e = (x - c[a][0]) * (c[b][1] - c[a][1]) - (y - c[a][1]) * (c[b][0] - c[a][0])
        m &= e >= 0
    return m


@pytest.mark.parametrize("W,H", [(160, 90), (64, 512), (333, 41)])
def test_box_holds_every_covered_pixel(W, H):
    rng = np.random.default_rng(7)
    boxed = pixels = thin = 0
    for k in range(400):
        a = rng.uniform(-1.3, 1.3, 2)
        length = np.exp(rng.normal(np.log(20.0), 1.0))
        t = rng.uniform(0, 2 * np.pi) if k % 4 else rng.integers(0, 4) * np.pi / 2
        b = a + length * np.array([np.cos(t) * 2 / W, np.sin(t) * 2 / H])
        spread = 10.0 ** rng.uniform(-3, 4)   # z and w differences: the wider, the thinner the quad
        p0 = np.array([a[0], a[1], 0.0, 1.0], f32)
        p1 = np.array([b[0], b[1], rng.uniform(0, 1) * spread, 1.0 + spread], f32)
        c = quad(p0, p1, rng.choice([0.5, 1.0, 3.0, 8.0]), W, H)
        box = line_box(c, W, H)
        if box is None:
            continue
        boxed += 1
        thin += np.hypot(*((c[0] - c[1]) * (W / 2, H / 2))) < 0.5
        m = covered(c, W, H)
        pixels += int(m.sum())
        x0, y0, x1, y1 = box
        m[y0:max(y1, y0), x0:max(x1, x0)] = False
        assert not m.any(), f"line {k}: pixels outside {box}"
    assert boxed > 300 and thin > 100 and pixels > 1000


def test_degenerate_quads_have_no_box():
    W, H = 160, 90
    p = np.array([0.1, 0.2, 0.0, 1.0], f32)
    q = np.array([0.4, -0.3, 0.0, 1.0], f32)
    assert line_box(quad(p, q, 2.0, W, H), W, H) is not None
    with np.errstate(all="ignore"):
        for a, b, w in ((p, p, 1.0), (p, q, 0.0), (p, q * f32(1e30), 1.0), (p, q, -1.0), (p * f32(np.nan), q, 1.0)):
            assert line_box(quad(a, b, w, W, H), W, H) is None
