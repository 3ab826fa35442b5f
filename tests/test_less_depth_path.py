"""The raster kernel's arithmetic for depth tests LESS and LESS_OR_EQUAL
(raster_tile.h), restated in float32: divide_exact equals the rounded
quotient, and depth_surely_not_less's bound never exceeds the depth that the
reference's operations give."""
from fractions import Fraction

import numpy as np
import pytest

f32, wide = np.float32, np.longdouble


def fma(a, b, c):
    """Rounded once: the product of two 24-bit significands and the sum are taken in 64 bits, which holds the
    residuals of divide_exact exactly."""
    return (a.astype(wide) * b.astype(wide) + c.astype(wide)).astype(f32)


def divide_exact(e, area):
    rinv = f32(1.0) / area
    q = e * rinv
    q = fma(fma(-area, q, e), rinv, q)
    return fma(fma(-area, q, e), rinv, q)


def _operands(kind, rng, n):
    if kind == "random":
        m = lambda: rng.integers(1 << 23, 1 << 24, n).astype(np.float64)  # noqa: E731
    else:   # significands at the ends of a binade, and quotients next to a midpoint
        ends = np.concatenate([np.arange(1 << 23, (1 << 23) + 40), np.arange((1 << 24) - 40, 1 << 24)])
        m = lambda: rng.choice(ends, n).astype(np.float64)  # noqa: E731
    e = np.ldexp(m(), rng.integers(-60 - 23, 43 - 23, n)).astype(f32)
    area = np.ldexp(m(), rng.integers(-60 - 23, 60 - 23, n)).astype(f32)
    if kind == "midpoint":
        q = rng.integers(1 << 23, 1 << 24, n) * 2 + 1                       # q + 1/2 in units of the quotient's last place
        e = np.ldexp((q * (area.astype(np.float64) / 2.0)), rng.integers(-20, -10, n)).astype(f32)
    ok = (e >= 2.0 ** -60) & (e <= 2.0 ** 43)
    return e[ok], area[ok]


@pytest.mark.parametrize("kind", ["random", "ends", "midpoint"])
def test_divide_exact_is_the_rounded_quotient(kind):
    e, area = _operands(kind, np.random.default_rng(11), 400_000)
    assert e.size > 100_000
    got, want = divide_exact(e, area), e / area
    for i in np.nonzero(got != want)[0]:   # the 64-bit sum of the last step may itself round to a tie: settle it exactly
        r = f32(1.0) / area[i]
        q = e[i] * r
        for _ in range(2):
            res = Fraction(float(e[i])) - Fraction(float(area[i])) * Fraction(float(q))
            x = Fraction(float(f32(float(res)))) * Fraction(float(r)) + Fraction(float(q))
            near = [f32(q), np.nextafter(q, f32(np.inf), dtype=f32), np.nextafter(q, f32(-np.inf), dtype=f32)]
            q = min(near, key=lambda v: abs(Fraction(float(v)) - x))
        assert q == want[i]


@pytest.mark.parametrize("extent", [64, 1920, 16384])
def test_depth_bound_is_below_the_depth(extent):
    rng = np.random.default_rng(extent)
    tight = 0
    for k in range(300):
        P = rng.uniform(-1.2, 1.2, (3, 2)) if k % 3 else rng.uniform(-1, 1, 2) + rng.normal(0, 20.0 / extent, (3, 2))
        if k % 5 == 0:
            P[2] = P[0] + (P[1] - P[0]) * rng.uniform(0, 1) + rng.normal(0, 1e-5, 2)   # slivers
        P = P.astype(f32)
        z = (rng.uniform(0, 1, 3) * (0.0 if k % 7 == 0 else 10.0 ** rng.integers(-30, 6))).astype(f32)
        area = (P[2, 0] - P[0, 0]) * (P[1, 1] - P[0, 1]) - (P[2, 1] - P[0, 1]) * (P[1, 0] - P[0, 0])
        s = [(1, 2), (2, 0), (0, 1)] if area >= 0 else [(2, 1), (0, 2), (1, 0)]
        area = abs(area)
        if not area >= 2.0 ** -60:
            continue
        w = rng.dirichlet((1, 1, 1), 400)
        c = (w @ P.astype(np.float64)).astype(f32)   # points inside: the pixel centres may lie anywhere
        e = [(c[:, 0] - P[a, 0]) * (P[b, 1] - P[a, 1]) - (c[:, 1] - P[a, 1]) * (P[b, 0] - P[a, 0]) for a, b in s]
        keep = (e[0] >= 0) & (e[1] >= 0) & (e[2] >= 0)
        e = [x[keep] for x in e]
        depth = (z[0] * (e[0] / area) + z[1] * (e[1] / area)) + z[2] * (e[2] / area)
        rinv = f32(1.0) / area
        q = [x * rinv for x in e]
        da = fma(np.full_like(q[2], z[2]), q[2], fma(np.full_like(q[1], z[1]), q[1], z[0] * q[0]))
        lo = fma(da, np.full_like(da, f32(1.0 - 2.0 ** -19)), np.full_like(da, f32(-2.0 ** -120)))
        assert (lo <= depth).all()
        tight += int((lo > depth * f32(1.0 - 2.0 ** -17)).sum())
    assert tight > 10_000
