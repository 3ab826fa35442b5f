"""The device's UNORM conversions (raster_device.h, unormN_to_float,
round_to_u32) restated and compared with the operations they replace: u / max
in float32 for every code, and roundf (half away from zero) for every float
near a half."""
import math

import numpy as np
import pytest

f32, wide = np.float32, np.longdouble


@pytest.mark.parametrize("bits,head,tail", [(8, "0x1.01p-8", "0x1.010102p-24"), (16, "0x1p-16", "0x1.0001p-32"),
                                            (24, "0x1p-24", "0x1.000002p-48")])
def test_unorm_to_float_is_the_rounded_quotient(bits, head, tail):
    head, tail = float.fromhex(head), float.fromhex(tail)
    assert float(f32(head)) == head and float(f32(tail)) == tail
    u = np.arange(1 << bits, dtype=np.int64)
    p = u.astype(f32) * f32(head)
    assert np.array_equal(p.astype(np.float64), u.astype(np.float64) * head)      # the product is exact
    # the fma: tail * u has at most 48 bits and the sum fits the 64 of a long double
    v = (u.astype(wide) * wide(tail) + p.astype(wide)).astype(f32)
    assert np.finfo(wide).nmant >= 63
    assert np.array_equal(v, u.astype(f32) / f32((1 << bits) - 1))


def test_round_to_u32_is_roundf():
    half = f32(float.fromhex("0x1.fffffep-2"))   # the float below 0.5
    n = np.unique(np.concatenate([np.arange(0, 70000), 2 ** np.arange(1, 24), 2 ** np.arange(1, 24) - 1,
                                  np.random.default_rng(3).integers(0, 1 << 24, 200_000)]))
    for at in (n.astype(f32), (n + 0.5).astype(f32), np.linspace(0, 1, 100_001).astype(f32)):
        for step in range(-3, 4):
            x = at.copy()
            for _ in range(abs(step)):
                x = np.nextafter(x, f32(math.inf if step > 0 else -math.inf), dtype=f32)
            x = x[(x >= 0) & (x <= 2.0 ** 24)]
            want = np.floor(x.astype(np.float64) + 0.5)   # half away from zero, exact in double
            assert np.array_equal((x + half).astype(np.uint32), want.astype(np.uint32))


@pytest.mark.parametrize("size", [1, 2, 64, 1024, 3, 7, 500])
def test_repeat_wrap(size):
    v = np.concatenate([np.arange(-3 * size - 2, 3 * size + 2), [-2**31, -2**31 + 1, 2**31 - 1]]).astype(np.int64)
    m = np.fmod(v, size)                          # C's remainder, the sign of v
    want = np.fmod(m + size, size)
    got = (v & (size - 1)) if size & (size - 1) == 0 else np.where(m < 0, m + size, m)
    assert np.array_equal(got, want)


@pytest.mark.parametrize("bits", [21, 13, 1])
def test_first_lerp_of_a_bilinear_sample_in_single_precision(bits):
    """lerp of UNORM8 values by a multiple of 2^-21: the double form is exact before its rounding, as the fma's sum is."""
    rng = np.random.default_rng(bits)
    a, b = (rng.integers(0, 256, 400_000).astype(f32) / f32(255) for _ in range(2))
    t = (rng.integers(0, 1 << bits, a.size) / float(1 << bits)).astype(f32)
    t[:1000] = f32(1.0) - f32(2.0 ** -bits)
    d = b - a
    ref = (a.astype(np.float64) + d.astype(np.float64) * t.astype(np.float64)).astype(f32)
    assert np.array_equal(ref, (a.astype(wide) + d.astype(wide) * t.astype(wide)).astype(f32))
    assert ((a.astype(wide) + d.astype(wide) * t.astype(wide)) == (a.astype(np.float64) + d.astype(np.float64) * t.astype(np.float64))).all()
