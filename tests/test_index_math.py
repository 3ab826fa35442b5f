"""Index arithmetic of the kernels (csrc/index_math.h), compiled for the host, at the ends of its ranges."""
import ctypes as C
import subprocess
from pathlib import Path

import numpy as np
import pytest

CSRC = Path(__file__).resolve().parent.parent / "cpvulkan_amd" / "csrc"

SOURCE = """
#include "index_math.h"
extern "C" void segment(unsigned n, unsigned seg, unsigned* be) { cpv::segment_range(n, seg, be[0], be[1]); }
extern "C" int plain(unsigned w, unsigned h) { return cpv::plain_extent(w, h); }
extern "C" int wrap(int v, int size, int mode) { return cpv::wrap_coord(v, size, mode); }
extern "C" unsigned items(unsigned t0, unsigned e) { return cpv::tile_items(t0, e); }
"""


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    d = tmp_path_factory.mktemp("index_math")
    (d / "m.cpp").write_text(SOURCE)
    subprocess.run(["g++", "-O1", "-fwrapv", "-std=c++17", "-shared", "-fPIC", f"-I{CSRC}", "-o", str(d / "m.so"), str(d / "m.cpp")], check=True)
    return C.CDLL(str(d / "m.so"))


@pytest.mark.parametrize("n", [0, 1, 63, 64, 65, 1023, 1024, 65535, 65536, 65537, 2**20, 2**31, 2**32 - 65537, 2**32 - 65536, 2**32 - 65535,
                               2**32 - 4096, 2**32 - 1024, 2**32 - 1023, 2**32 - 2, 2**32 - 1])
def test_sort_segments_cover_every_pair(lib, n):
    """The segments follow each other from 0 to n, and a workgroup's walk takes every item of its own and ends."""
    be, at = (C.c_uint32 * 2)(), 0
    for seg in range(1024):
        lib.segment(C.c_uint32(n), C.c_uint32(seg), be)
        b, e = be
        assert b == at and e >= b, (n, seg, b, e)
        at = e
    assert at == n
    # the last segment that holds anything (the one nearest to 2^32), from two tiles before its end
    t0, e = max(n - 5000, 0), n
    steps = 0
    while t0 < e:
        k = int(np.uint32(lib.items(C.c_uint32(t0), C.c_uint32(e))))
        assert 1 <= k <= 2048 and (k == 2048 or t0 + k == e)
        t0 = (t0 + k) & 0xFFFFFFFF   # the kernels' 32-bit sum
        steps += 1
        assert steps <= 3
    assert t0 == e


@pytest.mark.parametrize("mode", [0, 1, 2, 4])   # every address mode but CLAMP_TO_BORDER
@pytest.mark.parametrize("size", [1, 2, 3, 5, 64, 1000, 16384, 2**29 - 1, 2**29, 2**29 + 1, 3 * 2**28, 2**30 - 1, 2**30])
def test_texels_read_without_a_bounds_test_are_inside(lib, mode, size):
    """Wherever the sampler leaves out the bounds test, the wrapped coordinate is a texel of the level."""
    if not lib.plain(C.c_uint32(size), C.c_uint32(1)):
        assert size > 16384   # no image that Vulkan's limits allow takes the slow path
        return
    rng = np.random.default_rng(size % 1000)
    at = np.concatenate([np.arange(-5, 6), size * np.arange(-3, 4), size * np.arange(-3, 4) - 1, [-2**31, -2**31 + 1, 2**31 - 2, 2**31 - 1],
                         rng.integers(-2**31, 2**31, 3000)])
    for v in np.unique(at[(at >= -2**31) & (at < 2**31)]).tolist():
        assert 0 <= lib.wrap(v, size, mode) < size, (v, size, mode)


def test_plain_extents(lib):
    for w, h, ok in [(0, 0, 0), (0, 7, 0), (7, 0, 0), (1, 1, 1), (16384, 16384, 1), (32768, 32768, 1), (32769, 32768, 0), (2**29, 2, 1),
                     (2**29 + 1, 1, 0), (1, 2**30, 0), (2**32 - 1, 2**32 - 1, 0)]:
        assert lib.plain(C.c_uint32(w), C.c_uint32(h)) == ok, (w, h)


LONG = """
#include "index_math.h"
extern "C" int splits(unsigned from, unsigned filled, unsigned pairs, unsigned n, unsigned waves)
{ return cpv::splits_tile(cpv::LongTiles{0, from, filled, pairs}, n, waves); }
"""


def test_which_tiles_are_split(tmp_path):
    """Lists much alike are split only while their tiles leave the chip idle; lists far beyond the mean always."""
    (tmp_path / "l.cpp").write_text(LONG)
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", f"-I{CSRC}", "-o", str(tmp_path / "l.so"), str(tmp_path / "l.cpp")],
                   check=True)
    splits = C.CDLL(str(tmp_path / "l.so")).splits
    u = C.c_uint32
    for waves in (1, 2, 4):
        for filled, alike in ((1, 1), (300, 1), (1535 // waves, 1), (1536 // waves, 0), (8160, 0), (1 << 22, 0)):
            n = 500
            pairs = n * filled
            at = max(256, pairs // 8192)
            assert splits(u(at), u(filled), u(pairs), u(max(n, at)), u(waves)) == (alike or at >= 2 * n), (waves, filled)
            assert not splits(u(at), u(filled), u(pairs), u(at - 1), u(waves))
        # one tile in ten holds nine tenths of the pairs
        assert splits(u(256), u(10_000), u(1_000_000), u(900), u(waves)) and not splits(u(256), u(10_000), u(9_000_000), u(900), u(waves))
    assert splits(u(2**20), u(2**22), u(2**32 - 1), u(2**32 - 1), u(1))   # the products are taken in 64 bits
