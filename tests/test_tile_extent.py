"""The tile copies' resource sizes (csrc/tile_extent.h, plain arithmetic that the kernels and this test compile alike): every
tile's size is its rows times the row stride, for a K of 2 GiB and more and for the largest row stride that a launch can have,
and tiles past the range have none."""
import ctypes
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "amdgpu_rustdsl_amd", "csrc")
SOURCE = r"""
#include "tile_extent.h"
extern "C" unsigned extent(unsigned end, unsigned key, unsigned stride) { return tile_extent((int32_t)(end - key), stride); }
template <int LAG>
void walk(unsigned end, unsigned kkey, unsigned stride, int n, unsigned* sizes) {
    TileSizes<LAG> t;
    t.init(end, kkey, stride);
    for (int i = 0; i < n; ++i, t.advance(stride)) {
        sizes[2 * i] = t.k;
        sizes[2 * i + 1] = t.v;
    }
}
// sizes[2 i], [2 i + 1]: the K tile at kkey + 128 i and the V tile `lag` tiles behind it
extern "C" void sequence(unsigned end, unsigned kkey, unsigned stride, int lag, int n, unsigned* sizes) {
    (lag ? walk<1> : walk<0>)(end, kkey, stride, n, sizes);
}
"""


@pytest.fixture(scope="module")
def native(tmp_path_factory):
    d = tmp_path_factory.mktemp("tile_extent")
    src, so = d / "t.cpp", d / "t.so"
    src.write_text(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-I" + CSRC, str(src), "-o", str(so)], check=True)
    return ctypes.CDLL(str(so))


def _want(end, key, stride):
    return min(max(end - key, 0), 128) * stride


# (KV heads, keys): ordinary; a K of 2 GiB and a bit, by heads and by keys; strides whose multiples of 384 rows pass 2^31
SIZES = [(1, 1), (8, 2048), (8, 1337), (128, 131200), (8, 2097200), (1, 16777300), (43691, 129), (65535, 257), (65536, 64)]


@pytest.mark.parametrize("HK,SK", SIZES)
def test_tile_extents(native, HK, SK):
    stride = HK * 128
    tiles = (SK + 127) // 128
    some = sorted({t for t in (0, 1, 2, 3, tiles // 2, tiles - 1, tiles, tiles + 1, tiles + 2, tiles + 3) if t >= 0})
    for t in some:
        want = _want(SK, 128 * t, stride)
        assert want < 1 << 31
        assert native.extent(SK, 128 * t, stride) == want
        assert native.extent(SK, 128 * t, stride // 32) == want // 32   # the K scales' rows
    first = max(0, tiles - 6)   # the loop's copies start three tiles in, and run three tiles past the end
    n = tiles - first + 3
    for lag in (0, 1):
        got = (ctypes.c_uint * (2 * n))()
        native.sequence(SK, 128 * (first + 3), stride, lag, n, got)
        for i in range(n):
            key = 128 * (first + 3 + i)
            assert got[2 * i] == _want(SK, key, stride) and got[2 * i + 1] == _want(SK, key - 128 * lag, stride), (lag, i)
