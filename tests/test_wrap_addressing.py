"""REPEAT addressing of a bilinear fetch: `wrap_pair` in csrc/image_ops.hpp takes the two
texels i and i + 1 of an axis of n texels by an addition and a compare where i lies within
one image of the origin, and by the general remainder elsewhere.  The header's own
functions, built for the host, are checked against the remainder for every form: images of
one texel, both sides of each border, the ends of the 32-bit range."""
import ctypes as C
import subprocess

import numpy as np
import pytest

from vulkanpbrt_amd import build

SOURCE = r"""
#include "image_ops.hpp"
extern "C" void wrap_pairs(const int* i, long count, int n, int* out) {
    for (long k = 0; k < count; ++k) pbrt::wrap_pair(i[k], n, out[2 * k], out[2 * k + 1]);
}
extern "C" void wrap_coords(const int* i, long count, int n, int* out) {
    for (long k = 0; k < count; ++k) out[k] = pbrt::wrap_coord(i[k], n);
}
"""


@pytest.fixture(scope="module")
def wrap(tmp_path_factory):
    d = tmp_path_factory.mktemp("wrap")
    (d / "wrap.cpp").write_text(SOURCE)
    subprocess.run([build.HIPCC, "-x", "hip", "--offload-host-only", "-O2", "-fPIC", "-shared", "-std=c++17", "-I",
                    str(build.CSRC), str(d / "wrap.cpp"), "-o", str(d / "wrap.so")], check=True)
    return C.CDLL(str(d / "wrap.so"))


def run(function, i, n, width):
    i = np.ascontiguousarray(i, np.int32)
    out = np.full((len(i), width), -1, np.int32)
    function(i.ctypes.data_as(C.c_void_p), C.c_long(len(i)), C.c_int(n), out.ctypes.data_as(C.c_void_p))
    return out


@pytest.mark.parametrize("n", [1, 2, 3, 16, 1279, 1920, 65535])
def test_wrap_pair_equals_the_remainder(wrap, n):
    near = set(range(-3, 4)) | {k * n + d for k in range(-3, 4) for d in range(-3, 4)}
    far = {-2 ** 31, -2 ** 31 + 1, -2 ** 31 + n, 2 ** 31 - 2, 2 ** 31 - 1 - n, 2 ** 31 - 1 - 2 * n}
    i = np.array(sorted(near | far | set(range(-min(n, 70), min(n, 70)))), np.int64)
    expect = np.stack([i % n, (i + 1) % n], -1)
    assert np.array_equal(run(wrap.wrap_pairs, i, n, 2), expect)
    assert np.array_equal(run(wrap.wrap_coords, i, n, 1)[:, 0], i % n)
