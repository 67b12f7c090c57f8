"""Generic permutations by tiles: plans replayed on the CPU
(tests/native/tiles_check.cpp) against numpy's transpose, and the kernel on the
GPU, exactly."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

from hiputil import permute, say
from jet_amd import _native as nat

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

# (extents, output order): matrices with and without a divisor to split at, odd
# extents, a trailing axis that stays, an axis between, long and short axes, many axes.
SHAPES = [
    ([1260, 1014], [1, 0]), ([1009, 997], [1, 0]), ([5, 7, 6, 6, 1014], [4, 0, 1, 2, 3]),
    ([300, 7, 500], [2, 1, 0]), ([36, 35, 30, 10], [3, 2, 1, 0]), ([60, 50, 9, 7], [1, 0, 2, 3]),
    ([9, 11, 13, 8, 12, 5], [5, 2, 0, 4, 1, 3]), ([3] * 11, [10, 3, 7, 0, 9, 1, 5, 2, 8, 4, 6]),
    ([3] * 12, [11, 0, 10, 1, 9, 2, 8, 3, 7, 4, 6, 5]), ([2, 3] * 7, [13, 11, 9, 7, 5, 3, 1, 12, 10, 8, 6, 4, 2, 0]),
    ([2, 3] * 6, [11, 9, 7, 5, 3, 1, 10, 8, 6, 4, 2, 0]),
    ([4096, 33], [1, 0]), ([33, 4096], [1, 0]), ([131, 1024], [1, 0]), ([2, 70001], [1, 0]),
    ([5, 30000, 3], [2, 1, 0]), ([64, 65, 66], [2, 0, 1]), ([128, 127, 9], [1, 0, 2])]


@pytest.fixture(scope="module")
def lib():
    out = os.path.join(ROOT, "tests", "native", "_build", f"libtiles_check.{os.getpid()}.so")
    os.makedirs(os.path.dirname(out), exist_ok=True)
    subprocess.run(["g++", "-std=c++17", "-O2", "-fPIC", "-shared",
                    "-I" + os.path.join(ROOT, "include"), "-o", out,
                    os.path.join(ROOT, "tests", "native", "tiles_check.cpp"),
                    os.path.join(ROOT, "jet_amd", "csrc", "permute_plan.cpp")], check=True)
    L = ctypes.CDLL(out)
    os.remove(out)
    return L


@pytest.mark.parametrize("elem", [8, 16])
@pytest.mark.parametrize("shape,perm", SHAPES)
def test_plan(lib, elem, shape, perm):
    n = int(np.prod(shape))
    out = np.empty(n, np.int64)
    rc = lib.tiled_permutation(elem, len(shape), nat.i64(shape), nat.i32(perm),
                               out.ctypes.data_as(ctypes.POINTER(ctypes.c_int64)))
    assert rc >= 0, rc
    if rc == 0:   # small, or no divisor gives runs on both sides, or a long run that stays
        assert n < 1 << 17 or shape in ([1009, 997], [131, 1024], [2, 70001], [5, 30000, 3],
                                        [128, 127, 9], [60, 50, 9, 7])
        return
    want = np.arange(n).reshape(shape).transpose(perm).reshape(-1)
    assert np.array_equal(out, want)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [np.complex64, np.complex128])
@pytest.mark.parametrize("shape,perm", SHAPES)
def test_gpu(dtype, shape, perm):
    ctx = nat.default_context()
    n = int(np.prod(shape))
    x = (np.arange(n) + 1j * np.arange(n)[::-1]).astype(dtype)
    say(f"tiled permutation {shape} -> {perm} {np.dtype(dtype).name}")
    got = permute(ctx, x, shape, list(range(len(shape))), perm)
    assert np.array_equal(got, x.reshape(shape).transpose(perm).reshape(-1))
