"""Which form the planner gives a contraction (host only,
tests/native/route_check.cpp).

* Small contractions in scrambled orders run as one launch without workspace, in
  every precision mode, whatever kernel the table names for their shape.
* The in-place form for a few k and columns is for problems with enough rows or
  work per batch value, and large enough to hide its chain of sums.
* The two-launch form for few outputs leaves small problems to the fused pass,
  and in the operands' own order to the table; all of them sum in FP64.
"""
import ctypes
import math
import os
import random
import subprocess

import numpy as np
import pytest

from jet_amd import _native as nat
from jet_amd import build as jb

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PRODUCT, FUSED, SHORT_K, FEW_OUTPUTS = 0, 1, 2, 3
SPLIT_KERNELS = (4, 5, 7)


@pytest.fixture(scope="module")
def lib():
    jb.write_tuning_table()
    out = os.path.join(ROOT, "tests", "native", "_build", f"libroute_check.{os.getpid()}.so")
    os.makedirs(os.path.dirname(out), exist_ok=True)
    csrc = os.path.join(ROOT, "jet_amd", "csrc")
    subprocess.run(["g++", "-std=c++17", "-O2", "-fPIC", "-shared",
                    "-I" + os.path.join(ROOT, "include"), "-I" + jb.BUILD, "-o", out,
                    os.path.join(ROOT, "tests", "native", "route_check.cpp")] +
                   [os.path.join(csrc, f) for f in ("contract_plan.cpp", "permute_plan.cpp",
                                                    "tuning.cpp")], check=True)
    L = ctypes.CDLL(out)
    os.remove(out)
    return L


def route(lib, mode, a, b, c, ext=2):
    """Every mode of extent `ext`."""
    e = lambda ms: nat.i64([ext] * len(ms))
    out = (ctypes.c_int64 * 5)()
    assert lib.contraction_route(mode, len(a), nat.i32(a), e(a), len(b), nat.i32(b), e(b), len(c),
                                 nat.i32(c), out) == 0
    return dict(zip(("form", "kernel", "launches", "slices", "workspace"), out))


def modes(batch, m, n, k, rng=None):
    """Modes of A, B and C, in the order of a batched product or (rng) scrambled."""
    bb, mm = list(range(batch)), list(range(100, 100 + m))
    nn, kk = list(range(200, 200 + n)), list(range(300, 300 + k))
    a, b = bb + mm + kk, bb + nn + kk
    if rng is None:
        return a, b, bb + mm + nn
    rng.shuffle(a)
    rng.shuffle(b)
    c = [x for x in a if x < 200] + [x for x in b if 200 <= x < 300]
    return a, b, c


@pytest.mark.parametrize("mode", [0, 2, 3, 4])
def test_small_scrambled_contractions_are_one_launch(lib, mode):
    rng = random.Random(mode)
    named = [(0, 0, 0, 3), (0, 3, 3, 3), (0, 2, 6, 3), (0, 6, 6, 6), (0, 4, 4, 8), (0, 8, 8, 6)]
    drawn = [(rng.choice([0, 0, 2, 4]), rng.randint(0, 9), rng.randint(0, 9), rng.randint(0, 11))
             for _ in range(400)]
    for batch, m, n, k in named + [d for d in drawn if sum(d) <= 22]:
        r = route(lib, mode, *modes(batch, m, n, k, rng))
        if r["kernel"] not in SPLIT_KERNELS:
            assert r["launches"] == 1 and r["workspace"] == 0, ((batch, m, n, k), r)


def test_larger_scrambled_contractions_are_products(lib):
    """From 2^23 multiply-adds the matrix cores earn their copies."""
    rng = random.Random(1)
    for mode in (0, 2):
        for shape in ((0, 9, 9, 5), (0, 8, 8, 8), (0, 8, 9, 8), (2, 8, 7, 8)):
            assert route(lib, mode, *modes(*shape, rng))["form"] == PRODUCT, (mode, shape)


@pytest.mark.parametrize("mode", [0, 2])
@pytest.mark.parametrize("shape", [
    (15, 1, 4, 2), (15, 3, 1, 1), (15, 3, 2, 2), (8, 2, 3, 4), (14, 2, 2, 2), (15, 4, 0, 2),
    (12, 2, 2, 2)])
def test_few_rows_a_batch(lib, mode, shape):
    """Many batches of few rows and little work each: the table's kernel, which
    fills whole work-groups across batches."""
    r = route(lib, mode, *modes(*shape))
    assert r["form"] == PRODUCT and r["launches"] == 1, r
    # the same with the larger operand second
    a, b, c = modes(shape[0], shape[2], shape[1], shape[3])
    assert route(lib, mode, a, b, c)["form"] == PRODUCT


def test_short_k_where_it_pays(lib):
    rng = random.Random(2)
    for mode in (0, 2):
        # gates on states, and batches of enough rows
        for shape in ((0, 14, 2, 2), (0, 20, 1, 1), (0, 24, 2, 2), (0, 20, 4, 4)):
            assert route(lib, mode, *modes(*shape))["form"] == \
                (SHORT_K if sum(shape) > 20 else PRODUCT), (mode, shape)
        assert route(lib, mode, *modes(6, 12, 2, 2))["form"] == SHORT_K
        # small scrambled ones with many k and columns go to the fused pass
        a, b, c = modes(0, 12, 4, 4)
        assert route(lib, mode, a[::-1], b, c)["form"] == FUSED
        # table kernels in the operands' own order
        assert route(lib, mode, *modes(0, 12, 4, 4))["form"] == PRODUCT
    assert route(lib, 0, *modes(15, 4, 3, 4))["form"] == SHORT_K   # 2^15 of 16 x 8 x 16
    assert route(lib, 2, *modes(0, 15, 4, 4))["form"] == PRODUCT   # matrix cores
    assert route(lib, 2, *modes(0, 18, 4, 4))["form"] == SHORT_K


@pytest.mark.parametrize("mode", [0, 2])
def test_few_outputs(lib, mode):
    rng = random.Random(3)
    for shape in ((0, 4, 2, 12), (1, 3, 1, 12), (4, 2, 2, 12), (6, 1, 1, 12)):
        assert route(lib, mode, *modes(*shape, rng))["form"] == FUSED, shape
    for shape in ((0, 4, 2, 14), (0, 1, 1, 20), (0, 2, 1, 22), (6, 3, 3, 12)):
        assert route(lib, mode, *modes(*shape, rng))["form"] == FEW_OUTPUTS, shape
    for shape in ((0, 4, 2, 12), (2, 2, 2, 13), (0, 4, 2, 16), (0, 3, 1, 18), (4, 3, 1, 12)):
        r = route(lib, mode, *modes(*shape))
        assert r["form"] == PRODUCT and r["kernel"] in (1, 6), (shape, r)
    for shape in ((0, 2, 1, 22), (0, 4, 2, 20), (4, 3, 3, 15)):
        assert route(lib, mode, *modes(*shape))["form"] == FEW_OUTPUTS, shape


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k,batch", [
    (16, 4, 4096, 1), (4, 4, 8192, 4), (2, 2, 4096, 16), (7, 5, 1000, 3), (1, 1, 300, 1),
    (3, 2, 257, 2)])
def test_reductions_sum_in_fp64(m, n, k, batch):
    """In the operands' own order: one rounding to complex64 for each output."""
    from hiputil import contract, rand_c, say
    rng = np.random.default_rng(m * n + k)
    row = (ctypes.c_int32 * 7)(0, *[round(math.log2(x)) for x in (m, n, k, batch)], 1, 1)
    a, b = rand_c(rng, batch * m * k, np.complex64), rand_c(rng, batch * n * k, np.complex64)
    say(f"reduction {m}x{n}x{k} batch {batch}")
    try:
        nat.check(nat.lib().jet_hip_tuning_set(1, row))
        got, info = contract(nat.default_context(), a, [0, 1, 3], [batch, m, k], b, [0, 2, 3],
                             [batch, n, k], [0, 1, 2])
    finally:
        nat.check(nat.lib().jet_hip_tuning_set(-1, None))
    assert info["kernel"] == "valu_reduce"
    want = np.einsum("bmk,bnk->bmn", a.reshape(batch, m, k).astype(np.complex128),
                     b.reshape(batch, n, k).astype(np.complex128)).reshape(-1)
    err = np.abs(got - want)
    assert np.all(err <= 2.0 ** -23 * np.maximum(np.abs(want.real), np.abs(want.imag)))


@pytest.mark.parametrize("m,n,k,kernel", [
    (32, 32, 4096, 1), (32, 64, 2048, 1), (64, 32, 2048, 1),         # reductions
    (64, 64, 4096, 2), (128, 128, 4096, 2), (48, 48, 8192, 2)])      # slices of products
def test_long_k_with_few_outputs(lib, m, n, k, kernel):
    """Matrix-core slices in place of a reduction where they are faster with their sum."""
    i64 = lambda *v: (ctypes.c_int64 * len(v))(*v)
    out = (ctypes.c_int64 * 5)()
    assert lib.contraction_route(0, 2, nat.i32([0, 2]), i64(m, k), 2, nat.i32([1, 2]), i64(n, k),
                                 2, nat.i32([0, 1]), out) == 0
    assert out[0] == PRODUCT and out[1] == kernel, list(out)


@pytest.mark.parametrize("fp64,aligned,threads", [(0, 1, 256), (0, 0, 256), (1, 1, 512)])
@pytest.mark.parametrize("m", [1, 16, 32, 40])
def test_tiles_fit_a_launch(lib, fp64, aligned, threads, m):
    """Long thin products: 2^32 threads is what a launch takes."""
    lib.product_tiles.restype = ctypes.c_int64
    lib.product_tiles.argtypes = [ctypes.c_int] * 2 + [ctypes.c_int64] * 3
    for log2n in (20, 24, 28, 29):
        for a, b in ((m, 1 << log2n), (1 << log2n, m)):
            assert lib.product_tiles(fp64, aligned, a, b, 16) * threads < 2 ** 32, log2n
