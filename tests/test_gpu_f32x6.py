"""The FP32 GEMM on the BF16 matrix cores (three pieces of each value, six
products) against numpy in 64 bits, through contraction plans whose table
entry names the FP32 matrix-core kernel.

Tolerance: every partial sum is rounded at most 12 times per 16 k (relative
2^-24 each, independent), so the normwise error stays under
2^-24 (sqrt(K) + 8).
"""
import ctypes
import math

import numpy as np
import pytest

from hiputil import contract, rand_c, say
from jet_amd import _native as nat

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    return nat.default_context()


@pytest.fixture
def table():
    yield
    nat.check(nat.lib().jet_hip_tuning_set(-1, None))


def _force_fp32(M, N, K, B):
    row = (ctypes.c_int32 * 7)(0, *[int(round(math.log2(x))) for x in (M, N, K, B)], 2, 1)
    nat.check(nat.lib().jet_hip_tuning_set(1, row))


def _run(ctx, a, b, B, M, N, K):
    _force_fp32(M, N, K, B)
    say(f"fp32 on bf16 matrix cores: {M}x{N}x{K} batch {B}")
    got, info = contract(ctx, a, [0, 1, 3], [B, M, K], b, [0, 2, 3], [B, N, K], [0, 1, 2],
                         precision=nat.PREC_FP32)
    assert info["kernel"] == "fp32_mfma"
    return got.reshape(B, M, N)


# The smallest size, tile edges and remainders of every tile form (32x32,
# 64x32, 64x64, 128x128, 256x128), k remainders, batches, and odd k
# (dword loads), and 15 rows, which stay on the FP32 instruction.
@pytest.mark.parametrize("M,N,K,B", [
    (16, 16, 16, 1), (17, 33, 18, 1), (32, 32, 64, 3), (33, 65, 130, 1), (31, 95, 1000, 2),
    (129, 33, 62, 1), (500, 1030, 94, 1), (65, 63, 256, 40), (700, 900, 30, 1),
    (1100, 1030, 78, 1), (1030, 2050, 34, 1), (2040, 2040, 1022, 1), (4080, 4090, 130, 1),
    (60, 70, 33, 1), (33, 31, 17, 5), (400, 900, 255, 1),
    (1030, 2050, 51, 1), (15, 70, 64, 1),
    # slices of k: even, a short last one, odd k, a batch
    (64, 64, 4096, 1), (40, 70, 4000, 1), (33, 65, 5001, 1), (64, 96, 3000, 3)])
def test_against_64_bits(ctx, table, M, N, K, B):
    rng = np.random.default_rng(M * N + K)
    a, b = rand_c(rng, B * M * K, np.complex64), rand_c(rng, B * N * K, np.complex64)
    got = _run(ctx, a, b, B, M, N, K)
    want = np.matmul(a.reshape(B, M, K).astype(np.complex128),
                     b.reshape(B, N, K).astype(np.complex128).transpose(0, 2, 1))
    err = np.linalg.norm(got - want) / np.linalg.norm(want)
    assert err < 2.0 ** -24 * (math.sqrt(K) + 8), err


@pytest.mark.parametrize("M,N,K", [(40, 50, 64), (300, 260, 34), (40, 50, 35)])
def test_infinities_and_nan_propagate(ctx, table, M, N, K):
    """Rows and columns with an infinity or NaN give what the four real
    products give in 64 bits; the others are untouched, also where inputs are
    next to the largest and smallest normal numbers."""
    rng = np.random.default_rng(5)
    a, b = (rand_c(rng, n * K, np.complex64).reshape(n, K) for n in (M, N))
    a[3, 5] = complex(np.inf, 1)
    a[7, 0] = complex(2, -np.inf)
    b[2, 7] = complex(np.nan, 0)
    a[9] = 0
    a[9, 1] = np.float32(3.4028e38)       # rounds up past BF16's range
    b[:, 1] *= np.float32(0.125)
    a[11] *= np.float32(2.0 ** -100)
    with np.errstate(all="ignore"):
        ar, ai, br, bi = (x.astype(np.float64) for x in (a.real, a.imag, b.real, b.imag))
        re = np.einsum("mk,nk->mn", ar, br) - np.einsum("mk,nk->mn", ai, bi)
        im = np.einsum("mk,nk->mn", ar, bi) + np.einsum("mk,nk->mn", ai, br)
    got = _run(ctx, a.reshape(-1), b.reshape(-1), 1, M, N, K)[0]
    for g, w in ((got.real, re), (got.imag, im)):
        w = np.where(np.abs(w) > 3.4028235e38, np.sign(w) * np.inf, w)
        assert np.array_equal(np.isnan(g), np.isnan(w))
        assert np.array_equal(np.isinf(g), np.isinf(w))
        assert np.array_equal(np.sign(g[np.isinf(w)]), np.sign(w[np.isinf(w)]))
    ok = np.isfinite(re) & np.isfinite(im) & np.isfinite(got)
    for rows in (slice(0, 9), slice(9, 10), slice(11, 12), slice(12, None)):
        w, g, o = (re + 1j * im)[rows], got[rows], ok[rows]
        err = np.linalg.norm((g[o] - w[o]).astype(np.complex128)) / np.linalg.norm(w[o])
        assert err < 2.0 ** -24 * (math.sqrt(K) + 8), (rows, err)


# The wide tiles' stages of 16 k run three at a time, read ahead by one and loaded
# ahead by three: 3 to 12 stages, whole and partial last ones (256x128, then
# 128x128 tiles).
@pytest.mark.parametrize("M,N,K", [
    (4090, 4094, 34), (4096, 4096, 64), (4090, 4094, 80), (4096, 4096, 112), (4090, 4094, 146),
    (4096, 4080, 176), (4090, 4094, 178), (2040, 2044, 974), (2048, 2048, 992),
    (2040, 2044, 1006)])
def test_wide_tile_stages(ctx, table, M, N, K):
    test_against_64_bits(ctx, table, M, N, K, 1)
