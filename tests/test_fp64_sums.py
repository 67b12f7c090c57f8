"""complex64 products with few outputs and a long k sum in FP64.

The split-K form adds every product in FP64, so its result carries one rounding
to complex64 (each part within 2^-24 of itself).  Host: which shapes it keeps in
the FP32 and the split modes, none of them shapes that the in-place form or the
chunks of K take.  GPU: the error of such shapes; and of larger products that
replace a reduction over 256 threads, which rounds each of K / 256 sums in a
thread and eight more in a tree (random, relative to sums that grow with
sqrt(k): 2^-24 (5/4 + sqrt(K) / 48) covers it).
"""
import ctypes
import math

import numpy as np
import pytest

from hiputil import contract, rand_c, say
from jet_amd import _native as nat
from test_circuits_paths import _check_lib

SPLITK = 6
LONG_K = [(16, 32, 65536), (32, 32, 65536), (32, 32, 1 << 20), (32, 48, 262144), (20, 100, 100000),
          (33, 64, 65536), (64, 64, 65536), (16, 1024, 65536)]


def _kernel(mode, M, N, K):
    i32 = lambda *v: (ctypes.c_int32 * len(v))(*v)
    i64 = lambda *v: (ctypes.c_int64 * len(v))(*v)
    out = (ctypes.c_int64 * 7)()
    assert _check_lib().contraction_gemm_plan(mode, -1, i32(0), 2, i32(0, 2), i64(M, K), 2,
                                              i32(1, 2), i64(N, K), 2, i32(0, 1), out) == 0
    return out[0]


@pytest.mark.parametrize("mode", [0, 3, 4])
@pytest.mark.parametrize("M,N,K", LONG_K)
def test_long_k_takes_the_fp64_sums(mode, M, N, K):
    assert _kernel(mode, M, N, K) == SPLITK


def _error(M, N, K, precision):
    rng = np.random.default_rng(M + N + K)
    a, b = rand_c(rng, M * K, np.complex64), rand_c(rng, N * K, np.complex64)
    say(f"{M}x{N}x{K} precision {precision}")
    got, info = contract(nat.default_context(), a, [0, 2], [M, K], b, [1, 2], [N, K], [0, 1],
                         precision=precision)
    want = a.reshape(M, K).astype(np.complex128) @ b.reshape(N, K).astype(np.complex128).T
    return np.linalg.norm(got.reshape(M, N) - want) / np.linalg.norm(want), info["kernel"]


@pytest.mark.gpu
@pytest.mark.parametrize("precision", [nat.PREC_FP32, nat.PREC_F16X3_4M])
@pytest.mark.parametrize("M,N,K", [(16, 32, 65536), (32, 48, 100000), (64, 64, 65536)])
def test_long_k_error(M, N, K, precision):
    err, kernel = _error(M, N, K, precision)
    assert kernel == "splitk"
    assert err < 2.0 ** -24, err


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(32, 4096, 1024), (4096, 32, 4096), (4096, 32, 16384),
                                   (4000, 17, 16000), (100, 100, 1100), (90, 120, 3000)])
def test_replaced_reductions_error(M, N, K):
    err, _ = _error(M, N, K, nat.PREC_FP32)
    assert err < 2.0 ** -24 * (1.25 + math.sqrt(K) / 48), err
