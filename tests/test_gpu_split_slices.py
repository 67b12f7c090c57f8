"""4M split GEMMs whose k is cut into slices that fill the CUs (few 128x128
tiles, long k), against numpy in 64 bits.

Tolerance: the split keeps 22 (FP16) or 16 (BF16) significant bits of each
operand, normwise 2^-21 or 2^-15 per product, and the FP32 sums are rounded
at most 6 times per 32 k: 2^-24 sqrt(6 K / 32).
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


MODES = {"f16x3": (nat.PREC_F16X3_4M, 4, 7, 2.0 ** -21),
         "bf16x3_4m": (nat.PREC_BF16X3_4M, 3, 5, 2.0 ** -15)}


# k of 15 (one slice), 16 and 17 tiles of 32 (two slices, the second short),
# a k remainder, many slices, a batch, and 128 and 129 tiles.
@pytest.mark.parametrize("mode", sorted(MODES))
@pytest.mark.parametrize("M,N,K,B", [
    (128, 128, 480, 1), (128, 128, 512, 1), (130, 129, 544, 1), (200, 140, 1001, 1),
    (140, 150, 12000, 1), (129, 128, 2100, 3), (1024, 2048, 512, 1), (1025, 1800, 512, 1)])
def test_against_64_bits(ctx, table, mode, M, N, K, B):
    prec, mode_id, kernel, split = MODES[mode]
    row = (ctypes.c_int32 * 7)(mode_id, *[int(round(math.log2(x))) for x in (M, N, K, B)],
                               kernel, 1)
    nat.check(nat.lib().jet_hip_tuning_set(1, row))
    rng = np.random.default_rng(M + N + K)
    a, b = rand_c(rng, B * M * K, np.complex64), rand_c(rng, B * N * K, np.complex64)
    say(f"{mode} slices: {M}x{N}x{K} batch {B}")
    got, info = contract(ctx, a, [0, 1, 3], [B, M, K], b, [0, 2, 3], [B, N, K], [0, 1, 2],
                         precision=prec, workspace=True)
    assert info["kernel"] == nat.GEMM_KERNEL_NAMES[kernel]
    want = np.matmul(a.reshape(B, M, K).astype(np.complex128),
                     b.reshape(B, N, K).astype(np.complex128).transpose(0, 2, 1))
    err = np.linalg.norm(got.reshape(B, M, N) - want) / np.linalg.norm(want)
    assert err < split + 2.0 ** -24 * math.sqrt(6 * K / 32), err
