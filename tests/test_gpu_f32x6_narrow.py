"""FP32 products with a side below 16 on the BF16 matrix cores: every width from one,
odd k, batches, slices of k.  Tolerance as in test_gpu_f32x6.py: 2^-24 (sqrt(K) + 8)."""
import math

import numpy as np
import pytest

from hiputil import rand_c
from test_gpu_f32x6 import _run, ctx, table  # noqa: F401  (fixtures)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N,K,B", [
    (1, 1, 16, 1), (1, 40, 64, 1), (70, 1, 33, 1), (2, 3, 17, 5), (5, 5, 64, 300), (7, 500, 100, 1),
    (12, 3000, 1000, 1), (3000, 12, 64, 1), (15, 15, 4000, 1), (9, 2463, 256, 1), (300, 10, 87, 2),
    (3, 70, 5001, 1)])
def test_against_64_bits(ctx, table, M, N, K, B):  # noqa: F811
    rng = np.random.default_rng(M * N + K)
    a, b = rand_c(rng, B * M * K, np.complex64), rand_c(rng, B * N * K, np.complex64)
    got = _run(ctx, a, b, B, M, N, K)
    want = np.matmul(a.reshape(B, M, K).astype(np.complex128),
                     b.reshape(B, N, K).astype(np.complex128).transpose(0, 2, 1))
    err = np.linalg.norm(got - want) / np.linalg.norm(want)
    assert err < 2.0 ** -24 * (math.sqrt(K) + 8), err
