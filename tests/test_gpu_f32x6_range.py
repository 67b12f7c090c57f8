"""FP32 products on the BF16 matrix cores over the whole range of FP32.

A row scaled by a power of two and every column by its inverse leave the
products what they were, so the results of scaled operands equal those of the
operands themselves bit for bit, as far as no value leaves FP32's normal range:
operands down to 2^-125 keep their 24 bits.  Values and results too large for the
scaled sums are computed with the FP32 instruction: every partial sum rounded at
most four times a k, so the error stays under 2^-24 (4 K + 1) of the sum of
the products' magnitudes.
"""
import numpy as np
import pytest

from hiputil import say
from test_gpu_f32x6 import _run, ctx, table  # noqa: F401  (fixtures)

pytestmark = pytest.mark.gpu

# One shape for each tile form: 32x32 (odd k too), 64x32, 64x64, 128x128,
# 256x128, and slices of k.
SHAPES = [(40, 50, 64), (40, 50, 35), (700, 900, 30), (500, 1030, 94), (1030, 2050, 34),
          (4080, 4090, 66), (40, 70, 4000)]


def _values(rng, *shape):
    """Complex values whose parts have magnitudes from 1 to 2 and 24 bits."""
    def part():
        return (1 + rng.integers(0, 1 << 23, shape) / 2.0 ** 23) * rng.choice([-1.0, 1.0], shape)
    return (part() + 1j * part()).astype(np.complex64)


@pytest.mark.parametrize("shift", [100, 112, 118, 122, 125, -60, -76])
@pytest.mark.parametrize("M,N,K", SHAPES)
def test_scaled_operands_are_bitwise_the_same(ctx, table, M, N, K, shift):  # noqa: F811
    rng = np.random.default_rng(M + N + K)
    a, b = _values(rng, M, K), _values(rng, N, K)
    s = np.float32(2.0 ** shift)
    say(f"operands scaled by 2^{-shift}")
    want = _run(ctx, a.reshape(-1), b.reshape(-1), 1, M, N, K)
    # columns of b at most 2^77, so that its values stay in the scaled range
    cap = np.float32(2.0 ** max(-100, min(shift, 76)))
    got = _run(ctx, (a / s).reshape(-1), (b * cap).reshape(-1), 1, M, N, K)
    ratio = np.float32(cap / s)
    assert np.array_equal(got, want * ratio)


@pytest.mark.parametrize("rows,columns", [(103, -103), (126, -126), (126, 0), (60, 30), (50, 62), (112, -112), (48, 48)])
@pytest.mark.parametrize("M,N,K", SHAPES)
def test_large_values(ctx, table, M, N, K, rows, columns):  # noqa: F811
    """Some rows and all columns scaled: the sums' range is left, FP32's is not."""
    rng = np.random.default_rng(M + N + K)
    a, b = _values(rng, M, K), _values(rng, N, K)
    a /= np.float32(2.0 * K)
    a[::3] *= np.float32(2.0 ** rows)
    b *= np.float32(2.0 ** columns)
    got = _run(ctx, a.reshape(-1), b.reshape(-1), 1, M, N, K)[0].astype(np.complex128)
    m = min(M, 96)
    x, y = a[:m].astype(np.complex128), b.astype(np.complex128)
    want = x @ y.T
    bound = (np.abs(x.real) + np.abs(x.imag)) @ (np.abs(y.real) + np.abs(y.imag)).T
    err = np.abs(got[:m] - want)
    assert np.all(err <= 2.0 ** -24 * (4 * K + 1) * bound + 2.0 ** -148), (err / bound).max()


@pytest.mark.parametrize("M,N,K", [(40, 50, 35), (4080, 4090, 66)])
def test_operands_of_nan(ctx, table, M, N, K):  # noqa: F811
    a = np.full(M * K, complex(np.nan, np.nan), np.complex64)
    b = _values(np.random.default_rng(1), N, K).reshape(-1)
    got = _run(ctx, a, b, 1, M, N, K)
    assert np.all(np.isnan(got.real)) and np.all(np.isnan(got.imag))
