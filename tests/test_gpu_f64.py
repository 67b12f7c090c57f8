"""The FP64 matrix-core GEMM over its tile forms, slices of k and unaligned
operands, against numpy in extended precision.

Tolerance: each of the 2 K products of an output is rounded into its sum once,
independently: 2^-53 (sqrt(2 K) + 4) normwise.
"""
import ctypes
import math

import numpy as np
import pytest

from hiputil import code, contract, from_device, rand_c, say
from jet_amd import _native as nat

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    return nat.default_context()


@pytest.fixture
def table():
    yield
    nat.check(nat.lib().jet_hip_tuning_set(-1, None))


def _force(M, N, K, B):
    row = (ctypes.c_int32 * 7)(2, *[int(round(math.log2(x))) for x in (M, N, K, B)], 3, 1)
    nat.check(nat.lib().jet_hip_tuning_set(1, row))


def _want(a, b):
    """a b^T summed in extended precision."""
    out = np.zeros((a.shape[0], b.shape[0]), np.clongdouble)
    x, y = a.astype(np.clongdouble), b.astype(np.clongdouble)
    for k in range(a.shape[1]):
        out += np.outer(x[:, k], y[:, k])
    return out


def _close(got, want, K):
    err = np.sqrt(float((np.abs(got - want) ** 2).sum() / (np.abs(want) ** 2).sum()))
    assert err < 2.0 ** -53 * (math.sqrt(2 * K) + 4), err


# Smallest sizes, tile edges and remainders, k remainders of 8 and 16, batches,
# slices of k (an uneven last one), and the 128x128 form.
@pytest.mark.parametrize("M,N,K,B", [
    (1, 1, 1, 1), (16, 16, 7, 1), (33, 31, 8, 1), (17, 65, 17, 2), (64, 100, 40, 3),
    (40, 70, 4000, 1), (64, 64, 2048, 1), (33, 65, 3001, 2), (300, 200, 33, 1)])
def test_against_extended_precision(ctx, table, M, N, K, B):
    _force(M, N, K, B)
    rng = np.random.default_rng(M + N + K)
    a, b = (rand_c(rng, B * n * K, np.complex128).reshape(B, n, K) for n in (M, N))
    say(f"fp64 matrix cores: {M}x{N}x{K} batch {B}")
    got, info = contract(ctx, a.reshape(-1), [0, 1, 3], [B, M, K], b.reshape(-1), [0, 2, 3],
                         [B, N, K], [0, 1, 2], workspace=True)
    assert info["kernel"] == "fp64_mfma"
    got = got.reshape(B, M, N)
    for i in range(B):
        _close(got[i], _want(a[i], b[i]), K)


def test_large_tiles(ctx, table):
    M, N, K = 2060, 2100, 130
    _force(M, N, K, 1)
    rng = np.random.default_rng(1)
    a, b = (rand_c(rng, n * K, np.complex128).reshape(n, K) for n in (M, N))
    say(f"fp64 matrix cores, 128x128 tiles: {M}x{N}x{K}")
    got, _ = contract(ctx, a.reshape(-1), [0, 2], [M, K], b.reshape(-1), [1, 2], [N, K], [0, 1])
    rows = [*range(0, M, 97), M - 1]
    _close(got.reshape(M, N)[rows], _want(a[rows], b), K)


def test_unaligned_operands(ctx, table):
    """Operands on 8-byte boundaries take dword loads."""
    M, N, K = 70, 50, 41
    _force(M, N, K, 1)
    rng = np.random.default_rng(2)
    a, b = (rand_c(rng, n * K, np.complex128).reshape(n, K) for n in (M, N))
    plan = ctypes.c_void_p()
    nat.check(nat.lib().jet_hip_contraction_plan_create(
        ctx.handle, code(np.complex128), 0, nat.ROW_MAJOR, 2, nat.i32([0, 2]), nat.i64([M, K]), 2,
        nat.i32([1, 2]), nat.i64([N, K]), 2, nat.i32([0, 1]), ctypes.byref(plan)))
    bufs = []
    for x in (a, b):
        buf = nat.DeviceBuffer(x.nbytes + 16, ctx)
        buf.upload(np.concatenate([np.zeros(8, np.uint8), x.reshape(-1).view(np.uint8)]))
        bufs.append(buf)
    out = nat.DeviceBuffer(M * N * 16, ctx)
    say("fp64 matrix cores, operands on 8-byte boundaries")
    nat.check(nat.lib().jet_hip_contract(plan, bufs[0].ptr + 8, bufs[1].ptr + 8, out.ptr, None, 0,
                                         None))
    _close(from_device(out, M * N, np.complex128).reshape(M, N), _want(a, b), K)
