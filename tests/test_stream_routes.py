"""The cases of the in-place forms' tests reach those forms, and every k and column
count of the short-k form runs on the GPU through it.

Tolerance on the GPU as in test_stream.py: at most 16 products summed one after
the other, each rounded twice: under 8 units of 2^-24 (2^-53) normwise.
"""
import ctypes

import numpy as np
import pytest

import test_stream
from hiputil import contract, rand_c, say
from jet_amd import _native as nat
from test_routes import FEW_OUTPUTS, SHORT_K, lib as routes  # noqa: F401  (fixture)
from test_stream import _args, _case, _dot_case, _want, lib as streams  # noqa: F401


def _form(routes, mode, a, b, c, ext):  # noqa: F811
    out = (ctypes.c_int64 * 5)()
    assert routes.contraction_route(mode, *_args(a, b, c, ext), out) == 0
    return out[0]


def test_emulated_cases_are_accepted(streams):  # noqa: F811
    """Most random cases of the offset tests pass through the emulation."""
    size = lambda ms, ext: int(np.prod([ext[m] for m in ms])) if ms else 1
    p = lambda v: v.ctypes.data_as(ctypes.POINTER(ctypes.c_double))

    def accepted(call, a, b, c, ext):
        x, y = np.zeros(size(a, ext), complex), np.zeros(size(b, ext), complex)
        got = np.zeros(size(c, ext), complex)
        return call(*_args(a, b, c, ext), p(x), p(y), ctypes.c_int64(size(c, ext)), p(got)) == 0

    short = 0
    for seed in range(40):
        rng = np.random.default_rng(seed)
        rows, k = int(rng.integers(9, 12)), int(rng.integers(0, 5))
        n, batch = int(rng.integers(0, 5)), int(rng.integers(0, 3))
        case = _case(rng, rows, k, n, batch, ["natural", "scrambled"][seed % 2])
        short += accepted(streams.stream_shortk_emulate, *case)
    few = 0
    for elem in (8, 16):
        for seed in range(30):
            rng = np.random.default_rng(seed)
            m, n, batch = (int(x) for x in rng.integers(0, [5, 5, 4]))
            case = _dot_case(rng, int(rng.integers(12, 14)), m, n, batch, bool(seed % 2))
            few += accepted(lambda *v: streams.stream_dot_emulate(elem, *v), *case)
    assert short >= 20 and few >= 20, (short, few)


def test_few_output_cases_reach_the_form(routes):  # noqa: F811
    marks = [m for m in test_stream.test_gpu_few_outputs.pytestmark if m.name == "parametrize"]
    cases = next(m.args[1] for m in marks if m.args[0].startswith("k,"))
    for k, m, n, batch, spread in cases:
        if m + n == 0 and batch == 0:
            continue                       # a single product may stay with split-K
        a, b, c, ext = _dot_case(np.random.default_rng(k + 7 * m + 11 * n), k, m, n, batch, spread)
        for mode in (0, 2):
            assert _form(routes, mode, a, b, c, ext) == FEW_OUTPUTS, (k, m, n, batch, mode)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,mode,u", [(np.complex64, 0, 2.0 ** -24),
                                          (np.complex128, 2, 2.0 ** -53)])
@pytest.mark.parametrize("k", range(5))
@pytest.mark.parametrize("n", range(5))
def test_gpu_short_k(routes, dtype, mode, u, k, n):  # noqa: F811
    """From 2^21 multiply-adds; k or rows on the lowest address bits, batches."""
    rng = np.random.default_rng(10 * k + n)
    rows = 21 - k - n
    for batch in (0, 2):
        a, b, c, ext = _case(rng, rows - batch, k, n, batch, "natural")
        assert _form(routes, mode, a, b, c, ext) == SHORT_K
        size = lambda ms: int(np.prod([ext[m] for m in ms])) if ms else 1
        x, y = rand_c(rng, size(a), dtype), rand_c(rng, size(b), dtype)
        say(f"in place: {rows} rows, k {k}, n {n}, batch {batch}, {np.dtype(dtype).name}")
        got, _ = contract(nat.default_context(), x, a, [ext[m] for m in a], y, b,
                          [ext[m] for m in b], c, workspace=True)
        wide = np.complex128 if dtype == np.complex64 else np.clongdouble
        want = _want(a, b, c, ext, x.astype(wide), y.astype(wide))
        assert np.linalg.norm(got - want) < 8 * u * np.linalg.norm(want)
