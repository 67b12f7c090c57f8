"""In-place contractions of a small tensor with a large one, and of two large
tensors with few outputs: the plans' offset
arithmetic on the CPU (tests/native/stream_check.cpp) against numpy's einsum
over random mode orders, batch modes and permuted results, which forms are
refused, and the kernels on the GPU against numpy in 64 bits.

GPU tolerance: K <= 16 products summed one after the other, each rounded
twice: 2 K units of 2^-24 (2^-53) of the sum of magnitudes, normwise under
2^-24 * 8 (2^-53 * 8) for random operands.  The few-output form sums in FP64: 2^-23
for complex64 (the result's rounding), 2^-53 sqrt(K) for complex128.
"""
import ctypes
import os
import subprocess

import numpy as np
import pytest

from hiputil import contract, rand_c, say
from jet_amd import _native as nat
from jet_amd import build as jb

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LETTERS = "abcdefghijklmnopqrstuvwxyzABCDEFGHIJKLMNOPQRSTUVWXYZ"


@pytest.fixture(scope="module")
def lib():
    jb.write_tuning_table()
    out = os.path.join(ROOT, "tests", "native", "_build", f"libstream_check.{os.getpid()}.so")
    os.makedirs(os.path.dirname(out), exist_ok=True)
    csrc = os.path.join(ROOT, "jet_amd", "csrc")
    subprocess.run(["g++", "-std=c++17", "-O2", "-fPIC", "-shared",
                    "-I" + os.path.join(ROOT, "include"), "-I" + jb.BUILD, "-o", out,
                    os.path.join(ROOT, "tests", "native", "stream_check.cpp")] +
                   [os.path.join(csrc, f) for f in ("contract_plan.cpp", "permute_plan.cpp",
                                                    "tuning.cpp")], check=True)
    L = ctypes.CDLL(out)
    os.remove(out)
    return L


def _case(rng, rows, k, n, batch, order):
    """Modes of extent 2 (two of extent 4), scrambled; C in the operands'
    order ("natural": A's other modes, then B's) or scrambled."""
    ids = list(range(rows + k + n + batch))
    r, kk = ids[:rows], ids[rows:rows + k]
    nn, bb = ids[rows + k:rows + k + n], ids[rows + k + n:]
    big = [int(x) for x in rng.permutation(r + kk)]
    big = bb + big
    small = [int(x) for x in rng.permutation(kk + nn + bb)]
    flip = bool(rng.integers(2))
    a, b = (small, big) if flip else (big, small)
    c = bb + [m for m in a if m not in b] + [m for m in b if m not in a]
    if order == "scrambled":
        c = bb + [int(x) for x in rng.permutation(r + nn)]
    ext = {m: 2 for m in ids}
    for m in rng.choice(r + kk, 2, replace=False) if k < 3 else []:
        ext[int(m)] = 4
    return a, b, c, ext


def _args(a, b, c, ext):
    e = lambda ms: nat.i64([ext[m] for m in ms])
    return (len(a), nat.i32(a), e(a), len(b), nat.i32(b), e(b), len(c), nat.i32(c))


def _want(a, b, c, ext, x, y):
    sub = lambda ms: "".join(LETTERS[m] for m in ms)
    return np.einsum(f"{sub(a)},{sub(b)}->{sub(c)}", x.reshape([ext[m] for m in a]),
                     y.reshape([ext[m] for m in b]), optimize=True).reshape(-1)


@pytest.mark.parametrize("seed", range(40))
def test_offsets_match_einsum(lib, seed):
    rng = np.random.default_rng(seed)
    rows, k = int(rng.integers(9, 12)), int(rng.integers(0, 5))
    n, batch = int(rng.integers(0, 5)), int(rng.integers(0, 3))
    a, b, c, ext = _case(rng, rows, k, n, batch, ["natural", "scrambled"][seed % 2])
    size = lambda ms: int(np.prod([ext[m] for m in ms])) if ms else 1
    x = rng.standard_normal(size(a)) + 1j * rng.standard_normal(size(a))
    y = rng.standard_normal(size(b)) + 1j * rng.standard_normal(size(b))
    got = np.zeros(size(c), np.complex128)
    p = lambda v: v.ctypes.data_as(ctypes.POINTER(ctypes.c_double))
    rc = lib.stream_shortk_emulate(*_args(a, b, c, ext), p(x), p(y), ctypes.c_int64(size(c)),
                                   p(got))
    if rc == 1:   # refused: more than 16 k, or a scrambled result's lowest bits far up in rows
        log2k = sum(ext[m] // 2 for m in a if m in b and m not in c)
        assert log2k > 4 or seed % 2 == 1
        return
    assert rc == 0
    np.testing.assert_allclose(got, _want(a, b, c, ext, x, y), rtol=1e-12, atol=1e-12)


def test_refused_forms(lib):
    def route(a, b, c, ext):
        ws = ctypes.c_size_t()
        return lib.stream_route(*_args(a, b, c, ext), ctypes.byref(ws)), ws.value
    rows = list(range(16))
    two = {m: 2 for m in range(30)}
    gate = ([*rows[:7], 16, *rows[7:]], [17, 16], [*rows, 17])
    assert route(*gate, two) == (1, 0)
    assert route(*gate, {**two, 3: 3})[0] == 0                 # not a power of two
    assert route(*gate, {**two, 16: 32})[0] == 0               # 32 k
    assert route(*gate, {**two, 17: 32})[0] == 0               # 32 columns
    batched = ([18, *rows[:7], 16, *rows[7:]], [18, 17, 16], [18, *rows, 17])
    assert route(*batched, two) == (1, 0)
    assert route([*rows[:7], 16, *rows[7:], 18], [18, 17, 16], [18, *rows, 17], two)[0] == 0
    # the result's fastest mode is a far row
    assert route(gate[0], gate[1], [*rows[1:], 17, 0], two)[0] == 0
    # below 2^14 elements
    assert route([*rows[:5], 16, *rows[5:12]], [17, 16], [*rows[:12], 17], two)[0] == 0


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,u", [(np.complex64, 2.0 ** -24), (np.complex128, 2.0 ** -53)])
@pytest.mark.parametrize("seed", range(24))
def test_gpu(dtype, u, seed):
    """Every k and n count of the form, k or rows on the lowest address bit,
    either operand large, rows of one to many steps."""
    rng = np.random.default_rng(100 + seed)
    rows, k, n = int(rng.integers(12, 19)), seed % 5, (seed // 5) % 5
    a, b, c, ext = _case(rng, rows, k, n, int(rng.integers(0, 3)), "natural")
    size = lambda ms: int(np.prod([ext[m] for m in ms])) if ms else 1
    x, y = rand_c(rng, size(a), dtype), rand_c(rng, size(b), dtype)
    say(f"in place: {rows} rows, k {k}, n {n}, {np.dtype(dtype).name}, seed {seed}")
    got, _ = contract(nat.default_context(), x, a, [ext[m] for m in a], y, b,
                      [ext[m] for m in b], c, workspace=True)
    want = _want(a, b, c, ext, x.astype(np.complex128), y.astype(np.complex128))
    if dtype == np.complex128:
        want = _want(a, b, c, ext, x.astype(np.clongdouble), y.astype(np.clongdouble))
    assert np.linalg.norm(got - want) < 8 * u * np.linalg.norm(want)


def _dot_case(rng, k, m, n, batch, spread):
    """Modes of extent 2; batch modes leading, or anywhere (spread)."""
    ids = list(range(k + m + n + batch))
    kk, mm = ids[:k], ids[k:k + m]
    nn, bb = ids[k + m:k + m + n], ids[k + m + n:]
    head = [] if spread else bb
    tail = bb if spread else []
    a = head + [int(x) for x in rng.permutation(kk + mm + tail)]
    b = head + [int(x) for x in rng.permutation(kk + nn + tail)]
    c = [int(x) for x in rng.permutation(bb + mm + nn)]
    return a, b, c, {i: 2 for i in ids}


@pytest.mark.parametrize("elem", [8, 16])
@pytest.mark.parametrize("seed", range(30))
def test_few_outputs_match_einsum(lib, elem, seed):
    rng = np.random.default_rng(seed)
    m, n, batch = (int(x) for x in rng.integers(0, [5, 5, 4]))
    a, b, c, ext = _dot_case(rng, int(rng.integers(12, 14)), m, n, batch, bool(seed % 2))
    size = lambda ms: int(np.prod([ext[x] for x in ms])) if ms else 1
    x = rng.standard_normal(size(a)) + 1j * rng.standard_normal(size(a))
    y = rng.standard_normal(size(b)) + 1j * rng.standard_normal(size(b))
    got = np.zeros(size(c), np.complex128)
    p = lambda v: v.ctypes.data_as(ctypes.POINTER(ctypes.c_double))
    rc = lib.stream_dot_emulate(elem, *_args(a, b, c, ext), p(x), p(y), ctypes.c_int64(size(c)),
                                p(got))
    if rc == 1:   # refused: too many outputs, or low bits that do not fit a tile
        assert m + n > 4 or batch > 0
        return
    assert rc == 0
    np.testing.assert_allclose(got, _want(a, b, c, ext, x, y), rtol=1e-10, atol=1e-9)


def test_few_outputs_routes(lib):
    def route(k, m, n, batch, spread=False, ext=None):
        a, b, c, e = _dot_case(np.random.default_rng(1), k, m, n, batch, spread)
        ws = ctypes.c_size_t()
        return lib.stream_route(*_args(a, b, c, {**e, **(ext or {})}), ctypes.byref(ws)), ws.value
    assert route(18, 2, 1, 0)[0] == 2
    assert 0 < route(18, 2, 1, 4)[1] <= 4 << 20
    assert route(18, 3, 3, 0)[0] == 2
    assert route(18, 5, 0, 0)[0] == 0            # 32 rows
    assert route(18, 4, 4, 0)[0] == 0            # 256 outputs
    assert route(18, 2, 1, 0, ext={0: 3})[0] == 0
    assert route(11, 2, 1, 6)[0] == 0            # 2^11 k
    # one product of operands in the same order: split-K reads each once as it is
    one = {i: 2 for i in range(18)}
    ws = ctypes.c_size_t()
    assert lib.stream_route(*_args(list(range(18)), list(range(18)), [], one),
                            ctypes.byref(ws)) == 0


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [np.complex64, np.complex128])
@pytest.mark.parametrize("k,m,n,batch,spread", [
    (16, 0, 0, 0, False), (16, 2, 1, 0, False), (17, 0, 3, 0, False), (17, 3, 3, 0, False),
    (16, 4, 2, 0, False), (16, 2, 4, 0, False), (16, 1, 0, 5, False), (14, 1, 1, 6, False),
    (16, 1, 1, 2, True), (16, 0, 0, 4, True), (15, 2, 2, 3, True), (20, 1, 2, 0, False),
    (12, 4, 0, 8, False), (12, 0, 4, 10, False)])
def test_gpu_few_outputs(dtype, k, m, n, batch, spread):
    rng = np.random.default_rng(k + 7 * m + 11 * n)
    a, b, c, ext = _dot_case(rng, k, m, n, batch, spread)
    size = lambda ms: int(np.prod([ext[v] for v in ms])) if ms else 1
    x, y = rand_c(rng, size(a), dtype), rand_c(rng, size(b), dtype)
    say(f"few outputs: K 2^{k}, M 2^{m}, N 2^{n}, batch 2^{batch}, {np.dtype(dtype).name}")
    got, _ = contract(nat.default_context(), x, a, [ext[v] for v in a], y, b,
                      [ext[v] for v in b], c, workspace=True)
    want = _want(a, b, c, ext, x.astype(np.complex128), y.astype(np.complex128))
    tol = 2.0 ** -23 if dtype == np.complex64 else 2.0 ** -53 * np.sqrt(2.0 ** k)
    assert np.linalg.norm(got - want) < tol * np.linalg.norm(want)
