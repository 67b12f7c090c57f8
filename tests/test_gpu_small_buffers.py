"""Small tensors and the blocks they live in: blocks are reused while earlier
work on them is still queued, by several threads, and go back with the context."""
import ctypes
import threading

import numpy as np
import pytest

import jet_amd
from jet_amd import _native as nat

pytestmark = pytest.mark.gpu


def _ordered(ctx, nbytes):
    p = ctypes.c_void_p()
    nat.check(nat.lib().jet_hip_malloc_ordered(ctx.handle, nbytes, ctypes.byref(p)))
    return p.value


def test_blocks():
    ctx = nat.Context(nat.default_context().device)
    L = nat.lib()
    sizes = [0, 1, 256, 257, 65536, 65537, 1 << 21] + [4096] * 600
    ptrs = [_ordered(ctx, n) for n in sizes]
    spans = sorted((p, p + max(1, n)) for p, n in zip(ptrs, sizes))
    assert all(p % 256 == 0 for p in ptrs)
    assert all(a[1] <= b[0] for a, b in zip(spans, spans[1:]))
    for p in ptrs:
        nat.check(L.jet_hip_free(ctx.handle, p))
    again = [_ordered(ctx, 4096) for _ in range(600)]
    assert len(set(again)) == 600
    # 32 slabs of a megabyte at most: past them, allocations of their own
    many = [_ordered(ctx, 65536) for _ in range(600)]
    assert len(set(many)) == 600
    for p in again + many:
        nat.check(L.jet_hip_free(ctx.handle, p))
    ctx.synchronize()


def test_threads_reuse_blocks():
    """Chains of small contractions whose intermediates are dropped at once."""
    rng = np.random.default_rng(5)
    mats = rng.normal(size=(4, 2, 16, 16, 2)).view(np.complex128)[..., 0] / 6
    bad = []

    def work(t):
        for _ in range(20):
            x = jet_amd.Tensor(["a", "b"], [16, 16], mats[t][0].reshape(-1), dtype=np.complex128)
            y = mats[t][0]
            for i in range(12):
                m = jet_amd.Tensor(["b", "c"], [16, 16], mats[t][i % 2].reshape(-1),
                                   dtype=np.complex128)
                x = jet_amd.Tensor.ContractTensors(x, m)
                x.rename_index(1, "b")
                y = y @ mats[t][i % 2]
            # a chain of 12 products of 16 terms: 12 * 16 roundings and the tests' margin of 16
            if np.abs(x.get_data().reshape(16, 16) - y).max() > 16 * 192 * 2.3e-16 * np.abs(y).max():
                bad.append(t)

    threads = [threading.Thread(target=work, args=(t,)) for t in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad
