"""Small buffers' slabs serve other block sizes once nothing is in use of them, and
threads that share a context's blocks all finish their work."""
import threading

import numpy as np
import pytest

import jet_amd
from jet_amd import _native as nat
from test_gpu_small_buffers import _ordered

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("first,second", [(65536, 256), (256, 65536), (4096, 1000)])
def test_slabs_are_cut_for_other_sizes(first, second):
    """All 32 slabs of one size, given back: blocks of another size come from
    the same memory, not from allocations of their own; a slab with a block in
    use keeps its size."""
    ctx = nat.Context(nat.default_context().device)
    free = lambda p: nat.check(nat.lib().jet_hip_free(ctx.handle, p))
    ptrs = [_ordered(ctx, first) for _ in range(32 * (1 << 20) // first)]
    used = ptrs.pop(len(ptrs) // 2)
    for p in ptrs:
        free(p)
    spans = sorted(ptrs + [used])
    inside = lambda p: any(q <= p < q + first for q in spans[max(0, np.searchsorted(spans, p) - 1):
                                                             np.searchsorted(spans, p) + 1])
    block = 1 << max(8, (second - 1).bit_length())
    again = [_ordered(ctx, second) for _ in range(31 * (1 << 20) // block)]
    assert len(set(again)) == len(again)
    assert all(inside(p) and not (used <= p < used + first) for p in again)
    for p in again + [used]:
        free(p)
    ctx.synchronize()


def test_threads_all_finish():
    """Every thread contracts with new and reused blocks, and none fails."""
    rng = np.random.default_rng(6)
    mats = rng.normal(size=(4, 16, 16, 2)).view(np.complex128)[..., 0] / 6
    errors, done = [], []

    def work(t):
        try:
            for n in range(30):
                x = jet_amd.Tensor(["a", "b"], [16, 16], mats[t].reshape(-1), dtype=np.complex128)
                for _ in range(8):
                    m = jet_amd.Tensor(["b", "c"], [16, 16], mats[t].reshape(-1),
                                       dtype=np.complex128)
                    x = jet_amd.Tensor.ContractTensors(x, m)
                    x.rename_index(1, "b")
                want = np.linalg.matrix_power(mats[t], 9)
                got = x.get_data().reshape(16, 16)
                assert np.abs(got - want).max() < 16 * 128 * 2.3e-16 * np.abs(want).max()
                done.append((t, n))
        except BaseException as e:  # a failed thread must not pass
            errors.append((t, e))

    threads = [threading.Thread(target=work, args=(t,)) for t in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors and len(done) == 120, errors
