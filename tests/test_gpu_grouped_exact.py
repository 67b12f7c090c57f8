"""FP64 results between grouped steps, shown on integers.

Leaves of small Gaussian integers make every value of a network an integer that
FP64 holds exactly, and every product with a leaf (of two leaves here) one
that complex64 holds too, so that a complex64 network whose other results stay in
FP64 gives the exact integer rounded once.  Results rounded to complex64 anywhere
between (values pass 2^24) would show.
"""
import numpy as np
import pytest

from hiputil import from_device, say, to_device
from jet_amd import _native as nat
from jet_amd.network import DeviceDag, DeviceNetwork
from test_gpu_grouped import _network, _tree

pytestmark = pytest.mark.gpu


def _exact(idx, data, path):
    """Every node's value in Python integers (re, im)."""
    nodes = [(list(i), d.real.astype(int).astype(object), d.imag.astype(int).astype(object))
             for i, d in zip(idx, data)]
    for a, b in path:
        (la, xr, xi), (lb, yr, yi) = nodes[a], nodes[b]
        both = [l for l in la if l in lb]
        dot = lambda x, y: np.tensordot(x, y, axes=([la.index(l) for l in both],
                                                    [lb.index(l) for l in both]))
        nodes.append(([l for l in la if l not in both] + [l for l in lb if l not in both],
                      dot(xr, yr) - dot(xi, yi), dot(xr, yi) + dot(xi, yr)))
    size = lambda v: max(abs(int(x)) for x in np.asarray(v, object).reshape(-1))
    largest = [max(size(r), size(i)) for _, r, i in nodes]
    return nodes, largest


def _integers(rng, shp):
    return [(rng.integers(-3, 4, s) + 1j * rng.integers(-3, 4, s)).astype(np.complex64)
            for s in shp]


def _rounded(node):
    return np.asarray(node[1], np.float64) + 1j * np.asarray(node[2], np.float64)


@pytest.mark.parametrize("seed", range(6))
@pytest.mark.parametrize("n", [18, 20, 22, 24])
def test_network(n, seed):
    ctx = nat.default_context()
    rng = np.random.default_rng(100 * n + seed)
    idx, shp = _network(rng, n, 2, 1)
    steps = _tree(n)
    data = _integers(rng, shp)
    nodes, largest = _exact(idx, data, steps)
    assert max(largest) < 2 ** 51 and max(largest[n:-1]) > 2 ** 25
    say(f"integers: ring of {n}, seed {seed}")
    net = DeviceNetwork(idx, shp, steps, [], dtype=np.complex64, ctx=ctx)
    bufs = [to_device(ctx, d) for d in data]
    out = nat.DeviceBuffer(256, ctx)
    net.execute([b.ptr for b in bufs], out.ptr)
    want = _rounded(nodes[-1]).reshape(-1).astype(np.complex64)
    assert np.array_equal(from_device(out, want.size, np.complex64), want)


@pytest.mark.parametrize("seed", range(6))
def test_dag(seed):
    """Kept results, and others that several steps read."""
    ctx = nat.default_context()
    n = 24
    rng = np.random.default_rng(seed)
    idx, shp = _network(rng, n, 2, 1)
    steps = _tree(n)
    keep = [n + len(steps) - 1, n + 3]
    data = _integers(rng, shp)
    nodes, largest = _exact(idx, data, steps)
    assert max(largest) < 2 ** 51
    say(f"integers: DAG, seed {seed}")
    dag = DeviceDag(idx, shp, steps, keep, dtype=np.complex64, ctx=ctx)
    bufs = [to_device(ctx, d) for d in data]
    dag.launch([b.ptr for b in bufs])
    for k, (labels, got) in dag.kept_values().items():
        lw = nodes[k][0]
        want = _rounded(nodes[k])
        want = np.transpose(want, [lw.index(l) for l in labels]) if labels else want
        assert np.array_equal(got, want.astype(np.complex64)), k
