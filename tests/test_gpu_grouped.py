"""Groups of small network steps in one launch, against numpy in 64 bits:
executed eagerly and replayed as a graph with other work between replays, on
two sets of leaves in turn, in complex64 and complex128.

Tolerance: relative to the sum of absolute values, each of the at most 12
steps on a value's way rounds its products and sums (K <= 2^10, tree or
sequential) by less than 2^10 units: generous 1e-4 / 1e-12 on results of
order one; the step widths make the errors far smaller.
"""
import numpy as np
import pytest

from hiputil import from_device, say, to_device
from jet_amd import _native as nat
from jet_amd.network import DeviceDag, DeviceNetwork

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    return nat.default_context()


def _network(rng, n, bond, extra):
    """A ring of n tensors with `extra` modes shared by opposite ones."""
    idx, shp = [], []
    for i in range(n):
        idx.append([f"r{i}", f"r{(i + 1) % n}", f"x{i % (n // 2)}"])
        shp.append([bond, bond, extra])
    return idx, shp


def _leaves(rng, shp, dtype):
    return [((rng.standard_normal(s) + 1j * rng.standard_normal(s)) /
             np.sqrt(s[0] * s[2])).astype(dtype) for s in shp]


def _contract(idx, data, path):
    nodes = [(list(i), d.astype(np.complex128)) for i, d in zip(idx, data)]
    for a, b in path:
        (la, x), (lb, y) = nodes[a], nodes[b]
        both = [l for l in la if l in lb]
        z = np.tensordot(x, y, axes=([la.index(l) for l in both], [lb.index(l) for l in both]))
        nodes.append(([l for l in la if l not in both] + [l for l in lb if l not in both], z))
    return nodes


def _tree(n):
    """Pairwise levels, then a chain."""
    path, level, nxt = [], list(range(n)), n
    while len(level) > 1:
        up = []
        for i in range(0, len(level) - 1, 2):
            path.append((level[i], level[i + 1]))
            up.append(nxt)
            nxt += 1
        level = up + level[len(level) - len(level) % 2:]
    return path


# bond 2: every step grouped; bond 8 and 16: large steps between groups, k up to 2^8 and
# beyond the group's limits; n of 18 leaves just over the 16 steps that are worth a group.
@pytest.mark.parametrize("dtype,tol", [(np.complex64, 1e-4), (np.complex128, 1e-12)])
@pytest.mark.parametrize("n,bond,extra", [(18, 2, 1), (18, 4, 2), (20, 16, 1), (24, 8, 2)])
def test_network(ctx, dtype, tol, n, bond, extra):
    rng = np.random.default_rng(n + bond)
    idx, shp = _network(rng, n, bond, extra)
    path = _tree(n)
    say(f"grouped steps: ring of {n}, bond {bond}, extra {extra}, {np.dtype(dtype).name}")
    net = DeviceNetwork(idx, shp, path, [], dtype=dtype, ctx=ctx)
    sets = []
    for _ in range(2):
        data = _leaves(rng, shp, dtype)
        want = complex(_contract(idx, data, path)[-1][1])
        sets.append(([to_device(ctx, d) for d in data], want,
                     nat.DeviceBuffer(16, ctx)))
    for bufs, want, out in sets + sets:
        net.execute([b.ptr for b in bufs], out.ptr)
        assert abs(from_device(out, 1, dtype)[0] - want) < tol * max(1, abs(want))
    other = nat.DeviceBuffer(1 << 20, ctx)
    for bufs, want, out in sets + sets:
        for _ in range(3):
            net.launch([b.ptr for b in bufs], out.ptr)
            got = from_device(out, 1, dtype)[0]
            assert abs(got - want) < tol * max(1, abs(want))
            out.upload(np.zeros(1, dtype))
            other.upload(np.ones(1 << 17, np.float64))


@pytest.mark.parametrize("dtype,tol", [(np.complex64, 1e-4), (np.complex128, 1e-12)])
def test_open_modes(ctx, dtype, tol):
    """Batched slices: an open mode on every leaf is a batch bit of each step."""
    rng = np.random.default_rng(3)
    n = 18
    idx, shp = _network(rng, n, 2, 2)
    path = _tree(n)
    say(f"grouped steps with an open mode, {np.dtype(dtype).name}")
    data = _leaves(rng, shp, dtype)
    open_mode = "x1"
    net = DeviceNetwork(idx, shp, path, [open_mode], dtype=dtype, ctx=ctx)
    bufs = [to_device(ctx, d) for d in data]
    out = nat.DeviceBuffer(32, ctx)
    net.execute([b.ptr for b in bufs], out.ptr)
    got = from_device(out, 2, dtype)
    for v in range(2):
        cut = [(ix, d) if open_mode not in ix else
               ([l for l in ix if l != open_mode], np.take(d, v, axis=ix.index(open_mode)))
               for ix, d in zip(idx, data)]
        want = complex(_contract([c[0] for c in cut], [c[1] for c in cut], path)[-1][1])
        assert abs(got[v] - want) < tol * max(1, abs(want))


@pytest.mark.parametrize("dtype,tol", [(np.complex64, 1e-4), (np.complex128, 1e-12)])
def test_dag_kept_results(ctx, dtype, tol):
    """Steps whose results feed several steps, some kept."""
    rng = np.random.default_rng(7)
    n = 18
    idx, shp = _network(rng, n, 4, 1)
    steps = _tree(n) + [(0, 2), (1, 3), (n, 4)]
    keep = [n, n + 3, n + len(_tree(n)) - 1, n + len(steps) - 1]
    say(f"grouped steps of a DAG, {np.dtype(dtype).name}")
    data = _leaves(rng, shp, dtype)
    dag = DeviceDag(idx, shp, steps, keep, dtype=dtype, ctx=ctx)
    bufs = [to_device(ctx, d) for d in data]
    nodes = _contract(idx, data, steps)
    for _ in range(3):
        dag.launch([b.ptr for b in bufs])
        for k, (labels, got) in dag.kept_values().items():
            lw, want = nodes[k]
            want = np.transpose(want, [lw.index(l) for l in labels]) if labels else want
            assert np.linalg.norm(got - want) < tol * max(1, np.linalg.norm(want))
