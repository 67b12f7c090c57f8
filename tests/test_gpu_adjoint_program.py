"""AdjointProgram's environments: arrays in each leaf's label order, also of
leaves without indices, as views of the one region that an execution reads back."""
import numpy as np
import pytest

from hiputil import say, to_device
from jet_amd import _native as nat
from jet_amd.gradient import AdjointProgram

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,tol", [(np.complex64, 1e-5), (np.complex128, 1e-13)])
def test_environments(dtype, tol):
    ctx = nat.default_context()
    rng = np.random.default_rng(3)
    idx = [["a", "b", "c"], ["c", "d"], ["d", "b", "a"], []]
    dims = {"a": 4, "b": 2, "c": 8, "d": 16}
    shp = [[dims[l] for l in ix] for ix in idx]
    data = [np.asarray(rng.standard_normal(s) + 1j * rng.standard_normal(s)).astype(dtype)
            for s in shp]
    prog = AdjointProgram(idx, shp, [(0, 1), (4, 2), (5, 3)], [0, 1, 2, 3], dtype=dtype, ctx=ctx)
    say(f"environments of three tensors and a number, {np.dtype(dtype).name}")
    bufs = [to_device(ctx, d.reshape(-1)) for d in data]
    for _ in range(3):
        root, envs = prog.run([b.ptr for b in bufs])
        x, y, z, s = (d.astype(np.complex128) for d in data)
        ring = np.einsum("abc,cd,dba->", x, y, z)
        want = {0: s * np.einsum("cd,dba->abc", y, z), 1: s * np.einsum("abc,dba->cd", x, z),
                2: s * np.einsum("abc,cd->dba", x, y), 3: np.asarray(ring)}
        assert abs(root - complex(ring * s)) < tol * abs(ring * s) * 10
        for w, env in envs.items():
            assert isinstance(env, np.ndarray) and not env.flags.owndata, w
            assert env.shape == tuple(shp[w]) and env.dtype == dtype
            assert np.linalg.norm(env - want[w]) < tol * 10 * np.linalg.norm(want[w]), w
