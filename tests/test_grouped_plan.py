"""Launch plans of grouped small steps, on the CPU (tests/native/group_check.cpp):
steps run once and after their operands, results alive at the same time
never share memory, for circuits' networks (sliced ones too) and adjoint DAGs with and
without recomputation."""
import ctypes
import os
import subprocess

import pytest

from jet_amd import _native as nat
from jet_amd import build as jb
from jet_amd import circuits, paths
from jet_amd.gradient import adjoint_dag_steps
from jet_amd.network import LabelIds, _flatten

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def lib():
    jb.write_tuning_table()
    out = os.path.join(ROOT, "tests", "native", "_build", f"libgroup_check.{os.getpid()}.so")
    os.makedirs(os.path.dirname(out), exist_ok=True)
    csrc = os.path.join(ROOT, "jet_amd", "csrc")
    subprocess.run(["g++", "-std=c++17", "-O2", "-fPIC", "-shared",
                    "-I" + os.path.join(ROOT, "include"), "-I" + jb.BUILD, "-o", out,
                    os.path.join(ROOT, "tests", "native", "group_check.cpp")] +
                   [os.path.join(csrc, f) for f in ("network_plan.cpp", "contract_plan.cpp",
                                                    "permute_plan.cpp", "tuning.cpp")],
                   check=True)
    L = ctypes.CDLL(out)
    os.remove(out)
    return L


def _check(lib, dag, indices, shapes, steps, last):
    lab = LabelIds()
    ranks, modes, exts = _flatten(indices, shapes, lab)
    out = [int(x) if dag else lab(x) for x in last]
    nl, ng = ctypes.c_int(), ctypes.c_int()
    rc = lib.check_launches(int(dag), len(indices), nat.i32(ranks), nat.i32(modes), nat.i64(exts),
                            len(steps), nat.i32([x for p in steps for x in p]), len(out),
                            nat.i32(out), ctypes.byref(nl), ctypes.byref(ng))
    assert rc == 0, rc
    return nl.value, ng.value


@pytest.mark.parametrize("shape,n_sliced", [((3, 3, 4), 0), ((4, 4, 8), 0), ((4, 4, 10), 3),
                                            ((5, 5, 8), 2)])
def test_networks(lib, shape, n_sliced):
    circ = circuits.random_grid_circuit(*shape, seed=5)
    net = circuits.amplitude_network(circ)
    dims = {x: 2 for ix in net.indices for x in ix}
    path = paths.best_greedy_path(net.indices, dims, trials=2)
    sliced = paths.choose_slices(net.indices, dims, path, n_sliced) if n_sliced else []
    launches, grouped = _check(lib, False, net.indices, net.shapes, path, sliced)
    assert grouped > 0.8 * len(path) and launches < len(path) / 4, (launches, grouped, len(path))


@pytest.mark.parametrize("shape", [(4, 4, 8), (4, 5, 8)])
@pytest.mark.parametrize("every", [0, 1, 2, 4, 7])
def test_adjoint_dags(lib, shape, every):
    circ = circuits.random_grid_circuit(*shape, seed=5, random_angles=True)
    net = circuits.amplitude_network(circ)
    dims = {x: 2 for ix in net.indices for x in ix}
    path = paths.best_minfill_path(net.indices, dims, trials=2, seed=1)
    wanted = [circ.n_qubits + i for i, g in enumerate(circ.gates) if g.param_index is not None]
    plan = adjoint_dag_steps(net.indices, path, wanted, every)
    launches, grouped = _check(lib, True, net.indices + [[]], net.shapes + [[]], plan["steps"],
                               [plan["root_node"]] + [plan["env_node"][w] for w in wanted])
    assert launches < len(plan["steps"]) / 4, (launches, grouped, len(plan["steps"]))


def test_few_steps_run_alone(lib):
    indices = [["a", "b"], ["b", "c"], ["c", "a"]]
    assert _check(lib, False, indices, [[2, 2]] * 3, [(0, 1), (3, 2)], []) == (2, 0)
