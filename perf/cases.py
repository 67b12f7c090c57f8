"""Work that users of jet_amd have it do, as cases that can be timed and checked.

Every case goes through the public entry points: the pairwise contraction
plans of the C ABI on device buffers that the caller owns, the ``Tensor`` and
``TaskBasedContractor`` classes, and the planned networks behind slice loops,
batches of amplitudes and gradients.  Kinds:

* ``pair``: one contraction C[left, right] = sum over common of A * B, the
  modes of A and B in scrambled orders.  ``left``, ``right`` and ``common``
  list mode extents ("2^12" twelve modes of extent 2, "5x7x6" three modes).
  ``api`` "plan": a planned contraction on the caller's buffers (graph
  capture, serving loops); "tensor": ``contract_tensors`` on Tensor objects
  and the result read back (interactive use).
* ``transpose``: one reordering of a tensor's modes on the device.
* ``task``: one amplitude of a small grid circuit through TensorNetwork,
  PathInfo and TaskBasedContractor, contraction by contraction.
* ``amplitudes``: amplitudes of one grid circuit for several bitstrings, one
  launch of an UnevenBatch.
* ``sliced``: one execution of a sliced 7x7 depth-14 amplitude, 2^batch
  slices at once.
* ``gradient``: loss and gradient of |amplitude|^2 with respect to every
  fSim angle of a grid circuit.
"""
import ctypes
import json
import os
import random

import numpy as np
import torch

import jet_amd
from jet_amd import _native as nat
from jet_amd import circuits, paths
from jet_amd.batch import AmplitudeJob, UnevenBatch
from jet_amd.gradient import ParameterizedAmplitude
from jet_amd.network import SlicedContraction

_DATA = os.path.join(os.path.dirname(os.path.abspath(jet_amd.__file__)), "data")
_PRECISION = {"default": nat.PREC_DEFAULT, "f16x3": nat.PREC_F16X3_4M}
_CODE = {"complex64": nat.C64, "complex128": nat.C128}
_TORCH = {"complex64": torch.complex64, "complex128": torch.complex128}

# Circuits whose amplitude paths the package ships.
_AMPLITUDE_CIRCUITS = {"5x5x14": (5, 5, 14, 51), "6x7x10": (6, 7, 10, 53)}


def listed():
    return [
        # The smallest call: two tensors of a few thousand values (the sizes
        # of the package's smoke check), contracted and read back.
        _pair("tiny_tensors", "2x8", "32", "4x16", api="tensor"),
        # A 4x4 depth-8 amplitude contracted step by step: ~200 contractions
        # of a few values each, as scripts written against Jet's classes do.
        {"name": "task_4x4", "kind": "task", "rows": 4, "cols": 4, "depth": 8},
        # A two-qubit gate on a state of 26 qubits: bound by reading and
        # writing the state.
        _pair("gate_on_state", "2^24", "2^2", "2^2"),
        # Closing a network: two large tensors that share almost every index.
        _pair("closing_step", "2^2", "2^1", "2^22"),
        # Bond dimensions that are not powers of two (matrix product states,
        # lattice models), a middle size.
        _pair("ragged_bonds", "5x7x6x6", "11x9x12", "6x13x13"),
        # A large step in the default arithmetic of each data type.
        _pair("large_c64", "2^12", "2^12", "2^12"),
        _pair("large_c128", "2^11", "2^12", "2^11", dtype="complex128"),
        # The largest single contraction of the benchmark: rank 28 by rank 28
        # over 14 shared indices, split-FP16 arithmetic.
        _pair("rank28_split", "2^14", "2^14", "2^14", precision="f16x3"),
        # Reordering a 26-qubit tensor.
        {"name": "transpose_rank26", "kind": "transpose", "modes": "2^26",
         "dtype": "complex64", "order": 3},
        # 24 amplitudes of a 6x7 depth-10 circuit in one launch.
        {"name": "amplitudes_6x7", "kind": "amplitudes", "circuit": "6x7x10", "count": 24,
         "form": "stacked_pow2", "precision": "default"},
        # 32 slices of the 7x7 depth-14 amplitude along the shipped path.
        {"name": "sliced_7x7", "kind": "sliced", "batch": 5, "precision": "f16x3"},
        # One optimisation step's loss and gradient: 6x6 depth 10, 300 angles.
        {"name": "gradient_6x6", "kind": "gradient", "rows": 6, "cols": 6, "depth": 10},
    ]


def draw(rng):
    kind = rng.choice(["tensor", "gate", "closing", "pair", "pair", "pair", "pair",
                       "transpose", "transpose", "task", "amplitudes", "sliced", "gradient"])
    order = rng.randrange(1, 1000)
    dtype = rng.choice(["complex64", "complex64", "complex128"])
    if kind == "tensor":
        return _pair("", _extents(rng, rng.uniform(0, 6), 0.5), _extents(rng, rng.uniform(0, 6), 0.5),
                     _extents(rng, rng.uniform(1, 8), 0.5), api="tensor", dtype=dtype, order=order)
    if kind == "gate":
        q = rng.randint(1, 3)
        n = rng.randint(16, 27 if dtype == "complex64" else 26)
        return _pair("", f"2^{n - q}", f"2^{q}", f"2^{q}", dtype=dtype, order=order)
    if kind == "closing":
        return _pair("", _extents(rng, rng.uniform(0, 3), 0.3), _extents(rng, rng.uniform(0, 3), 0.3),
                     _extents(rng, rng.uniform(12, 22), 0.3), dtype=dtype, order=order)
    if kind == "pair":
        ragged = rng.choice([0.0, 0.0, 1.0])
        low, high = (4, 10.5) if ragged else (4, 13)
        split = dtype == "complex64" and rng.random() < 0.3
        m, n, k = (rng.uniform(low, high) for _ in range(3))
        if dtype == "complex128":  # the arithmetic costs ten times as much
            k = min(k, 34 - m - n)
        return _pair("", _extents(rng, m, ragged), _extents(rng, n, ragged),
                     _extents(rng, max(k, 2), ragged), dtype=dtype, order=order,
                     precision="f16x3" if split else "default")
    if kind == "transpose":
        return {"kind": "transpose", "modes": _extents(rng, rng.uniform(12, 26), 0.5),
                "dtype": dtype, "order": order}
    if kind == "task":
        return {"kind": "task", "rows": rng.randint(3, 4), "cols": rng.randint(3, 4),
                "depth": rng.randint(4, 10)}
    if kind == "amplitudes":
        name = rng.choice(sorted(_AMPLITUDE_CIRCUITS))
        return {"kind": "amplitudes", "circuit": name,
                "count": rng.randint(3, 8 if name == "5x5x14" else 32),
                "form": rng.choice(["each", "stacked", "stacked_pow2"]),
                "precision": rng.choice(["default", "f16x3"])}
    if kind == "sliced":
        precision = rng.choice(["default", "f16x3", "f16x3"])
        return {"kind": "sliced", "batch": rng.randint(0, 4 if precision == "f16x3" else 2),
                "precision": precision}
    return {"kind": "gradient", "rows": rng.randint(4, 6), "cols": rng.randint(4, 6),
            "depth": rng.randint(6, 9)}


def _pair(name, left, right, common, dtype="complex64", precision="default", api="plan", order=1):
    case = {"kind": "pair", "api": api, "left": left, "right": right, "common": common,
            "dtype": dtype, "precision": precision, "order": order}
    return {"name": name, **case} if name else case


def _extents(rng, log2_size, ragged):
    """Mode extents whose product is near 2^log2_size: all 2, or (with
    probability `ragged`) between 2 and 13."""
    if rng.random() >= ragged:
        return f"2^{round(log2_size)}" if round(log2_size) else "1"
    target, size, out = 2.0 ** log2_size, 1, []
    while True:
        e = rng.randint(2, 13)
        if size * e > target:
            break
        size *= e
        out.append(e)
    rest = int(target / size)
    if rest > 1:
        out.append(rest)
    return "x".join(map(str, out)) or "1"


def _modes(text):
    if "^" in text:
        base, count = text.split("^")
        return [int(base)] * int(count)
    return [int(e) for e in text.split("x")]


def _size(shape):
    return int(np.prod(shape, dtype=np.int64)) if len(shape) else 1


def _randn(shape, dtype, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return torch.randn(_size(shape), dtype=_TORCH[dtype], device="cuda", generator=g)


def _pair_layout(case):
    """Labels of A, B and C (A's other modes, then B's) and every extent."""
    left = [f"l{i}" for i in range(len(_modes(case["left"])))]
    right = [f"r{i}" for i in range(len(_modes(case["right"])))]
    common = [f"c{i}" for i in range(len(_modes(case["common"])))]
    dims = dict(zip(left + right + common,
                    _modes(case["left"]) + _modes(case["right"]) + _modes(case["common"])))
    order = random.Random(case["order"])
    a, b = left + common, common + right
    order.shuffle(a)
    order.shuffle(b)
    return a, b, [x for x in a if x in left] + [x for x in b if x in right], dims


def _transpose_layout(case):
    shape = _modes(case["modes"])
    perm = list(range(len(shape)))
    random.Random(case["order"]).shuffle(perm)
    return shape, perm


def _task_network(case, seed):
    circ = circuits.random_grid_circuit(case["rows"], case["cols"], case["depth"], seed=seed)
    return circuits.amplitude_network(circ)


def _amplitude_problem(case, seed):
    rows, cols, depth, path_seed = _AMPLITUDE_CIRCUITS[case["circuit"]]
    circ = circuits.random_grid_circuit(rows, cols, depth, seed=seed)
    rng = np.random.default_rng(seed)
    bits = [tuple(int(x) for x in rng.integers(0, 2, circ.n_qubits)) for _ in range(case["count"])]
    return circ, bits, paths.load_or_make_amplitude_path(rows, cols, depth, path_seed)


def _gradient_problem(case, seed):
    rows, cols, depth = case["rows"], case["cols"], case["depth"]
    circ = circuits.random_grid_circuit(rows, cols, depth, seed=seed, random_angles=True)
    if (rows, cols, depth) == (6, 6, 10):
        path = paths.load_or_make_amplitude_path(6, 6, 10, 2026, random_angles=True)
    else:
        net = circuits.amplitude_network(circ)
        dims = {x: 2 for ix in net.indices for x in ix}
        path = paths.best_minfill_path(net.indices, dims, trials=2, seed=1)
    return circ, path


def _sliced_plan():
    with open(os.path.join(_DATA, "grid_7x7x14_seed2026_s12_refined.json")) as f:
        return json.load(f)


def prepare(case, seed):
    state = _PREPARE[case["kind"]](case, seed)
    torch.cuda.synchronize()
    return {"kind": case["kind"], **state}


def run(state):
    return _RUN[state["kind"]](state)


def _prepare_pair(case, seed):
    a, b, c, dims = _pair_layout(case)
    ea, eb = [dims[x] for x in a], [dims[x] for x in b]
    da = _randn(ea, case["dtype"], 2 * seed)
    db = _randn(eb, case["dtype"], 2 * seed + 1)
    if case["api"] == "tensor":
        dt = np.dtype(case["dtype"])
        return {"pair": (jet_amd.Tensor(a, ea, da.cpu().numpy(), dtype=dt),
                         jet_amd.Tensor(b, eb, db.cpu().numpy(), dtype=dt))}
    ctx, lib = nat.default_context(), nat.lib()
    ids = {x: i for i, x in enumerate(dims)}
    plan, size = ctypes.c_void_p(), ctypes.c_size_t()
    nat.check(lib.jet_hip_contraction_plan_create(
        ctx.handle, _CODE[case["dtype"]], _PRECISION[case["precision"]], nat.ROW_MAJOR,
        len(a), nat.i32([ids[x] for x in a]), nat.i64(ea),
        len(b), nat.i32([ids[x] for x in b]), nat.i64(eb),
        len(c), nat.i32([ids[x] for x in c]), ctypes.byref(plan)))
    nat.check(lib.jet_hip_plan_workspace_size(plan, ctypes.byref(size)))
    out = torch.empty([dims[x] for x in c], dtype=_TORCH[case["dtype"]], device="cuda")
    return {"pair": None, "plan": plan, "a": da, "b": db, "out": out, "bytes": size.value,
            "workspace": torch.empty(max(size.value, 1), dtype=torch.uint8, device="cuda")}


def _run_pair(s):
    if s["pair"]:
        c = jet_amd.contract_tensors(*s["pair"])
        return c.get_data().reshape(c.shape)
    nat.check(nat.lib().jet_hip_contract(
        s["plan"], s["a"].data_ptr(), s["b"].data_ptr(), s["out"].data_ptr(),
        s["workspace"].data_ptr(), s["bytes"], None))
    return s["out"]


def _prepare_transpose(case, seed):
    shape, perm = _transpose_layout(case)
    out = torch.empty([shape[p] for p in perm], dtype=_TORCH[case["dtype"]], device="cuda")
    return {"in": _randn(shape, case["dtype"], seed), "out": out, "code": _CODE[case["dtype"]],
            "modes": nat.i32(range(len(shape))), "shape": nat.i64(shape), "rank": len(shape),
            "order": nat.i32(perm)}


def _run_transpose(s):
    nat.check(nat.lib().jet_hip_permute(
        nat.default_context().handle, s["code"], nat.ROW_MAJOR, s["rank"], s["modes"], s["shape"],
        s["order"], s["in"].data_ptr(), s["out"].data_ptr(), None))
    return s["out"]


def _prepare_task(case, seed):
    net = _task_network(case, seed)
    tn = jet_amd.TensorNetwork(jet_amd.Tensor)
    for ix, sh, d, tags in zip(net.indices, net.shapes, net.data, net.tags):
        tn.add_tensor(jet_amd.Tensor(ix, sh, d.astype(np.complex64), dtype=np.complex64), tags)
    dims = {x: 2 for ix in net.indices for x in ix}
    path = paths.best_greedy_path(net.indices, dims, trials=4, seed=0)
    return {"network": tn, "info": jet_amd.PathInfo(tn, path)}


def _run_task(s):
    tbc = jet_amd.TaskBasedContractor(dtype=np.complex64)
    tbc.add_contraction_tasks(s["network"], s["info"])
    tbc.contract()
    return tbc.results[0].get_data()


def _prepare_amplitudes(case, seed):
    circ, bits, path = _amplitude_problem(case, seed)
    return {"batch": UnevenBatch([AmplitudeJob(circ, bits, path, form=case["form"])],
                                 precision=case["precision"])}


def _run_amplitudes(s):
    s["batch"].launch()
    return s["batch"].amplitudes(0)


def _prepare_sliced(case, seed):
    plan = _sliced_plan()
    net = circuits.amplitude_network(circuits.random_grid_circuit(7, 7, 14, seed=seed))
    batch = plan["sliced"][len(plan["sliced"]) - case["batch"]:]
    return {"slices": SlicedContraction(net.indices, net.shapes, net.data,
                                        [tuple(p) for p in plan["path"]], plan["sliced"],
                                        batch=batch, precision=case["precision"])}


def _run_sliced(s):
    sc = s["slices"]
    sc.run([0])
    return {"slices": sc.slice_results(sc.n_batch),
            "sum": np.complex64(sc.reduce(sc.n_batch))}


def _prepare_gradient(case, seed):
    circ, path = _gradient_problem(case, seed)
    problem = ParameterizedAmplitude(circ, path)
    return {"problem": problem, "angles": problem.theta.copy()}


def _run_gradient(s):
    loss, grad = s["problem"].loss_and_gradient(s["angles"])
    # computed in complex64
    return {"loss": np.float32(loss), "gradient": grad.astype(np.float32)}


_PREPARE = {"pair": _prepare_pair, "transpose": _prepare_transpose, "task": _prepare_task,
            "amplitudes": _prepare_amplitudes, "sliced": _prepare_sliced,
            "gradient": _prepare_gradient}
_RUN = {"pair": _run_pair, "transpose": _run_transpose, "task": _run_task,
        "amplitudes": _run_amplitudes, "sliced": _run_sliced, "gradient": _run_gradient}


# ---------------------------------------------------------------------------
# What a pass cannot do without.
# ---------------------------------------------------------------------------
def work(case):
    kind = case["kind"]
    if kind == "pair":
        m, n, k = (_size(_modes(case[g])) for g in ("left", "right", "common"))
        return {"bytes": np.dtype(case["dtype"]).itemsize * float(m * k + n * k + m * n),
                "flops": 8.0 * m * n * k}
    if kind == "transpose":
        return {"bytes": 2.0 * np.dtype(case["dtype"]).itemsize * _size(_modes(case["modes"])),
                "flops": 0.0}
    if kind == "task":
        net = _task_network(case, 0)
        dims = {x: 2 for ix in net.indices for x in ix}
        path = paths.best_greedy_path(net.indices, dims, trials=4, seed=0)
        return _path_work(net.indices, path)
    if kind == "amplitudes":
        circ, bits, path = _amplitude_problem(case, 0)
        one = _path_work(circuits.amplitude_network(circ).indices, path)
        return {"bytes": one["bytes"], "flops": one["flops"] * case["count"]}
    if kind == "sliced":
        plan = _sliced_plan()
        net = circuits.amplitude_network(circuits.random_grid_circuit(7, 7, 14, seed=0))
        batch = set(plan["sliced"][len(plan["sliced"]) - case["batch"]:])
        loop = set(plan["sliced"]) - batch
        return _path_work([[x for x in ix if x not in loop] for ix in net.indices],
                          plan["path"], batch)
    circ, path = _gradient_problem(case, 0)
    one = _path_work(circuits.amplitude_network(circ).indices, path)
    return {"bytes": one["bytes"], "flops": 3.0 * one["flops"]}


def _path_work(indices, path, keep=frozenset()):
    """Flops of the contractions of a path (every extent 2) and the bytes of
    its leaves; labels in `keep` are never summed."""
    tensors = [frozenset(ix) for ix in indices]
    held = {}
    for t in tensors:
        for x in t:
            held[x] = held.get(x, 0) + 1
    flops = 0.0
    for i, j in path:
        a, b = tensors[i], tensors[j]
        flops += 8.0 * 2.0 ** len(a | b)
        out = set(a | b)
        for x in a & b:
            held[x] -= 1
            if held[x] == 1 and x not in keep:
                out.discard(x)
        tensors.append(frozenset(out))
    return {"bytes": 8.0 * sum(2 ** len(ix) for ix in indices), "flops": flops}


# ---------------------------------------------------------------------------
# The same results in 64 bits, from torch and numpy alone.
# ---------------------------------------------------------------------------
def _gathered(data, labels, dims, order):
    """data (modes `labels`, row-major) in complex128 with modes `order`."""
    n = data.numel()
    stride, size = {}, 1
    for x in reversed(labels):
        stride[x] = size
        size *= dims[x]
    out = torch.empty(n, dtype=torch.complex128, device=data.device)
    for first in range(0, n, 1 << 26):
        left = torch.arange(first, min(n, first + (1 << 26)), device=data.device)
        source = torch.zeros_like(left)
        for x in reversed(order):
            source += (left % dims[x]) * stride[x]
            left = left // dims[x]
        out[first:first + source.numel()] = data[source]
    return out


def _product(a, b):
    """a @ b.T in complex128; long sums in pieces that are summed after."""
    k = a.shape[1]
    if k <= 1 << 16:
        return a @ b.T.contiguous()
    out = torch.zeros(a.shape[0], b.shape[0], dtype=a.dtype, device=a.device)
    for i in range(0, k, 1 << 16):
        out += a[:, i:i + (1 << 16)] @ b[:, i:i + (1 << 16)].T.contiguous()
    return out


def _contract64(indices, data, path):
    """Every node's (labels, complex128 array) along an SSA path."""
    nodes = [(list(ix), np.asarray(d, np.complex128).reshape([2] * len(ix)))
             for ix, d in zip(indices, data)]
    for i, j in path:
        nodes.append(_pairwise64(nodes[i], nodes[j]))
    return nodes


def _pairwise64(x, y):
    (la, a), (lb, b) = x, y
    both = [l for l in la if l in lb]
    out = np.tensordot(a, b, axes=([la.index(l) for l in both], [lb.index(l) for l in both]))
    return [l for l in la if l not in both] + [l for l in lb if l not in both], out


def exact(case, seed):
    kind = case["kind"]
    if kind == "pair":
        a, b, c, dims = _pair_layout(case)
        da = _randn([dims[x] for x in a], case["dtype"], 2 * seed)
        db = _randn([dims[x] for x in b], case["dtype"], 2 * seed + 1)
        left, right = [x for x in a if x in c], [x for x in b if x in c]
        common = [x for x in a if x not in c]
        k = _size([dims[x] for x in common])
        ma = _gathered(da, a, dims, left + common).reshape(-1, k)
        mb = _gathered(db, b, dims, right + common).reshape(-1, k)
        return _as(_product(ma, mb).reshape([dims[x] for x in c]), case)
    if kind == "transpose":
        shape, perm = _transpose_layout(case)
        dims = dict(enumerate(shape))
        data = _gathered(_randn(shape, case["dtype"], seed), list(dims), dims, perm)
        return data.reshape([shape[p] for p in perm])
    if kind == "task":
        net = _task_network(case, seed)
        dims = {x: 2 for ix in net.indices for x in ix}
        path = paths.best_greedy_path(net.indices, dims, trials=4, seed=0)
        return _contract64(net.indices, net.data, path)[-1][1].reshape(1)
    if kind == "amplitudes":
        circ, bits, path = _amplitude_problem(case, seed)
        if work(case)["flops"] > 1.6e12:
            return None
        out = []
        for b in bits:
            net = circuits.amplitude_network(circ, b)
            out.append(complex(_contract64(net.indices, net.data, path)[-1][1]))
        return np.array(out)
    if kind == "gradient":
        return _gradient64(case, seed)
    return None


def _as(values, case):
    """Results of tensors that are read back are arrays."""
    return values.cpu().numpy() if case["api"] == "tensor" else values


def _gradient64(case, seed):
    circ, path = _gradient_problem(case, seed)
    net = circuits.amplitude_network(circ)
    if _path_work(net.indices, path)["flops"] > 2e10:
        return None
    nodes = _contract64(net.indices, net.data, path)
    env = {len(nodes) - 1: ([], np.ones((), np.complex128))}
    n = len(net.indices)
    for s in range(len(path) - 1, -1, -1):
        e = env.pop(n + s)
        for u, other in (path[s], path[s][::-1]):
            env[u] = _pairwise64(e, nodes[other])
    amplitude = complex(nodes[-1][1])
    angles = max(g.param_index for g in circ.gates if g.param_index is not None) + 2
    grad = np.zeros(angles)
    for gi, g in enumerate(circ.gates):
        if g.param_index is None:
            continue
        leaf = circ.n_qubits + gi
        labels, e = env[leaf]
        e = np.transpose(e, [labels.index(l) for l in net.indices[leaf]]).reshape(4, 4)
        theta, phi = g.params
        d_theta = np.zeros((4, 4), np.complex128)
        d_theta[1, 1] = d_theta[2, 2] = -np.sin(theta)
        d_theta[1, 2] = d_theta[2, 1] = -1j * np.cos(theta)
        for slot, dz in ((0, np.sum(e * d_theta)), (1, -1j * np.exp(-1j * phi) * e[3, 3])):
            grad[g.param_index + slot] = 2 * np.real(np.conj(amplitude) * dz)
    return {"loss": np.float64(abs(amplitude) ** 2), "gradient": grad}
