"""The work that a user of this framework has it do, as cases that can be timed.

Kinds of case, each through the public entry points:

  apply         one k-qubit operator on a 2^n state (pq_contract; the smallest
                through pq_contract_noalloc, the form for serving loops)
  pair          two many-qubit tensors contracted over k shared bonds whose
                orders differ in the two operands (one step of contract_network)
  bonds         two tensors with general bond dimensions (MPS / PEPS sites)
  overlap       two states closed onto each other, up to 2 qubits left open
  permute       a state's axes brought into another order in memory
  wavefunction  a whole full_wavefunction_contraction of a QFT circuit
  plan          a whole compiled contraction plan of a grid circuit: sliced or
                not, one amplitude, open output qubits or a batch of bitstrings
  mps           a whole MPS contraction of a brickwork circuit

Qubits have extent 2; dtype is the element type of the tensors ("c128" is the
plain drop-in method, "c64" the single-precision one).
"""
import ctypes
import functools
import math
import pathlib
import sys

import numpy as np
import torch

sys.path.insert(0, str(pathlib.Path(__file__).resolve().parents[1] / "picoquant.jl_amd"))

import picoquant_hip as P  # noqa: E402
from picoquant_hip import circuits, executor, planner  # noqa: E402

NP = {"c128": np.complex128, "c64": np.complex64}
TORCH = {"c128": torch.complex128, "c64": torch.complex64}
SIZE = {"c128": 16, "c64": 8}


def listed():
    return [
        # the smallest call: a two-qubit gate on a 12-qubit state, where only
        # the launch and the host path count
        {"name": "gate_12q", "kind": "apply", "n": 12, "k": 2, "order": 1, "dtype": "c128", "into": True},
        # one gate of a large single-precision state: memory-bound
        {"name": "gate_25q", "kind": "apply", "n": 25, "k": 2, "order": 2, "dtype": "c64", "into": False},
        # an ordinary step of the plain ComplexF64 driver on a grid circuit
        {"name": "pair_c128", "kind": "pair", "m": 11, "n": 9, "k": 7, "order": 3, "dtype": "c128"},
        # the largest steps of a sweep over a wide grid
        {"name": "pair_c64", "kind": "pair", "m": 13, "n": 11, "k": 9, "order": 4, "dtype": "c64"},
        # PEPS-like sites whose bond dimensions are whatever truncation left
        {"name": "bonds_c128", "kind": "bonds", "a1": 37, "a2": 45, "b1": 21, "b2": 33, "k1": 13, "k2": 27,
         "dtype": "c128"},
        # the last step of a plan that meets in the middle; a fidelity
        {"name": "overlap_23q", "kind": "overlap", "n": 23, "m": 0, "order": 5, "dtype": "c128"},
        # the final permutation to the output qubits' order
        {"name": "permute_24q", "kind": "permute", "n": 24, "order": 6, "dtype": "c64"},
        # the 12-qubit QFT wavefunction, gate by gate through the drivers
        {"name": "qft_12q", "kind": "wavefunction", "n": 12},
        # 64 independent amplitudes of the 5x5 depth-12 circuit in ComplexF64
        {"name": "grid5x5_bits", "kind": "plan", "rows": 5, "cols": 5, "depth": 12, "precision": "uniform",
         "sliced": 0, "cap": 28, "out": "bits", "count": 64},
        # the 6x6 depth-14 circuit: 1024 slices, the last column open
        {"name": "grid6x6", "kind": "plan", "rows": 6, "cols": 6, "depth": 14, "precision": "mixed",
         "sliced": 10, "cap": 28, "out": "column", "count": 0},
        # one 7x7 depth-12 amplitude, 256 slices under a size cap, FP16 split
        {"name": "grid7x7_split", "kind": "plan", "rows": 7, "cols": 7, "depth": 12, "precision": "mixed16",
         "sliced": 8, "cap": 22, "out": "one", "count": 0},
        # an MPS of a 14-qubit brickwork circuit with bonds capped at 32
        {"name": "mps_14q", "kind": "mps", "n": 14, "depth": 12, "cap": 32},
    ]


def draw(rng):
    kind = rng.choice(["apply", "apply", "pair", "pair", "bonds", "bonds", "overlap", "permute", "wavefunction",
                       "plan", "plan", "mps"])
    dtype = rng.choice(["c128", "c64"])
    order = rng.randrange(1 << 20)
    if kind == "apply":
        n = rng.randint(8, 24 if dtype == "c128" else 25)
        return {"kind": kind, "n": n, "k": rng.randint(1, 3), "order": order, "dtype": dtype,
                "into": rng.random() < 0.3}
    if kind == "pair":
        m, n = rng.randint(4, 13), rng.randint(3, 11)
        return {"kind": kind, "m": m, "n": n, "k": rng.randint(2, 9), "order": order, "dtype": dtype}
    if kind == "bonds":
        d = [max(1, round(math.exp(rng.uniform(0.0, math.log(48.0))))) for _ in range(6)]
        return {"kind": kind, "a1": d[0], "a2": d[1], "b1": d[2], "b2": d[3], "k1": d[4], "k2": d[5],
                "dtype": dtype}
    if kind == "overlap":
        return {"kind": kind, "n": rng.randint(10, 23), "m": rng.randint(0, 2), "order": order, "dtype": dtype}
    if kind == "permute":
        return {"kind": kind, "n": rng.randint(10, 24), "order": order, "dtype": dtype}
    if kind == "wavefunction":
        return {"kind": kind, "n": rng.randint(5, 16)}
    if kind == "plan":
        rows, cols = rng.randint(4, 6), rng.randint(4, 6)
        out = rng.choice(["one", "column", "bits"])
        if out == "bits":
            rows, cols = min(rows, 5), min(cols, 5)
        return {"kind": kind, "rows": rows, "cols": cols, "depth": rng.randint(6, 12),
                "precision": rng.choice(["uniform", "mixed", "mixed16"]), "sliced": rng.choice([0, 0, 4, 8]),
                "cap": 28, "out": out, "count": rng.choice([3, 8, 32]) if out == "bits" else 0}
    return {"kind": "mps", "n": rng.randint(6, 14), "depth": rng.randint(4, 12),
            "cap": round(math.exp(rng.uniform(math.log(4.0), math.log(48.0))))}


# ---------------------------------------------------------------- contractions
def _contraction(case):
    """(dims of A, labels of A, dims of B, labels of B) of a pairwise
    contraction: labels > 0 are summed, labels < 0 stay open."""
    kind = case["kind"]
    if kind == "bonds":
        return ([case["a1"], case["k1"], case["a2"], case["k2"]], [-1, 1, -2, 2],
                [case["k2"], case["b1"], case["k1"], case["b2"]], [2, -3, 1, -4])
    rng = np.random.Generator(np.random.PCG64(case["order"]))
    if kind == "apply":
        n, k = case["n"], case["k"]
        qubits = rng.permutation(n)[:k].tolist()
        ia = [-(q + 1) for q in range(n)]
        for j, q in enumerate(qubits):
            ia[q] = j + 1
        return [2] * n, ia, [2] * (2 * k), list(range(1, k + 1)) + [-(n + 1 + j) for j in range(k)]
    if kind == "overlap":
        n, m = case["n"], case["m"]
        k, open_a, open_b = n - m, m, 0
    else:
        k, open_a, open_b = case["k"], case["m"], case["n"]
    ia = list(range(1, k + 1)) + [-(j + 1) for j in range(open_a)]
    ib = list(range(1, k + 1)) + [-(open_a + j + 1) for j in range(open_b)]
    ia, ib = [ia[i] for i in rng.permutation(len(ia))], [ib[i] for i in rng.permutation(len(ib))]
    return [2] * len(ia), ia, [2] * len(ib), ib


def _open_dims(dims_a, ia, dims_b, ib):
    return [d for d, x in zip(dims_a, ia) if x < 0] + [d for d, x in zip(dims_b, ib) if x < 0]


def _perm(case):
    return (np.random.Generator(np.random.PCG64(case["order"])).permutation(case["n"]) + 1).tolist()


def _random(shape, dtype, gen, scale):
    """Normal complex elements, the column-major tensor as its reversed shape."""
    x = torch.randn(*reversed(shape), dtype=TORCH[dtype], device="cuda", generator=gen)
    return x * scale


class _Memory:
    """A contiguous device tensor's memory, for torch.as_tensor: the
    column-major tensor as a torch tensor of the reversed shape."""

    def __init__(self, backend, handle):
        ctx = backend.ctx
        base, off = ctypes.c_void_p(), ctypes.c_int64()
        ctx.check(ctx.lib.pq_tensor_device_ptr(ctx.ptr, handle, ctypes.byref(base), ctypes.byref(off), None))
        dtype = np.dtype(backend.dtype)
        self.backend = backend
        self.__cuda_array_interface__ = {
            "shape": tuple(reversed(ctx.shape(handle))), "strides": None, "typestr": dtype.str,
            "data": (base.value + off.value * dtype.itemsize, False), "version": 3}


def _view(backend, handle):
    return torch.as_tensor(_Memory(backend, handle), device="cuda")


def _device_tensor(backend, data):
    """A framework tensor holding `data` (a torch tensor of the reversed shape)."""
    shape = tuple(reversed(data.shape))
    h = backend.ctx.upload(np.zeros(shape, dtype=backend.dtype, order="F"))
    _view(backend, h).copy_(data)
    return h


def _operands(case, seed):
    """The operands' elements, each as its reversed shape."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    if case["kind"] == "permute":
        return [_random([2] * case["n"], case["dtype"], gen, 2.0 ** (-case["n"] / 2))]
    da, ia, db, ib = _contraction(case)
    kt = math.prod(d for d, x in zip(da, ia) if x > 0)
    return [_random(da, case["dtype"], gen, 1.0), _random(db, case["dtype"], gen, kt ** -0.5)]


# --------------------------------------------------------------------- circuits
def _basis_input(n, seed):
    rng = np.random.Generator(np.random.PCG64(seed))
    return "".join("01+-"[i] for i in rng.integers(0, 4, n))


def _brickwork(n, depth, seed):
    """Random two-qubit unitaries on neighbours, even and odd pairs in turn."""
    rng = np.random.Generator(np.random.PCG64(seed))
    gates = []
    for layer in range(depth):
        for q in range(layer % 2, n - 1, 2):
            z = rng.standard_normal((4, 4)) + 1j * rng.standard_normal((4, 4))
            u, r = np.linalg.qr(z)
            gates.append((u * (np.diag(r) / np.abs(np.diag(r))), [q, q + 1]))
    return gates


def _bitstrings(case, seed):
    """Output configurations: 'x' leaves a qubit open."""
    n = case["rows"] * case["cols"]
    rng = np.random.Generator(np.random.PCG64(seed + 1))
    rows = rng.integers(0, 2, (max(1, case["count"]), n))
    out = ["".join(str(b) for b in r) for r in rows]
    if case["out"] == "column":
        out = ["".join("x" if q % case["cols"] == case["cols"] - 1 else c for q, c in enumerate(out[0]))]
    return out


def _grid_network(case, seed, backend):
    n = case["rows"] * case["cols"]
    gates = circuits.grid_circuit_gates(case["rows"], case["cols"], case["depth"], seed)
    tn = P.network_from_gates(n, gates, backend=backend, decompose=True)
    P.add_input(tn, "0" * n)
    P.add_output(tn, _bitstrings(case, seed)[0])
    return tn


class _NoData:
    """A backend for planning: the network's structure without its data."""

    def __init__(self):
        self.metrics = P.Metrics()

    def save_tensor_data(self, label, data):
        pass


@functools.lru_cache(maxsize=None)
def _grid_plan(rows, cols, depth, column, sliced, cap):
    """(pair plan, sliced bonds, multiply-adds): the reconfigured column sweep.
    It depends on the circuit's couplers only, so a program plans once and
    runs every circuit of that shape."""
    case = {"rows": rows, "cols": cols, "depth": depth, "out": "column" if column else "one", "count": 1}
    tn = _grid_network(case, 1, _NoData())
    plan = planner.sweep_plan(tn, planner.grid_site_order(rows, cols, "col"))
    plan = planner.reconfigure(tn, plan, windows=(12,))
    if not sliced:
        return plan, [], planner.plan_ledger(tn, plan)["macs"]
    bonds, macs, _ = planner.choose_slices(tn, plan, sliced, max_elems=2 ** cap)
    return plan, bonds, macs


def _plan_of(case):
    return _grid_plan(case["rows"], case["cols"], case["depth"], case["out"] == "column", case["sliced"],
                      case["cap"])


# ------------------------------------------------------------------ the passes
def prepare(case, seed):
    kind = case["kind"]
    state = {"case": case, "result": None}
    if kind in ("wavefunction", "mps", "plan"):
        b = state["backend"] = P.HIPBackend(np.complex128)
        if kind == "wavefunction":
            state["gates"], state["input"] = circuits.qft_gates(case["n"]), _basis_input(case["n"], seed)
        elif kind == "mps":
            state["gates"] = _brickwork(case["n"], case["depth"], seed)
        else:
            tn = _grid_network(case, seed, b)
            plan, bonds, _ = _plan_of(case)
            state["bits"] = _bitstrings(case, seed) if case["out"] == "bits" else None
            state["plan"] = executor.compile_plan(tn, plan, bonds, precision=case["precision"],
                                                  bitstrings=state["bits"])
        return state
    b = state["backend"] = P.HIPBackend(NP[case["dtype"]])
    state["operands"] = [_device_tensor(b, x) for x in _operands(case, seed)]
    if kind == "permute":
        state["perm"] = _perm(case)
    else:
        da, state["ia"], db, state["ib"] = _contraction(case)
        if case.get("into"):
            dims = _open_dims(da, state["ia"], db, state["ib"])
            state["result"] = b.ctx.upload(np.zeros(dims, dtype=b.dtype, order="F"))
            state["view"] = _view(b, state["result"])
    torch.cuda.synchronize()
    return state


def run(state):
    case, b = state["case"], state["backend"]
    kind = case["kind"]
    if kind == "wavefunction":
        tn = P.network_from_gates(case["n"], state["gates"], backend=b)
        P.add_input(tn, state["input"])
        P.full_wavefunction_contraction(tn, "vector")
        return b.load_tensor_data("result")
    if kind == "mps":
        tn = P.network_from_gates(case["n"], state["gates"], backend=b, decompose=True)
        P.add_input(tn, "0" * case["n"])
        nodes = P.contract_mps_tensor_network_circuit(tn, max_rank=case["cap"])
        P.calculate_mps_amplitudes(tn, nodes)
        return b.load_tensor_data("result")
    if kind == "plan":
        out = state["plan"].run(state["bits"])
        # the amplitudes of a mixed-precision plan carry single precision
        return out if case["precision"] == "uniform" else out.astype(np.complex64)
    ctx = b.ctx
    if case.get("into"):
        ctx.contract_into(state["operands"][0], state["ia"], state["operands"][1], state["ib"], state["result"])
        return state["view"]
    if state["result"] is not None:
        ctx.free(state["result"])
    if kind == "permute":
        h = ctx.permute(state["operands"][0], state["perm"])
        state["result"] = ctx.materialize(h)
        ctx.free(h)
    else:
        state["result"] = ctx.contract(state["operands"][0], state["ia"], state["operands"][1], state["ib"])
    return _view(b, state["result"])


# ------------------------------------------------------------------------- work
def _mps_flops(case):
    """Real operations of the site contractions and economy SVDs, with each
    bond at the dimension it can reach."""
    n, cap = case["n"], case["cap"]
    bond, flops = [1] * (n + 1), 0.0
    for layer in range(case["depth"]):
        for q in range(layer % 2, n - 1, 2):
            left, mid, right = bond[q], bond[q + 1], bond[q + 2]
            rows, cols = 2 * left, 2 * right
            flops += 8.0 * 4 * 2 * 2 * mid * (left + right)       # the gate's halves into the two sites
            flops += 8.0 * rows * cols * 4 * mid                  # the sites contracted
            small, large = min(rows, cols), max(rows, cols)
            flops += 4.0 * (6 * large * small ** 2 + 16 * small ** 3)  # economy SVD of a complex matrix
            bond[q + 1] = min(small, 4 * mid, cap)
    for q in range(1, n):
        flops += 8.0 * 2 ** (q + 1) * bond[q] * bond[q + 1]
    return flops


def work(case):
    kind = case["kind"]
    if kind == "permute":
        return {"bytes": 2 * SIZE[case["dtype"]] * 2 ** case["n"], "flops": 0}
    if kind == "wavefunction":
        n = case["n"]
        return {"bytes": 16 * 2 ** n, "flops": 8.0 * 2 ** n * sum(2 ** len(q) for _, q in circuits.qft_gates(n))}
    if kind == "mps":
        return {"bytes": 16 * 2 ** case["n"], "flops": _mps_flops(case)}
    if kind == "plan":
        n = case["rows"] * case["cols"]
        amps = 2 ** case["rows"] if case["out"] == "column" else max(1, case["count"])
        runs = max(1, case["count"]) if case["out"] == "bits" else 1
        gates = circuits.grid_circuit_gates(case["rows"], case["cols"], case["depth"], 1)
        leaves = sum(16 * 4 ** len(q) for _, q in gates) + 2 * 32 * n
        return {"bytes": leaves + 16 * amps, "flops": 8.0 * runs * _plan_of(case)[2]}
    da, ia, db, ib = _contraction(case)
    out = math.prod(_open_dims(da, ia, db, ib))
    kt = math.prod(d for d, x in zip(da, ia) if x > 0)
    return {"bytes": SIZE[case["dtype"]] * (math.prod(da) + math.prod(db) + out), "flops": 8.0 * out * kt}


# ------------------------------------------------------------------------ exact
def _contract64(x, ia, y, ib):
    """The contraction of two column-major tensors in complex128; tensors
    and result as their reversed shapes."""
    x, y = x.cpu().numpy().T.astype(np.complex128), y.cpu().numpy().T.astype(np.complex128)
    summed = sorted(i for i in ia if i > 0)
    a_open, b_open = [i for i, v in enumerate(ia) if v < 0], [i for i, v in enumerate(ib) if v < 0]
    a = x.transpose(a_open + [ia.index(s) for s in summed])
    b = y.transpose([ib.index(s) for s in summed] + b_open)
    dims = [x.shape[i] for i in a_open] + [y.shape[i] for i in b_open]
    k = math.prod(x.shape[ia.index(s)] for s in summed)
    a, b = a.reshape((-1, k), order="F"), b.reshape((k, -1), order="F")
    at = torch.from_numpy(np.ascontiguousarray(a.T)).cuda()
    bt = torch.from_numpy(np.ascontiguousarray(b.T)).cuda()
    return (bt @ at).reshape(list(reversed(dims)))


def _state_vector(n, gates, config):
    """The circuit's state, axis q = qubit q, in complex128."""
    vecs = {"0": [1, 0], "1": [0, 1], "+": [0.5 ** 0.5, 0.5 ** 0.5], "-": [0.5 ** 0.5, -(0.5 ** 0.5)]}
    psi = torch.ones((), dtype=torch.complex128, device="cuda")
    for c in config:
        psi = psi.unsqueeze(-1) * torch.tensor(vecs[c], dtype=torch.complex128, device="cuda")
    for u, qs in gates:
        k = len(qs)
        # the first qubit of a gate is its least significant bit
        g = torch.from_numpy(np.ascontiguousarray(u)).to("cuda", torch.complex128)
        order = list(reversed(qs))
        rest = [q for q in range(n) if q not in order]
        flat = psi.permute(*order, *rest).reshape(2 ** k, -1)
        flat = (g @ flat).reshape([2] * n)
        back = [0] * n
        for i, q in enumerate(order + rest):
            back[q] = i
        psi = flat.permute(*back)
    return psi


def exact(case, seed):
    kind = case["kind"]
    if kind == "permute":
        (x,) = _operands(case, seed)
        x = x.cpu().numpy().T.transpose([p - 1 for p in _perm(case)])
        return np.ascontiguousarray(x.T.astype(np.complex128))
    if kind == "wavefunction":
        psi = _state_vector(case["n"], circuits.qft_gates(case["n"]), _basis_input(case["n"], seed))
        return np.ravel(psi.cpu().numpy(), order="F")
    if kind == "mps":
        n = case["n"]
        if case["cap"] < 2 ** (n // 2):
            return None       # a truncated state has no value but the method's own
        psi = _state_vector(n, _brickwork(n, case["depth"], seed), "0" * n)
        return np.ravel(psi.cpu().numpy(), order="F")
    if kind == "plan":
        n = case["rows"] * case["cols"]
        if n > 25:
            return None       # no state vector of this many qubits
        gates = circuits.grid_circuit_gates(case["rows"], case["cols"], case["depth"], seed)
        psi = _state_vector(n, gates, "0" * n)
        amps = [psi[tuple(slice(None) if c == "x" else int(c) for c in bits)] for bits in _bitstrings(case, seed)]
        return (torch.stack(amps) if case["out"] == "bits" else amps[0]).cpu().numpy()
    _, ia, _, ib = _contraction(case)
    x, y = _operands(case, seed)
    return _contract64(x, ia, y, ib)
