"""Batches of independent output bitstrings in one planned run
(compile_plan(bitstrings=...), pq_plan_desc.n_out_bits): every closed output
qubit's leaf holds one column per bitstring, the batch bonds lie above the
slice group, and the FP64 sum keeps one result per bitstring.

  * config 2 (5x5 depth 12): the 8 committed brute-force amplitudes, sliced
    and replayed as a graph, ComplexF64 ........................... 1e-12
    and the bench's precision split ................................ 1e-5
  * Plan.set_bitstrings rewrites the batch in place: the same compiled
    plan and captured graph give the new bitstrings' amplitudes
  * a batch of 5 (padded to 8) with open qubits, against the brute-force
    state vector ................................................... 1e-12
  * fused chains that run once per bitstring (tensors depending on the
    batch bonds only) against the state vector, complex64 ............ 2e-6
"""
import json

import numpy as np
import pytest

from oracle import pq_oracle as O
import picoquant_hip as P
from picoquant_hip import _lib, circuits as C, planner as PL
from picoquant_hip.executor import closed_output_qubits, compile_plan

pytestmark = pytest.mark.gpu


def _net(rows, cols, depth, seed, cfg, dtype=np.complex128):
    n = rows * cols
    tn = P.network_from_gates(n, C.grid_circuit_gates(rows, cols, depth, seed),
                              backend=P.HIPBackend(dtype), decompose=True)
    P.add_input(tn, "0" * n)
    P.add_output(tn, cfg)
    return tn


def _amp(sv, bits):
    return sv[sum(int(b) << q for q, b in enumerate(bits))]


def _rel(got, want):
    got, want = np.asarray(got).reshape(-1), np.asarray(want).reshape(-1)
    return float(np.max(np.abs(got - want) / np.abs(want)))


@pytest.mark.parametrize("precision,tol", [("uniform", 1e-12), ("mixed", 1e-5)])
def test_grid5x5_committed_bitstrings(golden_dir, precision, tol):
    g = json.load(open(golden_dir / "grid5x5_d12.json"))
    bits = g["bitstrings"]
    want = np.array([complex(a, b) for a, b in g["amplitudes"]])
    tn = _net(5, 5, 12, g["seed"], bits[0])
    plan = PL.sweep_plan(tn, PL.grid_site_order(5, 5, "col"))
    sliced = PL.choose_slices(tn, plan, 4)[0]
    p = compile_plan(tn, plan, sliced, group_bits=2, precision=precision, bitstrings=bits)
    assert p.n_out_bits == 3
    for use_graph in (False, True, True):
        p.execute(use_graph)
        got = p.result()
        assert got.shape == (8,)
        assert _rel(got, want) < tol
    # a new batch without recompiling: the captured graph reads the rewritten leaves
    order = [5, 2, 7, 0, 1, 6, 3, 4]
    p.set_bitstrings([bits[i] for i in order])
    for _ in range(2):
        p.execute(True)
        assert _rel(p.result(), want[order]) < tol
    with pytest.raises(ValueError):
        p.set_bitstrings(bits[:3])
    p.close()


def test_plan_run_and_cost_through_the_c_abi(golden_dir):
    """pq_plan_run with raw 64-bit bitstring words (the boundary's one-call
    batched path: set the batch, replay, FP64 result) gives the committed
    config-2 amplitudes, also for a batch shorter than the compiled one
    (padded on the device); pq_plan_cost counts the plan's exact MACs."""
    import ctypes as ct
    g = json.load(open(golden_dir / "grid5x5_d12.json"))
    bits = g["bitstrings"]
    want = np.array([complex(a, b) for a, b in g["amplitudes"]])
    tn = _net(5, 5, 12, g["seed"], bits[0])
    plan = PL.sweep_plan(tn, PL.grid_site_order(5, 5, "col"))
    sliced = PL.choose_slices(tn, plan, 4)[0]
    p = compile_plan(tn, plan, sliced, group_bits=2, precision="uniform", bitstrings=bits)
    ctx, lib = p.ctx, p.ctx.lib
    words = (ct.c_uint64 * 8)(*[sum(int(c) << i for i, c in enumerate(b)) for b in bits])
    n_out = int(np.prod(p.out_shape)) if p.out_shape else 1
    assert n_out == 1
    out = np.empty(2 * 8, dtype=np.float64)
    order = [3, 1, 4, 1, 5, 0, 2, 6]
    for sel in (list(range(8)), order):
        w = (ct.c_uint64 * 8)(*[words[i] for i in sel])
        ctx.check(lib.pq_plan_run(ctx.ptr, p.ptr, 8, w, out.ctypes.data_as(ct.POINTER(ct.c_double))))
        assert _rel(out[0::2] + 1j * out[1::2], want[sel]) < 1e-12
    # three bitstrings: the other five results repeat the first
    w = (ct.c_uint64 * 3)(words[6], words[2], words[5])
    ctx.check(lib.pq_plan_run(ctx.ptr, p.ptr, 3, w, out.ctypes.data_as(ct.POINTER(ct.c_double))))
    assert _rel(out[0::2] + 1j * out[1::2], want[[6, 2, 5, 6, 6, 6, 6, 6]]) < 1e-12
    # a bad count is an error, not a run
    w9 = (ct.c_uint64 * 9)()
    assert lib.pq_plan_run(ctx.ptr, p.ptr, 9, w9, None) != 0
    # cost: the steps' MACs, every step's MACs per slice times the slices it runs for
    c = p.cost()
    assert c["steps"] == len(p.steps) and c["macs"] == pytest.approx(float(np.sum(c["step_macs"])))
    assert c["macs"] == pytest.approx(p.stats()["alg_flops"] / 8, rel=1e-12)
    assert c["launches"] == p.stats()["launches"]
    p.close()


def test_bitstring_batch_with_open_qubits():
    """Five bitstrings (padded to 8 on the device) over a 3x3 grid whose
    qubits 2, 4 and 7 stay open: 5 x 8 amplitudes."""
    cfg = "1x0x11x01"
    sv = O.statevector(9, O.grid_circuit_gates(3, 3, 6, 21))
    rng = np.random.default_rng(4)
    batch = []
    for _ in range(5):
        b = "".join(str(int(v)) for v in rng.integers(0, 2, 9))
        batch.append("".join("x" if c == "x" else b[i] for i, c in enumerate(cfg)))
    tn = _net(3, 3, 6, 21, batch[0])
    open_q = [i + 1 for i, ch in enumerate(cfg) if ch == "x"]
    plan = PL.sweep_plan(tn, PL.grid_site_order(3, 3, open_last=open_q))
    sliced = PL.choose_slices(tn, plan, 2)[0]
    p = compile_plan(tn, plan, sliced, group_bits=1, bitstrings=batch)
    p.execute(True)
    got = p.result()
    assert got.shape == (5, 2, 2, 2)
    for b, bitsb in enumerate(batch):
        for j in range(8):
            full = list(bitsb)
            for t, q in enumerate(open_q):
                full[q - 1] = str((j >> t) & 1)
            want = _amp(sv, full)
            g = got[b].reshape(-1, order="F")[j]
            assert abs(g - want) <= 1e-12 * abs(want)
    p.close()


def test_fused_chains_run_once_per_bitstring():
    cfg0 = "0110" + "x" * 4 + "1001" + "01" + "x" * 2
    sv = O.statevector(16, O.grid_circuit_gates(4, 4, 8, 7))
    rng = np.random.default_rng(9)
    batch = ["".join("x" if c == "x" else str(int(rng.integers(0, 2))) for c in cfg0) for _ in range(4)]
    tn = _net(4, 4, 8, 7, batch[0])
    plan = PL.reconfigure(tn, PL.sweep_plan(tn, PL.grid_site_order(4, 4, "col")), windows=(8,))
    p = compile_plan(tn, plan, precision="mixed", small_elems=16, bitstrings=batch,
                     fuse={"tile_bits": 10, "min_elems": 64, "op_elems": 256})
    chains = [i for i, st in enumerate(p.steps) if st[0] == 2]
    assert chains and any(p.step_info(i)["dep"] for i in chains)
    ctx = tn.backend.ctx
    ctx.profile_enable(True)
    p.execute(False)
    launches = ctx.profile_read(_lib.KC_CHAIN)["launches"]
    ctx.profile_enable(False)
    # a chain that depends on the batch bonds launches once per bitstring
    assert launches == sum(4 if p.step_info(i)["dep"] else 1 for i in chains)
    p.execute(True)
    p.execute(True)
    got = p.result()
    open_q = [i for i, ch in enumerate(cfg0) if ch == "x"]
    for b, bits in enumerate(batch):
        want = []
        for j in range(2 ** len(open_q)):
            full = list(bits)
            for t, q in enumerate(open_q):
                full[q] = str((j >> t) & 1)
            want.append(_amp(sv, full))
        want = np.array(want)
        g = got[b].reshape(-1, order="F")
        assert np.linalg.norm(g - want) / np.linalg.norm(want) < 2e-6
    p.close()


def test_bad_bitstring_batches_are_rejected():
    tn = _net(2, 2, 3, 1, "0110")
    plan = PL.sweep_plan(tn, PL.grid_site_order(2, 2))
    with pytest.raises(ValueError):
        compile_plan(tn, plan, bitstrings=["01x0"])          # an open character at a closed qubit
    with pytest.raises(ValueError):
        compile_plan(tn, plan, bitstrings=["011"])           # too short
    with pytest.raises(ValueError):
        compile_plan(tn, plan, bitstrings=[])


@pytest.mark.parametrize("n_sliced,group_bits,precision,count", [
    (0, 0, "uniform", 1), (0, 0, "uniform", 2), (0, 0, "uniform", 37), (3, 3, "uniform", 5), (3, 3, "mixed", 16),
    (8, 8, "uniform", 32), (3, 1, "uniform", 5)])
def test_bitstring_batch_inside_the_slice_group(n_sliced, group_bits, precision, count):
    """Every slice in one group: the batch's bitstrings join it as more copies
    (13 bits with 8 slices' bonds and 32 bitstrings, one more than a group
    holds, so two groups run); with slice groups left over (the last case)
    they stay one group each.  Replays with rewritten batches, padded counts
    and an open qubit, against brute force; FP64 as the plan executor's other
    tests, mixed precision at its 1e-5."""
    n = 12
    sv = O.statevector(n, O.grid_circuit_gates(3, 4, 8, 5))
    rng = np.random.default_rng(count + n_sliced)
    batches = [["".join("x" if i == 7 else str(int(v)) for i, v in enumerate(rng.integers(0, 2, n)))
                for _ in range(count)] for _ in range(2)]
    tn = _net(3, 4, 8, 5, batches[0][0])
    plan = PL.sweep_plan(tn, PL.grid_site_order(3, 4, open_last=[8]))
    sliced = PL.choose_slices(tn, plan, n_sliced)[0]
    p = compile_plan(tn, plan, sliced, group_bits=group_bits, precision=precision, bitstrings=batches[0])
    for batch in batches + batches[:1]:
        got = p.run(batch)
        assert got.shape == (count, 2)
        want = np.array([[_amp(sv, list(b.replace("x", v))) for v in "01"] for b in batch])
        assert np.max(np.abs(got - want)) <= (1e-12 if precision == "uniform" else 1e-5) * np.max(np.abs(want))
    p.close()


def test_bitstring_batch_keeps_to_the_budget():
    """budget_bytes bounds the plan's memory with bitstrings inside the slice
    group: less of it, fewer join, down to one group per bitstring; any
    number that compile_plan took before is taken (0, floats, infinity)."""
    n, count = 12, 32
    sv = O.statevector(n, O.grid_circuit_gates(3, 4, 8, 5))
    rng = np.random.default_rng(2)
    batch = ["".join(str(int(v)) for v in rng.integers(0, 2, n)) for _ in range(count)]
    want = np.array([_amp(sv, list(b)) for b in batch])
    tn = _net(3, 4, 8, 5, batch[0])
    plan = PL.sweep_plan(tn, PL.grid_site_order(3, 4))

    def run(**kw):
        p = compile_plan(tn, plan, bitstrings=batch, **kw)
        st = p.stats()
        assert np.max(np.abs(p.run(batch) - want)) <= 1e-12 * np.max(np.abs(want))
        p.close()
        return st["arena_bytes"], st["launches"]

    full, one = run(), run(budget_bytes=0)
    assert run(budget_bytes=float("inf")) == full
    assert full[0] > one[0] and full[1] < one[1]
    last = full
    for budget in (full[0] - 1, (full[0] + one[0]) / 2, one[0]):
        got = run(budget_bytes=budget)
        assert got[0] <= budget and got[1] >= last[1] and got != full
        last = got
    assert run(budget_bytes=one[0] - 1) == one


def test_rewritten_bitstrings_are_there_for_other_streams():
    """pq_tensor_device_ptr of an output column, taken after set_bitstrings
    behind 10 ms of queued work, is safe to read from another stream."""
    import ctypes as ct
    n = 4
    rng = np.random.default_rng(3)
    batches = [["".join(str(int(v)) for v in rng.integers(0, 2, n)) for _ in range(8)] for _ in range(2)]
    tn = _net(2, 2, 3, 5, batches[0][0])
    p = compile_plan(tn, PL.sweep_plan(tn, PL.grid_site_order(2, 2)), bitstrings=batches[0])
    ctx, hip = p.ctx, p.ctx.lib                            # the HIP runtime, through the library that links it
    stream = ct.c_void_p()
    assert hip.hipStreamCreateWithFlags(ct.byref(stream), ct.c_uint(1)) == 0        # does not wait for others
    cols = {}

    def read(where):
        for qubit, src in where.items():
            out = np.empty((8, 2), np.complex128)
            assert hip.hipMemcpyAsync(ct.c_void_p(out.ctypes.data), ct.c_void_p(src), ct.c_size_t(out.nbytes),
                                      ct.c_int(2), stream) == 0
            assert hip.hipStreamSynchronize(stream) == 0
            cols[qubit] = out

    def pointers():
        base, off, where = ct.c_void_p(), ct.c_int64(), {}
        for node, qubit in closed_output_qubits(tn):
            ctx.check(hip.pq_tensor_device_ptr(ctx.ptr, p.batch_handles[node], ct.byref(base), ct.byref(off), None))
            where[qubit] = base.value + 16 * off.value
        return where

    read(pointers())                                       # the copies' own first use
    big = ctx.upload(np.ones((4096, 4096), np.complex128))
    first = ctx.contract(big, [-1, 1], big, [1, -2])       # memory and kernels are there
    ctx.synchronize()
    ctx.free(first)
    busy = ctx.contract(big, [-1, 1], big, [1, -2])
    p.set_bitstrings(batches[1])
    read(pointers())
    for qubit, col in cols.items():
        assert np.array_equal(col, [[1 - int(b[qubit]), int(b[qubit])] for b in batches[1]])
    ctx.synchronize()
    hip.hipStreamDestroy(stream)
    ctx.free(busy)
    ctx.free(big)
    p.close()
