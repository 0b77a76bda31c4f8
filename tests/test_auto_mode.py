"""What mode "auto" picks for circuits with ops of five qubits, which no block
pass holds, and that the plans it picks from give the same state."""
import ctypes

import numpy as np
import pytest

from helpers import rand_unitary
from oracle import statevector as O
from test_compiler import _sim_ops


def _circuits(n):
    """name -> (circuit, the plan that measured fastest on its family from 22 qubits on)."""
    from blackwell_backend import workloads as W
    from blackwell_backend.circuit import QuantumCircuit
    rng = np.random.default_rng(n)
    pick = lambda k, of=n: [int(q) for q in rng.choice(of, k, replace=False)]
    layers = QuantumCircuit(n)            # ry and four X of four controls
    for _ in range(4):
        for q in range(n):
            layers.ry(float(rng.uniform(0, 6)), q)
        for _ in range(4):
            s = pick(5)
            layers.mcx(s[:4], s[4])
    dense = QuantumCircuit(n)
    for i in range(12):
        s = pick(5)
        dense.unitary(rand_unitary(32, i), s).ry(0.1 + i, s[0])
    same = QuantumCircuit(n)
    for i in range(30):
        same.mcx([0, 3, 5, n - 2], n - 1).ry(0.1 + i, n - 1)
    oracles = QuantumCircuit(n)           # X of four controls between H, X and CX layers
    for _ in range(5):
        for q in range(n):
            oracles.h(q).x(q)
        for _ in range(3):
            s = pick(5)
            oracles.mcx(s[:4], s[4])
        for q in range(n - 1):
            oracles.cx(q, q + 1)
    few = QuantumCircuit(n)               # SU(4) gates on the same five qubits
    for i in range(60):
        a, b = pick(2, 5)
        few.unitary(rand_unitary(4, i), [(1, 4, 6, n - 3, n - 1)[a], (1, 4, 6, n - 3, n - 1)[b]])
    return {"layers": (layers, "blocks"), "dense": (dense, "blocks"), "same": (same, "blocks"),
            "few": (few, "blocks"), "oracles": (oracles, "passes"), "volume": (W.su4_volume(n, 4, 1), "passes")}


def _compiled(qc):
    from blackwell_backend import compiler as C
    from blackwell_backend.circuit import instructions
    from blackwell_backend.executor import CompiledCircuit
    return CompiledCircuit(qc.num_qubits, 0, C.compile_ops(instructions(qc)))


@pytest.mark.parametrize("n", [22, 25, 28])
def test_auto_weighs_blocks_against_passes(n):
    for name, (qc, mode) in _circuits(n).items():
        assert _compiled(qc).resolve_mode("auto") == mode, name


def test_five_qubit_ops_between_passes_share_blocks():
    from blackwell_backend import compiler as C
    from blackwell_backend.executor import CompiledCircuit
    x = lambda t, *c: C.Op("x", [t], controls=c)
    ops = [C.Op("m2", [0, 1], rand_unitary(4, 0)), x(1, 3, 5, 9, 11), x(9, 3, 5, 1, 11), x(11, 9, 3, 5, 1),
           x(2, 4, 6, 8, 10, 12, 13), C.Op("m2", [2, 1], rand_unitary(4, 1))]
    steps = CompiledCircuit(14, 0, ops)._build("passes", "cpu").steps
    assert [k for k, _ in steps] == ["passes", "blocks", "qsim_apply_mcx", "passes"]
    assert steps[1][1][1] == 1            # one block for the three


def test_block_count():
    from blackwell_backend import compiler as C
    from blackwell_kernels import _lib
    rng = np.random.default_rng(3)
    for n, seed in ((12, 0), (20, 1), (30, 2)):
        ops = [C.Op("m2", rng.choice(n, 2, replace=False), rand_unitary(4, i)) for i in range(120)]
        greedy = sum(isinstance(e, C.Block) for e in C.plan_blocks(ops, n, k=5, effort=0))
        assert 0.7 * greedy <= C.count_blocks(ops, n) <= 1.5 * greedy
    x = lambda *q: C.Op("x", q[:1], controls=q[1:])
    assert C.count_blocks([], 9) == 0
    assert C.count_blocks([x(0, 1, 2, 3, 4, 5)], 9) == 0                       # wider than a block
    assert C.count_blocks([x(0, 1), x(0, 1, 2, 3, 4, 5), x(1, 0)], 9) == 2     # and in the way
    assert C.count_blocks([x(0, 1), x(8, 3, 4, 5, 6, 7), x(1, 0)], 9) == 1
    assert C.count_blocks([x(0, 1), C.Op("measure", [0]), x(0, 1)], 9) == 2
    lib, out = _lib.load(), ctypes.c_int()

    def call(n=8, k=5, masks=(3,), count=None):
        m = np.array(masks, dtype=np.uint64)
        return lib.qsim_count_blocks(n, k, len(masks) if count is None else count,
                                     ctypes.c_void_p(m.ctypes.data), ctypes.byref(out))
    assert call() == 0 and out.value == 1
    assert call(n=0) == 2 and call(n=35) == 2 and call(k=0) == 2 and call(k=7) == 2
    assert call(masks=(0,)) == 1 and call(masks=(1 << 8,)) == 1 and call(count=-1) == 1
    assert lib.qsim_count_blocks(8, 5, 1, None, ctypes.byref(out)) == 1


@pytest.mark.gpu
@pytest.mark.parametrize("n", [10, 12, 13, 14, 17])
def test_plans_of_five_qubit_ops_match_fp64(dev, n):
    from blackwell_backend import BlackwellSimulator
    sim = BlackwellSimulator(dev)
    picked = set()
    for name, (qc, _) in _circuits(n).items():
        cc = sim.compile(qc)
        ref = _sim_ops(n, cc.ops)
        picked.add(cc.resolve_mode("auto"))
        for mode in ("auto", "passes"):
            got, _ = sim.run_statevector(qc, mode=mode)
            # at most 32 products to an amplitude, a few ulp a gate over at most 440 gates
            assert np.linalg.norm(got - ref) <= len(cc.ops) * 4 * 2.0 ** -24, (name, mode)
    assert picked >= {"blocks", "passes"}


@pytest.mark.gpu
def test_served_circuits_take_the_auto_plan(dev):
    """A circuit of five-qubit ops through the server, run and replayed as a graph."""
    from blackwell_backend import BlackwellSimulator
    from blackwell_backend.serving import Request, Server
    sim = BlackwellSimulator(dev)
    server = Server(sim, graph_repeats=4)
    for name in ("layers", "oracles"):
        qc = _circuits(16)[name][0]
        ref = _sim_ops(16, sim.compile(qc).ops)
        reqs = [Request(i, 0.0, 16, 0, i, circuit=qc, keep_state=True) for i in range(4)]
        server.serve(reqs, realtime=False)
        for r in reqs:
            assert np.linalg.norm(r.state - ref) <= 440 * 4 * 2.0 ** -24, name


@pytest.mark.gpu
def test_tune_times_the_passes_too(dev):
    """An SU(4) volume circuit runs in passes in less than half the time of every
    other mode; five-qubit ops on one set of qubits are one block."""
    from blackwell_backend import BlackwellSimulator, workloads as W
    sim = BlackwellSimulator(dev, mode="tune")
    for qc, want in ((W.su4_volume(18, 12, 3), "passes"), (_circuits(18)["same"][0], "blocks")):
        cc = sim.compile(qc)
        got, _ = sim.run_statevector(qc)
        mode = cc.resolve_mode("tune", sim.device)
        assert mode.startswith(want)
        assert np.linalg.norm(got - _sim_ops(18, cc.ops)) <= len(cc.ops) * 4 * 2.0 ** -24
