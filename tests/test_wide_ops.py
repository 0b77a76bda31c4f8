"""Ops on more qubits than a block or a pass holds: the planners let them
through in order, and circuits with them run in every mode."""
import numpy as np
import pytest

from helpers import rand_unitary
from oracle import statevector as O
from test_compiler import _sim_ops
from test_passes import _replay


def _circuit(n, widths, seed):
    """Layers of ry and CX with an X of w controls after each, w in widths."""
    from blackwell_backend.circuit import QuantumCircuit
    rng = np.random.default_rng(seed)
    qc = QuantumCircuit(n)
    for w in widths:
        for q in range(n):
            qc.ry(float(rng.uniform(0, 6)), q)
        for q in range(0, n - 1, 2):
            qc.cx(q, q + 1)
        s = [int(x) for x in rng.choice(n, w + 1, replace=False)]
        qc.mcx(s[:w], s[w])
    return qc


@pytest.mark.parametrize("n,widths", [(14, (8,)), (14, (10, 7, 4, 8)), (13, (9, 3, 10))])
def test_planners_let_wide_ops_through(n, widths):
    from blackwell_backend import compiler as C
    from blackwell_backend.circuit import instructions
    ops = C.compile_ops(instructions(_circuit(n, widths, n)))
    ref = _sim_ops(n, ops)
    psi = O.zero_state(n)
    passed = []
    for e in C.plan_passes(ops, n, 11, 4):
        if isinstance(e, C.PassRun):
            psi = _replay(psi, n, e)
        else:
            passed.append(len(e.all_qubits))
            psi = O.apply_matrix(psi, e.full_matrix(), list(e.all_qubits))
    assert passed == [w + 1 for w in widths if w > 3]
    # coefficients are within 2^-26, 32 products to a row, over at most one block per op
    assert np.max(np.abs(psi - ref)) < len(ops) * 32 * 2.0 ** -26
    for k in (4, 5, 6):
        psi = O.zero_state(n)
        for e in C.plan_blocks(ops, n, k=k):
            block = isinstance(e, C.Block)
            assert block or len(e.all_qubits) > k
            psi = O.apply_matrix(psi, e.mat if block else e.full_matrix(), list(e.qubits if block else e.all_qubits))
        # FP64 products of at most 32 x 32 matrices
        assert np.max(np.abs(psi - ref)) < len(ops) * 64 * 2.0 ** -52


def _apply(psi, n, op):
    """O.apply_matrix, but X with many controls as the permutation it is."""
    if op.kind != "x" or len(op.controls) < 6:
        return O.apply_matrix(psi, op.full_matrix(), list(op.all_qubits))
    i = np.arange(1 << n)
    on = np.all([(i >> c) & 1 for c in op.controls], axis=0)
    return psi[np.where(on, i ^ (1 << op.qubits[0]), i)]


@pytest.mark.gpu
@pytest.mark.parametrize("n,widths", [(12, (8, 11)), (14, (8, 12, 4)), (18, (9, 12, 6))])
def test_wide_ops_run_between_blocks_and_passes(dev, n, widths):
    """Up to 12 controls, past the seven that the plain kernel takes, on qubits
    with and without the low ones."""
    from blackwell_backend import BlackwellSimulator, compiler as C
    from blackwell_backend.circuit import instructions
    from blackwell_kernels._lib import QsimError
    sim = BlackwellSimulator(dev)
    qc = _circuit(n, widths, n)
    ref = O.zero_state(n)
    for op in C.compile_ops(instructions(qc)):
        ref = _apply(ref, n, op)
    for mode in ("auto", "passes", "blocks"):
        got, _ = sim.run_statevector(qc, mode=mode)
        # FP32 rounding of at most a few ulp per gate, over fewer than 100 gates
        assert np.linalg.norm(got - ref) <= 100 * 4 * 2.0 ** -24, mode
    with pytest.raises(QsimError, match="controls must have 0-7 elements"):
        sim.run_statevector(qc, mode="plain")


def test_tile_plans_let_dense_ops_of_six_qubits_through():
    """An LDS program runs dense ops of at most five qubits; it used to leave
    larger ones out without an error."""
    from blackwell_backend import compiler as C
    from blackwell_backend.executor import tile_ops
    ops = [C.Op("m1", [3], rand_unitary(2, 0)), C.Op("mk", [0, 2, 3, 5, 6, 8], rand_unitary(64, 1)),
           C.Op("mk", [0, 2, 4, 5, 7], rand_unitary(32, 2))]
    plan = C.plan_tiles(ops, 9, m=9)
    assert [isinstance(e, C.TilePass) for e in plan] == [True, False, True] and plan[1] is ops[1]
    assert [o for e in plan if isinstance(e, C.TilePass) for o in e.ops] == [ops[0], ops[2]]
    with pytest.raises(ValueError, match="dense op of 6 qubits"):
        tile_ops(ops, 0x1ff)


@pytest.mark.gpu
def test_dense_ops_of_six_qubits_run_or_are_refused(dev):
    from blackwell_backend import BlackwellSimulator, compiler as C
    from blackwell_backend.circuit import QuantumCircuit, instructions
    sim = BlackwellSimulator(dev)
    u = rand_unitary(64, 5)

    def circuit(n):
        qc = QuantumCircuit(n)
        for q in range(n):
            qc.ry(0.3 + q, q)
        return qc.unitary(u, [0, 3, 4, 6, 7, n - 1]).cx(0, n - 1)
    qc = circuit(14)
    ref = _sim_ops(14, C.compile_ops(instructions(qc)))
    for mode in ("auto", "passes", "blocks", "tiles", "plain"):
        got, _ = sim.run_statevector(qc, mode=mode)
        # 64-term FP32 sums in one block, a few ulp per gate elsewhere
        assert np.linalg.norm(got - ref) <= (64 + 4 * 16) * 2.0 ** -24, mode
    for n in (9, 12):
        for mode in ("auto", "whole", "tiles", "plain"):
            with pytest.raises(RuntimeError, match="wider blocks are not supported"):
                sim.run_statevector(circuit(n), mode=mode)
