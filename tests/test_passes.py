"""Block passes: the planner's passes replayed in FP64 from their packed
records and fragments equal the circuit (CPU), and the kernel equals the FP64
oracle at every tile size, with remainders of waves and tiles (GPU)."""
import ctypes

import numpy as np
import pytest

from helpers import rand_state, rand_unitary
from oracle import statevector as O
from test_compiler import _sim_ops, random_circuit


def _sw(p):
    j = 1 << p
    return j ^ ((j >> 5) & 31) ^ ((j >> 10) & 31)


def _matrix(frag):
    """16 x 16 complex matrix of a block's fragments bf16 [3][2][64][8]."""
    f = (np.asarray(frag).astype(np.uint32) << 16).view(np.float32).astype(np.float64).reshape(3, 2, 64, 8).sum(axis=0)
    a = np.zeros((32, 32))
    for t in range(2):
        for h in range(2):
            for j in range(8):
                amp = 4 * (2 * t + (j >> 2)) + 2 * h + ((j >> 1) & 1)
                a[:, 2 * amp + (j & 1)] = f[t, 32 * h:32 * h + 32, j]
    assert np.array_equal(a[1::2, 1::2], a[0::2, 0::2]) and np.array_equal(a[0::2, 1::2], -a[1::2, 0::2])
    return a[0::2, 0::2] + 1j * a[1::2, 0::2]


def _replay(psi, n, run):
    for p in run.passes:
        tile = [q for q in range(n) if int(p["tile_mask"]) >> q & 1]
        for b in range(int(p["first_block"]), int(p["first_block"] + p["n_blocks"])):
            bits = [int(v).bit_length() - 1 for v in run.blocks["bit"][b][:len(tile)]]
            assert sorted(bits) == list(range(len(tile)))
            assert [int(v) for v in run.blocks["bit"][b][:len(tile)]] == [_sw(x) for x in bits]
            assert not run.blocks["bit"][b][len(tile):].any()
            psi = O.apply_matrix(psi, _matrix(run.frags[b]), [tile[x] for x in bits[:4]])
    return psi


@pytest.mark.parametrize("n,m,low", [(10, 10, 4), (10, 13, 4), (12, 10, 4), (13, 11, 5), (14, 12, 3), (15, 13, 4)])
def test_planned_passes_equal_the_circuit(n, m, low):
    from blackwell_backend import compiler as C
    from blackwell_backend.circuit import instructions
    qc = random_circuit(n, 150, n * 100 + m)
    ops = C.compile_ops(instructions(qc))
    psi, wide = O.zero_state(n), 0
    for e in C.plan_passes(ops, n, m, low):
        if isinstance(e, C.PassRun):
            for p in e.passes:
                assert bin(int(p["tile_mask"])).count("1") == min(m, n)
                assert int(p["tile_mask"]) & ((1 << low) - 1) == (1 << low) - 1
            psi = _replay(psi, n, e)
        else:
            assert len(e.all_qubits) > 4
            wide += 1
            psi = O.apply_matrix(psi, e.full_matrix(), list(e.all_qubits))
    assert wide == sum(len(o.all_qubits) > 4 for o in ops)
    # coefficients are within 2^-26, two parts of 16 to a row, over at most 150 blocks
    assert np.max(np.abs(psi - _sim_ops(n, ops))) < 150 * 32 * 2.0 ** -26


def test_pass_arguments_are_checked():
    from blackwell_kernels import _lib
    lib = _lib.load()
    passes = np.zeros(1, _lib.PASS_DTYPE)
    blocks = np.zeros(1, _lib.PASS_BLOCK_DTYPE)
    blocks["bit"][0, :10] = [_sw(p) for p in range(10)]
    vp = lambda a: ctypes.c_void_p(a.ctypes.data)
    one = ctypes.c_void_p(16)            # never dereferenced: every call below is refused

    def call(n=12, mask=(1 << 10) - 1, first=0, count=1, blk=blocks):
        passes["tile_mask"], passes["first_block"], passes["n_blocks"] = mask, first, count
        return lib.qsim_apply_passes(None, one, n, vp(passes), 1, vp(blk), one, one, 1)
    assert call(n=35) == 2                               # QSIM_ERANGE
    assert call(mask=1 << 12 | 1023) == 1                # above n_qubits
    assert call(mask=2046) == 1                          # qubit 0 missing
    assert call(mask=511) == 2 and call(n=16, mask=(1 << 14) - 1) == 2
    assert call(first=-1) == 1 and call(first=1) == 1 and call(count=2) == 1 and call(count=0) == 1
    for at, v in ((0, 0), (3, _sw(2)), (9, _sw(10)), (4, 3)):
        bad = blocks.copy()
        bad["bit"][0, at] = v
        assert call(blk=bad) == 1, (at, v)
    nq, qs, mat = np.array([2], np.int32), np.full((1, 8), -1, np.int32), np.eye(4, dtype=np.complex128)
    qs[0, :2] = 0, 9
    out = [np.zeros(1, np.int32), passes, blocks, np.zeros(3072, np.uint16)]
    a, b = ctypes.c_int(), ctypes.c_int()

    def plan(n=12, m=10, low=4, w=2, q=9):
        nq[0], qs[0, 1] = w, q
        return lib.qsim_plan_passes(n, m, low, 1, vp(nq), vp(qs), vp(mat), *[vp(o) for o in out],
                                    ctypes.byref(a), ctypes.byref(b))
    assert plan() == 0 and (a.value, b.value) == (1, 1)
    assert plan(n=9) == 2 and plan(n=35) == 2 and plan(m=9) == 2 and plan(m=14) == 2
    assert plan(low=0) == 1 and plan(low=7) == 1 and plan(w=0) == 1 and plan(w=9) == 1
    assert plan(q=12) == 1 and plan(q=0) == 1


@pytest.mark.gpu
@pytest.mark.parametrize("n,m", [(10, 10), (11, 11), (11, 10), (12, 12), (13, 13), (14, 10), (14, 13), (17, 11), (18, 12)])
def test_pass_kernel_matches_fp64(bk, dev, n, m):
    """Random 1-, 2- and 4-qubit unitaries on spread-out qubits (every tile
    bit takes part) on a random state.  One block costs at most 8e-6 max|a|
    (32-term dot products accumulated in FP32 on groups of 16 amplitudes)."""
    import torch
    from blackwell_backend import compiler as C
    from blackwell_backend.executor import CompiledCircuit
    rng = np.random.default_rng(n * 20 + m)
    ops = []
    for i in range(14):
        k = int(rng.choice([1, 2, 2, 4]))
        ops.append(C.Op({1: "m1", 2: "m2"}.get(k, "mk"), rng.choice(n, k, replace=False), rand_unitary(1 << k, i)))
    ops += [C.Op("m2", [q, (q + 5) % n], rand_unitary(4, 100 + q)) for q in range(n)]
    psi = rand_state(n, n)
    cc = CompiledCircuit(n, 0, ops)
    plan = cc._build_passes(C.plan_passes(ops, n, m, 4), dev)
    n_blocks = sum(len(a[1]) for kind, a in plan.steps if kind == "passes")
    got = plan.run(torch.from_numpy(psi.copy()).to(dev)).cpu().numpy()
    ref = psi.astype(np.complex128)
    for op in ops:
        ref = O.apply_matrix(ref, op.full_matrix(), list(op.all_qubits))
    assert np.max(np.abs(got - ref)) <= 8e-6 * n_blocks * np.max(np.abs(ref))


@pytest.mark.gpu
def test_passes_apply_permutations_and_wide_ops(dev):
    """Permutation gates of up to four qubits in a pass against the permuted
    amplitudes; ops of five and more qubits run between passes."""
    from blackwell_backend import BlackwellSimulator
    from blackwell_backend.circuit import QuantumCircuit
    sim = BlackwellSimulator(dev)
    qc = QuantumCircuit(14)
    for q in range(14):
        qc.ry(0.3 + q, q).rz(0.1 * q, q)
    ref, _ = sim.run_statevector(qc, mode="passes")
    perm = qc.copy()
    perm.cx(0, 13).ccx(4, 9, 2).swap(3, 11).mcx([1, 5, 7], 12).cx(8, 6)
    sv, _ = sim.run_statevector(perm, mode="passes")
    psi = ref.astype(np.complex128)
    for name, qs in (("cx", (0, 13)), ("ccx", (4, 9, 2)), ("swap", (3, 11)), ("mcx", (1, 5, 7, 12)), ("cx", (8, 6))):
        i = np.arange(1 << 14)
        if name == "swap":
            a, b = (i >> qs[0]) & 1, (i >> qs[1]) & 1
            j = np.where(a != b, i ^ (1 << qs[0]) ^ (1 << qs[1]), i)
        else:
            on = np.all([(i >> c) & 1 for c in qs[:-1]], axis=0)
            j = np.where(on, i ^ (1 << qs[-1]), i)
        psi = psi[j]
    assert np.max(np.abs(sv - psi)) <= 8e-6 * np.max(np.abs(psi))
    wide = QuantumCircuit(12, 1)
    wide.h(0).cx(0, 11)
    wide.unitary(rand_unitary(32, 3), [1, 4, 7, 9, 11])
    wide.mcx([0, 2, 3, 5, 6], 8)
    wide.ry(0.7, 8).cx(8, 3)
    got, _ = sim.run_statevector(wide, mode="passes")
    exp, _ = sim.run_statevector(wide, mode="plain")
    assert O.fidelity(exp, got) >= 1 - 1e-7 and np.max(np.abs(exp - got)) <= 2e-6


@pytest.mark.gpu
@pytest.mark.parametrize("ns", [[13, 10, 16, 11, 12, 15], [10] * 70 + [13], [18, 14]])
def test_batched_passes_have_the_bits_of_single_ones(dev, ns):
    """Every tile size, more records than lanes of the search, states with
    fewer passes than others: each state equals qsim_apply_passes on it alone."""
    import ctypes
    import torch
    from blackwell_backend import compiler as C, workloads as W
    from blackwell_backend.executor import pass_shape
    from blackwell_kernels import _lib
    from blackwell_kernels.cuquantum import pass_step_records, run_pass_steps
    vp = ctypes.c_void_p
    plans, single, batch = [], [], []
    for i, n in enumerate(ns):
        pairs, us = W.su4_arrays(n, 2 + i % 3, 7 + i)
        qb = np.full((len(pairs), 8), -1, dtype=np.int32)
        qb[:, :2] = pairs
        m = 13 if n in (13, 16) else pass_shape(n)[0]
        refs, *plan = C.plan_passes_arrays(n, np.full(len(pairs), 2, np.int32), qb, us, m, 4)
        assert (refs >= 0).all()
        plans.append(C.PassRun(*plan))
        psi = torch.from_numpy(rand_state(n, i).astype(np.complex64)).to(dev)
        single.append(psi.clone())
        batch.append(psi.clone())
    up = lambda a: torch.from_numpy(a.view(np.uint8).reshape(-1).copy()).to(dev)
    s = _lib.stream_handle(dev)
    for n, p, st in zip(ns, plans, single):
        b, f = up(p.blocks), up(p.frags)
        _lib.call("qsim_apply_passes", s, _lib.ptr(st), n, vp(p.passes.ctypes.data), len(p.passes),
                  vp(p.blocks.ctypes.data), _lib.ptr(b), _lib.ptr(f), len(p.blocks))
    blocks = np.concatenate([p.blocks for p in plans])
    first = np.cumsum([0] + [len(p.blocks) for p in plans])[:-1]
    recs, off = pass_step_records([st.data_ptr() for st in batch], ns, [p.passes for p in plans], first)
    assert off[-1] == len(recs) == sum(len(p.passes) for p in plans)
    bd, fd, rd = up(blocks), up(np.concatenate([p.frags for p in plans])), up(recs)
    run_pass_steps(s, recs, rd.data_ptr(), off, blocks, bd.data_ptr(), fd.data_ptr())
    for a, b in zip(single, batch):
        assert np.array_equal(a.cpu().numpy().view(np.uint32), b.cpu().numpy().view(np.uint32))
