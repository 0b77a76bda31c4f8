"""The arithmetic of the block passes: FP32 amplitudes and coefficients as
three bf16 each.  Errors stay where three FP32 roundings a block put them,
permutations keep every bit, and the variants that large states run by default
(nontemporal from 26 qubits, byte offsets up to bit 31 at 29, 64-bit offsets
from 30) agree with the per-gate kernels."""
import numpy as np
import pytest

from helpers import rand_state, rand_unitary
from oracle import statevector as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,m", [(10, 10), (11, 11), (12, 12), (13, 13), (14, 12), (16, 11)])
def test_pass_errors_are_those_of_fp32_sums(dev, n, m):
    """A block sums 32 products to a component in two steps and adds the small
    ones: three roundings to nearest, the first at half the magnitude, each off by
    0.41 * 2^-24 of the value in the root mean square, 0.65 * 2^-24 together; and
    blocks add in squares.  2^-24 a block is half as much again; in a model of
    the sums a block is off by 58 * 2^-24 without the products of the lowest
    parts, and by 74 without that of the middle parts too."""
    import torch
    from blackwell_backend import compiler as C
    from blackwell_backend.executor import CompiledCircuit
    rng = np.random.default_rng(n * 50 + m)
    ops = [C.Op("mk", rng.choice(n, 4, replace=False), rand_unitary(16, 7 * n + i)) for i in range(24)]
    psi = rand_state(n, n)
    cc = CompiledCircuit(n, 0, ops)
    plan = cc._build_passes(C.plan_passes(ops, n, m, 4), dev)
    assert sum(len(a[1]) for kind, a in plan.steps) == len(ops)
    got = plan.run(torch.from_numpy(psi.copy()).to(dev)).cpu().numpy()
    ref = psi.astype(np.complex128)
    for op in ops:
        ref = O.apply_matrix(ref, op.mat, list(op.qubits))
    assert np.linalg.norm(got - ref) <= np.sqrt(len(ops)) * 2.0 ** -24 * np.linalg.norm(ref)


@pytest.mark.parametrize("n", [10, 11, 12, 13, 15])
def test_permutations_in_passes_keep_every_bit(dev, n):
    """X, CX, SWAP and X of two and three controls on amplitudes of full 24-bit
    mantissas and of exponents from 2^-80 to 2^100."""
    import torch
    from blackwell_backend import compiler as C
    from blackwell_backend.executor import CompiledCircuit
    rng = np.random.default_rng(n)
    ops = []
    for i in range(40):
        q = [int(v) for v in rng.choice(n, 4, replace=False)]
        ops.append(C.Op("swap", q[:2]) if i % 5 == 4 else C.Op("x", q[:1], controls=q[1:1 + i % 5]))
    v = rng.standard_normal((2, 1 << n)) * 2.0 ** rng.integers(-80, 100, (2, 1 << n))
    psi = (v[0] + 1j * v[1]).astype(np.complex64)
    cc = CompiledCircuit(n, 0, ops)
    plan = cc._build_passes(C.plan_passes(ops, n, min(n, 12), 4), dev)
    assert [kind for kind, _ in plan.steps] == ["passes"]
    got = plan.run(torch.from_numpy(psi.copy()).to(dev)).cpu().numpy()
    i = np.arange(1 << n)
    for op in ops:
        if op.kind == "swap":
            a, b = op.qubits
            j = np.where((i >> a & 1) != (i >> b & 1), i ^ (1 << a) ^ (1 << b), i)
        else:
            on = np.all([i >> c & 1 for c in op.controls], axis=0) if op.controls else np.ones(1 << n, bool)
            j = np.where(on, i ^ (1 << op.qubits[0]), i)
        psi = psi[j]
    assert np.array_equal(got.view(np.uint32), psi.view(np.uint32))


@pytest.mark.parametrize("n", [26, 28, 29, 30])
def test_large_states_in_passes_agree_with_the_gate_kernels(dev, n):
    """auto on three layers of SU(4) gates, the ends of the register among them,
    against one launch a gate on the same random state, and a layer of
    permutations bit for bit.  Errors as above, and one rounding a gate."""
    import torch
    import blackwell_kernels as bk
    from blackwell_backend import compiler as C, workloads as W
    from blackwell_backend.circuit import QuantumCircuit, instructions
    from blackwell_backend.executor import CompiledCircuit
    print(f"[large passes] {n} qubits", flush=True)
    qc = W.su4_volume(n, 3, 5)
    for i, (a, b) in enumerate(((0, n - 1), (n - 2, 3), (n - 1, n - 3))):
        qc.unitary(rand_unitary(4, i), [a, b])
    perm = QuantumCircuit(n)
    perm.cx(0, n - 1).mcx([n - 1, 2, n - 2], 1).swap(n - 3, 4).cx(n - 2, 0).ccx(5, n - 4, n - 1).swap(0, n - 2)
    g = torch.Generator(device=dev)
    g.manual_seed(n)
    keep = torch.randn(1 << n, dtype=torch.complex64, device=dev, generator=g)
    for circuit in (qc, perm):
        cc = CompiledCircuit(n, 0, C.compile_ops(instructions(circuit)))
        assert cc.resolve_mode("auto") == "passes"
        plan = cc.plan("passes", dev)
        ref = cc.plan("plain", dev).run(keep.clone())
        got = plan.run(keep.clone())
        if circuit is perm:
            assert torch.equal(got.view(torch.int32), ref.view(torch.int32))
        else:
            blocks = sum(len(a[1]) for kind, a in plan.steps)
            total = float(bk.norm2(ref))
            err = float(bk.norm2(got.sub_(ref)))
            assert 0.0 < (err / total) ** 0.5 <= 2.0 ** -24 * (blocks ** 0.5 + len(cc.ops) ** 0.5)
        del ref, got
    del keep
    torch.cuda.empty_cache()


def test_28q_circuit_then_inverse_in_auto(dev):
    import torch
    import blackwell_kernels as bk
    from blackwell_backend import BlackwellSimulator, workloads as W
    from test_gpu_fullsize import _inverse_appended
    sim = BlackwellSimulator(dev)
    print("[large passes] su4 28q forward+inverse in auto", flush=True)
    cc = sim.compile(_inverse_appended(W.su4_volume(28, 28, 2024)))
    assert cc.resolve_mode("auto") == "passes"
    st = cc.plan("passes", sim.device).run(bk.state_init(28, device=sim.device))
    p0, nrm = abs(complex(st[0].item())) ** 2, float(bk.norm2(st))
    del st
    torch.cuda.empty_cache()
    assert p0 >= 1 - 1e-6 and abs(nrm - 1) <= 1e-6, (p0, nrm)
