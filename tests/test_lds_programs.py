"""LDS programs at the edges of their op chunks and workgroup sizes."""
import os
import sys

import numpy as np
import pytest
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
for _p in (ROOT, os.path.join(ROOT, "qiskit-blackwell_amd")):
    if _p not in sys.path:
        sys.path.insert(0, _p)

from helpers import rand_state, rand_unitary
from oracle import statevector as O


@pytest.mark.gpu
@pytest.mark.parametrize("n,n_ops", [(2, 1), (3, 16), (6, 17), (10, 15), (10, 33), (11, 16), (12, 32), (13, 18)])
def test_whole_program_matches_fp64(n, n_ops):
    """One tile, ops of every kind, some whose coefficients are not staged
    (three qubits).  Per op the state's error in the 2-norm grows by at most
    2^-24 sqrt(2) for the rounded amplitudes and 4 sqrt(2) 2^-24 for the rounded
    coefficients: 8 * 2^-24 per op."""
    from blackwell_backend import compiler as C
    from blackwell_backend.executor import CompiledCircuit
    rng = np.random.default_rng(100 * n + n_ops)
    ops = []
    for i in range(n_ops):
        kinds = ["m1", "d1", "ph", "x", "m2", "swap"] + (["mk", "cx"] if n > 2 else [])
        kind = kinds[i % len(kinds)]
        k = {"m2": 2, "swap": 2, "mk": 3, "cx": 2}.get(kind, 1)
        q = [int(v) for v in rng.choice(n, k, replace=False)]
        if kind in ("m1", "m2", "mk"):
            ops.append(C.Op(kind, q, rand_unitary(1 << k, i)))
        elif kind in ("d1", "ph"):
            ops.append(C.Op(kind, q, np.exp(1j * rng.uniform(0, 6, 2 if kind == "d1" else 1))))
        elif kind == "cx":
            ops.append(C.Op("x", q[:1], controls=q[1:]))
        else:
            ops.append(C.Op(kind, q))
    psi = rand_state(n, n).astype(np.complex64)
    got = CompiledCircuit(n, 0, ops).plan("whole", "cuda:0").run(torch.from_numpy(psi.copy()).to("cuda:0")).cpu().numpy()
    ref = psi.astype(np.complex128)
    for op in ops:
        ref = O.apply_matrix(ref, op.full_matrix(), list(op.all_qubits))
    assert np.linalg.norm(got - ref) <= 8 * 2.0 ** -24 * n_ops * np.linalg.norm(ref)
