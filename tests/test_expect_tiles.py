"""Tiled expectation passes: many x masks per read of the state."""
import os
import sys

import numpy as np
import pytest
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
for _p in (ROOT, os.path.join(ROOT, "qiskit-blackwell_amd")):
    if _p not in sys.path:
        sys.path.insert(0, _p)


def strings(n, seed):
    """(x, z) masks: every kind of group (x = 0, x = 1, even and odd x, near
    and far) with 1, 2, 3, 8 and 9 terms of either Y parity, more groups than
    one pass holds, and masks of more qubits than a tile has."""
    rng = np.random.default_rng(seed)
    lim = 1 << n
    out = [(0, z) for z in [0, 1, lim - 1] + [int(v) for v in rng.integers(0, lim, 18)]]
    xs = [1, 2, 3, 1 << (n - 1), (1 << (n - 1)) | 1, 3 << (n - 2), 6, 0x41, 0x80]
    for x, cnt in zip(xs, (2, 1, 3, 8, 9, 2, 5, 1, 2)):
        out += [(x, int(v)) for v in rng.integers(0, lim, cnt)]
    out += [(x, 0) for x in range(64, 64 + 70)]
    out += [(lim - 1, int(v)) for v in rng.integers(0, lim, 3)]
    out += [(int(x), int(z)) for x, z in rng.integers(0, lim, (12, 2))]
    return [out[i] for i in rng.permutation(len(out))]


@pytest.mark.gpu
@pytest.mark.parametrize("n", [9, 10, 11, 12, 13, 14, 17])
def test_tiled_expectations_match_numpy(n):
    """Each value against the FP64 sum over the same complex64 state.  The
    products are exact, so both sides differ from the true sum by at most
    2^n * 2^-53 of the sum of magnitudes, which is at most |psi|^2; twice
    that, and every call gives the same bits."""
    import blackwell_kernels as bk
    rng = np.random.default_rng(n)
    psi = (rng.standard_normal(1 << n) + 1j * rng.standard_normal(1 << n)).astype(np.complex64)
    st = torch.from_numpy(psi).to("cuda:0")
    terms = strings(n, n)
    xs, zs = [t[0] for t in terms], [t[1] for t in terms]
    got = bk.expectation_paulis(st, xs, zs).cpu().numpy()
    p64 = psi.astype(np.complex128)
    i = np.arange(1 << n)
    parity = np.array([bin(v).count("1") & 1 for v in range(1 << n)])
    want = [(1j ** (bin(x & z).count("1") % 4) * np.vdot(p64, np.where(parity[(i ^ x) & z], -1, 1) * p64[i ^ x])).real
            for x, z in terms]
    tol = 2.0 * 2.0 ** (n - 53) * float(np.vdot(p64, p64).real)
    assert np.max(np.abs(got - np.array(want))) <= tol
    assert np.array_equal(bk.expectation_paulis(st, xs, zs).cpu().numpy(), got)


@pytest.mark.gpu
@pytest.mark.parametrize("n,odd", [(20, 0), (20, 1), (22, 0)])
def test_groups_that_share_a_unit_match_numpy(n, odd):
    """Even masks of one and two terms in every combination: masks that hold
    each other's highest bit, neighbours and far ones, z with bit 0, on the
    other mask's qubits and outside the tile, two Y; an even and an odd number
    of groups, beside some that share none.  Tolerance as above."""
    import blackwell_kernels as bk
    rng = np.random.default_rng(n + odd)
    hi = 1 << (n - 1)
    masks = [(2, 1), (4, 2), (6, 2), (10, 1), (12, 2), (8, 2), (hi, 1), (hi | 2, 1), (3 << 9, 2), (1 << 10, 1)]
    terms = [(0, 5), (0, hi | 1), (3, 0), (2, 2), (1, 8)]
    for x, cnt in masks + [(hi | 4, 1)] * odd:
        for _ in range(cnt):
            z = int(rng.integers(0, 1 << n))
            while bin(z & x).count("1") & 1 or (x, z) in terms:
                z = int(rng.integers(0, 1 << n))
            terms.append((x, z))
    psi = (rng.standard_normal(1 << n) + 1j * rng.standard_normal(1 << n)).astype(np.complex64)
    xs, zs = [t[0] for t in terms], [t[1] for t in terms]
    got = bk.expectation_paulis(torch.from_numpy(psi).to("cuda:0"), xs, zs).cpu().numpy()
    p64 = psi.astype(np.complex128)
    i = np.arange(1 << n)
    for (x, z), v in zip(terms, got):
        par = (i ^ x) & z
        for sh in (16, 8, 4, 2, 1):
            par ^= par >> sh
        want = (1j ** (bin(x & z).count("1") % 4) * np.vdot(p64, np.where(par & 1, -1, 1) * p64[i ^ x])).real
        assert abs(v - want) <= 2.0 * 2.0 ** (n - 53) * float(np.vdot(p64, p64).real), (x, z)
