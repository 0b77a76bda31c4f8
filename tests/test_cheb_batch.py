"""The tiled matrix-free Chebyshev term (qsim_cheb_pauli_batch_step) and its
group records."""
import ctypes
import os
import sys

import numpy as np
import pytest
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
for _p in (ROOT, os.path.join(ROOT, "qiskit-blackwell_amd")):
    if _p not in sys.path:
        sys.path.insert(0, _p)

from blackwell_backend.hamiltonian import (HamiltonianCSR, PauliTables, SparsePauliOp, constant_group_entries,
                                            pauli_groups, real_group_records)
from blackwell_backend.chebyshev import chebyshev_evolve_batch
from blackwell_kernels import _lib
from blackwell_kernels._lib import ptr


def mixed_terms(n, seed, real=True):
    """Every kind of group: constant entries (X only), one and two terms on
    near and far masks, a pair that cancels in half of the rows, three and
    nine terms, a label given twice, and pairs whose masks stay above the
    wave's bits."""
    rng = np.random.default_rng(seed)

    def lab(**ops):
        s = ["I"] * n
        for q, ch in ops.items():
            s[n - 1 - int(q[1:])] = ch
        return "".join(s)

    q = lambda i: f"q{i}"
    out = [(lab(**{q(i): "X"}), rng.uniform(-1, 1)) for i in range(n)]
    out += [(lab(**{q(n - 1): "Z"}), 0.75), (lab(**{q(0): "Z", q(1): "Z"}), -0.3)]
    for i in range(n - 1):
        c = rng.uniform(-1, 1)
        out += [(lab(**{q(i): "X", q(i + 1): "X"}), c), (lab(**{q(i): "Y", q(i + 1): "Y"}), c)]
    for z in range(3, 6):                                   # three terms on a far mask
        out.append((lab(**{q(0): "X", q(n - 1): "X", q(z): "Z"}), rng.uniform(-1, 1)))
    for z in (0, 1, 3, 4, 5, 6, 7, 8, 0):                   # nine, one of them twice
        out.append((lab(**{q(2): "X", q(z): "Z"}), rng.uniform(-1, 1)))
    out.append((lab(**{q(3): "X", q(n - 2): "Z"}), 0.5))
    out.append((lab(**{q(5): "X", q(6): "X", q(n - 1): "Z", q(n - 2): "Z"}), 0.25))
    out.append(out[-1])
    if not real:
        out.append((lab(**{q(4): "Y"}), 0.5))
    return out


def test_group_records_give_the_entries():
    """Per row of a 9-qubit Hamiltonian, the entry from the records is the
    FP64 sum over the tables rounded to FP32; imaginary entries have none."""
    n = 9
    terms = mixed_terms(n, 1)
    tables = lambda ts: pauli_groups([t[0] for t in ts], [t[1] for t in ts])
    records = lambda xm, *tab: real_group_records(xm, *tab, constant_group_entries(*tab))
    xm, toff, sm, coef = tables(terms)
    recs = records(xm, toff, sm, coef)
    rows = np.arange(1 << n, dtype=np.uint64)
    par = lambda m: np.array([bin(int(r) & int(m)).count("1") & 1 for r in rows])
    assert set(recs["kind"]) == {_lib.PAULI_CONST, _lib.PAULI_PAIR, _lib.PAULI_TERMS}
    for g, rec in enumerate(recs):
        want = np.zeros(1 << n)
        for t in range(toff[g], toff[g + 1]):
            want += np.where(par(sm[t]), -coef[t].real, coef[t].real)
        want = want.astype(np.float32)
        if rec["kind"] == _lib.PAULI_CONST:
            got = np.full(1 << n, rec["same"])
        elif rec["kind"] == _lib.PAULI_PAIR:
            p0, p1 = par(rec["m"][0]), par(rec["m"][1])
            got = np.where(p0, -1.0, 1.0) * np.where(p0 == p1, rec["same"], rec["diff"])
            assert np.array_equal(np.where(p0, -rec["c"][0], rec["c"][0]) +
                                  np.where(p1, -rec["c"][1], rec["c"][1]),
                                  np.where(p0, -1.0, 1.0) * np.where(p0 == p1, rec["c"][0] + rec["c"][1],
                                                                     rec["c"][0] - rec["c"][1]))
        else:
            assert (rec["t0"], rec["nt"]) == (toff[g], toff[g + 1] - toff[g])
            continue
        assert np.array_equal(got.astype(np.float32), want), g
    bad = mixed_terms(n, 1, real=False)
    assert records(*tables(bad)) is None


@pytest.mark.gpu
@pytest.mark.parametrize("n,R", [(9, 1), (9, 3), (10, 2), (11, 33), (14, 5), (17, 4), (18, 1), (16, 32)])
def test_tiled_term_has_the_bits_of_the_untiled_one(n, R):
    """One term, first and later, on R vectors: T_{k+1}, accumulator and
    compensation are those of qsim_cheb_pauli_step on each vector alone."""
    dev = torch.device("cuda", 0)
    terms = mixed_terms(n, n)
    pt = PauliTables([t[0] for t in terms], [t[1] for t in terms], dev)
    assert pt.groups is not None
    g = torch.Generator(device=dev).manual_seed(n * 100 + R)
    new = lambda: torch.view_as_complex(torch.randn(R, 1 << n, 2, device=dev, generator=g))
    T, prev, acc, comp = new(), new(), new(), new() * 1e-8
    s = _lib.stream_handle(dev)
    for first in (1, 0):
        want, got = [[x.clone() for x in (prev, acc, comp)] for _ in range(2)]
        for j in range(R):
            _lib.call("qsim_cheb_pauli_step", s, n, *pt.step_args(), 0.21, ptr(T[j]), *(ptr(x[j]) for x in want),
                      0.3, -0.2, first)
        _lib.call("qsim_cheb_pauli_batch_step", s, n, *pt.batch_args(), R, 0.21, ptr(T), *(ptr(x) for x in got),
                  0.3, -0.2, first)
        for a, b in zip(want, got):
            assert np.array_equal(torch.view_as_real(a).cpu().numpy(), torch.view_as_real(b).cpu().numpy()), first


@pytest.mark.gpu
def test_batch_evolution_by_tiles_equals_the_csr_terms():
    """17 qubits, three states in a strided view: the default route reports
    matrix-free terms and gives the CSR route's bits; the states are left as
    they were; a Hamiltonian with imaginary entries stays on the CSR."""
    dev = torch.device("cuda", 0)
    n = 17
    g = torch.Generator(device=dev).manual_seed(5)
    X = torch.view_as_complex(torch.randn(6, 1 << n, 2, device=dev, generator=g))
    X = (X / torch.linalg.vector_norm(X, dim=1, keepdim=True))[::2]
    keep = X.clone()
    h = HamiltonianCSR.from_sparse_pauli_op(SparsePauliOp.from_list(mixed_terms(n, 3)), device=dev)
    a, ia = chebyshev_evolve_batch(X, h, 0.4, 1e-8)
    b, ib = chebyshev_evolve_batch(X, h, 0.4, 1e-8, matrix_free=False)
    assert ia["matrix_free"] and not ib["matrix_free"] and ia["chebyshev_degree"] == ib["chebyshev_degree"]
    assert a.shape == b.shape and a.is_contiguous() and torch.equal(keep, X)
    assert np.array_equal(a.cpu().numpy(), b.cpu().numpy())
    h = HamiltonianCSR.from_sparse_pauli_op(SparsePauliOp.from_list(mixed_terms(n, 3, real=False)), device=dev)
    _, ic = chebyshev_evolve_batch(X, h, 0.1, 1e-6)
    assert not ic["matrix_free"]


def test_tiled_term_checks_its_arguments():
    lib = _lib.load()
    z = (1.0, 16, 16, 16, 16, 0.0, 0.0, 0)
    assert lib.qsim_cheb_pauli_batch_step(None, 8, 1, 16, 16, 16, 1, *z) == 2
    assert lib.qsim_cheb_pauli_batch_step(None, 10, 1, None, 16, 16, 1, *z) == 1
    assert lib.qsim_cheb_pauli_batch_step(None, 10, 1, 16, 16, 16, 0, *z) == 1
    assert lib.qsim_cheb_pauli_batch_step(None, 10, 1, 16, 16, 16, 1, 1.0, 24, 16, 16, 16, 0.0, 0.0, 0) == 1


def dense_terms(n, seed):
    """More groups than lanes of a wave (X pairs), one of them with more terms
    than lanes (Z strings)."""
    rng = np.random.default_rng(seed)
    pairs = [(i, j) for i in range(n) for j in range(i)]

    def lab(ch, qs):
        return "".join(ch if n - 1 - p in qs else "I" for p in range(n))

    out = [(lab("Z", q), rng.uniform(-1, 1)) for q in pairs + [(i,) for i in range(n)]]
    for q in pairs:
        out += [(lab("X", q), rng.uniform(-1, 1)), (lab("Y", q), rng.uniform(-1, 1))]
    return out


@pytest.mark.gpu
@pytest.mark.parametrize("n,R,K,make", [(9, 1, 1, mixed_terms), (10, 1, 5, mixed_terms), (12, 1, 4, dense_terms),
                                        (19, 1, 3, mixed_terms), (21, 1, 2, mixed_terms), (10, 3, 2, mixed_terms),
                                        (12, 4, 5, dense_terms)])
def test_whole_series_has_the_bits_of_its_terms(n, R, K, make):
    """Odd and even term counts, every number of rows per thread: the series in
    one call equals start, terms and finish by the untiled kernels."""
    dev = torch.device("cuda", 0)
    terms = make(n, n)
    pt = PauliTables([t[0] for t in terms], [t[1] for t in terms], dev)
    assert pt.groups is not None
    g = torch.Generator(device=dev).manual_seed(n + R + K)
    T0 = torch.view_as_complex(torch.randn(R, 1 << n, 2, device=dev, generator=g))
    if K == 1:
        T0[0, 5] = complex(float("inf"), 1.0)               # a zero entry takes nothing from it
    c = np.random.default_rng(K).standard_normal((K + 1, 2)).view(np.complex128).reshape(-1)
    s = _lib.stream_handle(dev)
    a, b, acc, comp = T0.clone(), *[torch.full_like(T0, float("nan")) for _ in range(3)]
    _lib.call("qsim_cheb_pauli_evolve", s, n, *pt.batch_args(), R, 0.1, ptr(a), ptr(b), ptr(acc), ptr(comp),
              ctypes.c_void_p(c.ctypes.data), K)
    got = (b if K % 2 else a).cpu().numpy()
    for j in range(R):
        cur, prv, acc, comp = T0[j].clone(), *[torch.empty_like(T0[j]) for _ in range(3)]
        _lib.call("qsim_cheb_init_acc", s, ptr(acc), ptr(comp), ptr(cur), 1 << n, c[0].real, c[0].imag)
        for k in range(1, K + 1):
            _lib.call("qsim_cheb_pauli_step", s, n, *pt.step_args(), 0.1, ptr(cur), ptr(prv), ptr(acc), ptr(comp),
                      c[k].real, c[k].imag, int(k == 1))
            cur, prv = prv, cur
        _lib.call("qsim_cheb_finish", s, ptr(prv), ptr(acc), ptr(comp), 1 << n)
        assert np.array_equal(prv.cpu().numpy(), got[j], equal_nan=True)
        assert np.isfinite(got[j]).any()


def test_series_checks_its_arguments():
    lib = _lib.load()
    c = np.zeros(4)
    call = lambda n=10, g=16, R=1, t0=16, t1=16, cf=c.ctypes.data, K=1: lib.qsim_cheb_pauli_evolve(
        None, n, 1, g, 16, 16, R, 1.0, t0, t1, 16, 16, cf, K)
    assert call(n=8) == 2 and call(g=None) == 1 and call(R=0) == 1 and call(cf=None) == 1 and call(K=0) == 1
    assert call(t0=24) == 1 and call(t1=24) == 1 and call(t1=None) == 1


def _ising(n, extra=0):
    """ZZ on every pair, or `extra` Z strings in their place, and X on every qubit."""
    rng = np.random.default_rng(n + extra)
    lab = lambda ch, qs: "".join(ch if n - 1 - p in qs else "I" for p in range(n))
    qs = [rng.choice(n, 4, replace=False) for _ in range(extra)] or [(i, j) for i in range(n) for j in range(i)]
    return [(lab("Z", q), rng.uniform(-1, 1)) for q in qs] + [(lab("X", (q,)), rng.uniform(-1, 1)) for q in range(n)]


def test_tiled_terms_are_chosen_by_the_hamiltonian():
    """Against the faster route of each as measured: (tables, qubits, states,
    tiled).  All-to-all Ising and one X mask of a thousand terms are the CSR's
    at 17 qubits, and the untiled kernel's for one state of 18 qubits and more."""
    from blackwell_backend.chebyshev import tiled_term
    tables = lambda terms: PauliTables([t[0] for t in terms], [t[1] for t in terms], "cpu")
    chain = lambda n: tables([("".join(ch if n - 1 - p in (i, i + 1) else "I" for p in range(n)), 0.3 + i + j)
                              for i in range(n - 1) for j, ch in enumerate("ZXY")] + _ising(n, 1)[1:])
    for n in (17, 20):
        t = chain(n)
        assert t.long_terms == n - 1
        assert [tiled_term(t, n, R) for R in (1, 2, 4, 8, 32)] == [True] * 5
        t = tables(_ising(n))
        assert (t.n_groups, t.long_terms) == (n + 1, n * (n - 1) // 2)
        assert [tiled_term(t, n, R) for R in (1, 4, 8)] == ([True, False, False] if n == 17 else [False, True, True])
        t = tables(_ising(n, 1000))
        assert [tiled_term(t, n, R) for R in (1, 2, 4, 8, 32)] == [n == 17, False, False, False, False]
    assert not tiled_term(chain(16), 16, 8) and tiled_term(chain(16), 16, 16) and not tiled_term(chain(16), 16, 0)
    assert tiled_term(chain(12), 12, 1) and not tiled_term(chain(8), 8, 1) and not tiled_term(chain(12), 12, 32)


@pytest.mark.gpu
@pytest.mark.parametrize("n,R,matrix_free", [(17, 4, False), (18, 1, True), (18, 3, True)])
def test_evolution_of_many_terms_a_mask_has_the_same_bits_by_either_route(n, R, matrix_free):
    dev = torch.device("cuda", 0)
    g = torch.Generator(device=dev).manual_seed(n)
    X = torch.view_as_complex(torch.randn(R, 1 << n, 2, device=dev, generator=g))
    X = X / torch.linalg.vector_norm(X, dim=1, keepdim=True)
    h = HamiltonianCSR.from_sparse_pauli_op(SparsePauliOp.from_list(_ising(n, 300)), device=dev)
    a, ia = chebyshev_evolve_batch(X, h, 0.05, 1e-7)
    b, ib = chebyshev_evolve_batch(X, h, 0.05, 1e-7, matrix_free=False)
    assert ia["matrix_free"] == matrix_free and not ib["matrix_free"]
    assert np.array_equal(a.cpu().numpy(), b.cpu().numpy())
