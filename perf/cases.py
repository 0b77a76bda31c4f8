"""The measured work of this framework: what its users have it do, through
its public entry points, over the range of sizes they use.

Families (the "kind" of a case):
  gates    one call of the kernel API per gate on a resident state
  circuit  a whole circuit, either run_statevector() (state back on the host)
           or a compiled plan run on a device state, as programs do that go
           on working with the state
  evolve   exp(-iHt) of a spin chain on one state or on a batch of states
  observe  energy of a state and shots from it
  serve    a mixed stream of small circuits through the batching server

A case is a dict of plain values; every input is made from (case, seed).
"""
import math
import os
import sys

import numpy as np
import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "qiskit-blackwell_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

DEV = "cuda:0"


def listed():
    return [
        # the plugin API at a size where only call and launch cost count: a
        # hybrid loop applying single gates to a small register
        {"name": "gates_12q", "kind": "gates", "n": 12, "shift": 0},
        # the 12-qubit, 564-gate rotation ladder: a deep variational circuit on
        # a small register, latency of the whole call
        {"name": "ladder_12q", "kind": "circuit", "family": "ladder", "n": 12, "depth": 12, "host": True},
        # QFT of a product state at the size where tile programs run it
        {"name": "qft_16q", "kind": "circuit", "family": "qft", "n": 16, "depth": 1, "host": True},
        # quantum-volume circuits: the dense two-qubit workload, from a state
        # that stays in cache to one that streams through HBM
        {"name": "volume_20q", "kind": "circuit", "family": "volume", "n": 20, "depth": 20, "host": True},
        {"name": "volume_24q", "kind": "circuit", "family": "volume", "n": 24, "depth": 24, "host": False},
        {"name": "volume_28q", "kind": "circuit", "family": "volume", "n": 28, "depth": 28, "host": False},
        # rotations, CNOT ladder and multi-controlled X gates: the shallow,
        # permutation-heavy ansatz, on an odd register size
        {"name": "mcx_27q", "kind": "circuit", "family": "mcx", "n": 27, "depth": 4, "host": False},
        # the plugin API on a state far beyond the caches: one pass per gate
        {"name": "gates_28q", "kind": "gates", "n": 28, "shift": 0},
        # time evolution of one state (a quench of a spin chain)
        {"name": "evolve_19q", "kind": "evolve", "n": 19, "rhs": 1, "t": 1.0},
        # the same for an ensemble of 32 initial states at once
        {"name": "evolve_20q_x32", "kind": "evolve", "n": 20, "rhs": 32, "t": 1.0},
        # readout: energy of the chain and shots
        {"name": "observe_24q", "kind": "observe", "n": 24, "shots": 65536},
        # a statevector service: circuits of 10..18 qubits, states returned
        {"name": "serve_48", "kind": "serve", "count": 48, "n_min": 10, "n_max": 18},
    ]


def draw(rng):
    """One more case of the same families; a register above 27 qubits only one
    gate at a time, so that no drawn case costs more than the largest listed."""
    kind = rng.choice(["gates", "circuit", "circuit", "circuit", "evolve", "observe", "serve"])
    if kind == "gates":
        n = rng.randint(10, 28)
        return {"kind": kind, "n": n, "shift": rng.randrange(n)}
    if kind == "evolve":
        if rng.random() < 0.5:
            return {"kind": kind, "n": rng.randint(10, 21), "rhs": 1, "t": round(rng.uniform(0.3, 2.0), 3)}
        return {"kind": kind, "n": rng.randint(10, 19), "rhs": rng.choice([3, 8, 32, 32]),
                "t": round(rng.uniform(0.3, 2.0), 3)}
    if kind == "observe":
        return {"kind": kind, "n": rng.randint(12, 26), "shots": int(2 ** rng.uniform(10, 18))}
    if kind == "serve":
        n_max = rng.randint(14, 18)
        return {"kind": kind, "count": rng.randint(8, 56), "n_min": rng.randint(8, 12), "n_max": n_max}
    family = rng.choice(["ladder", "qft", "volume", "volume", "mcx"])
    n = rng.randint(10, 27)
    depth = {"ladder": rng.randint(2, 12), "qft": 1, "volume": rng.randint(4, n), "mcx": rng.randint(1, 6)}[family]
    return {"kind": "circuit", "family": family, "n": n, "depth": depth, "host": n <= 20}


# ------------------------------------------------------------------ inputs
def _haar(rng, count):
    z = rng.standard_normal((count, 4, 4)) + 1j * rng.standard_normal((count, 4, 4))
    q, r = np.linalg.qr(z)
    d = np.diagonal(r, axis1=1, axis2=2)
    return q * (d / np.abs(d))[:, None, :]


def _volume_arrays(n, depth, rng):
    p = n // 2
    pairs = np.concatenate([rng.permutation(n)[:2 * p].reshape(p, 2) for _ in range(depth)])
    return pairs.astype(np.int64), _haar(rng, depth * p)


def _gate_list(case, seed):
    """[(name, qubits, params)] of a circuit case, in circuit order."""
    n, depth, family = case["n"], case["depth"], case["family"]
    rng = np.random.default_rng(seed)
    out = []
    if family == "volume":
        pairs, us = _volume_arrays(n, depth, rng)
        return [("unitary", [int(a), int(b)], [u]) for (a, b), u in zip(pairs, us)]
    if family == "qft":
        th, ph = rng.uniform(0, 2 * math.pi, n), rng.uniform(0, 2 * math.pi, n)
        for q in range(n):
            out += [("ry", [q], [th[q]]), ("rz", [q], [ph[q]])]
        for j in reversed(range(n)):
            out.append(("h", [j], []))
            out += [("cp", [j, k], [math.pi / (1 << (j - k))]) for k in reversed(range(j))]
        return out + [("swap", [i, n - 1 - i], []) for i in range(n // 2)]
    for _ in range(depth):
        th, ph = rng.uniform(0, 2 * math.pi, n), rng.uniform(0, 2 * math.pi, n)
        if family == "ladder":
            out += [("h", [q], []) for q in range(n)]
        for q in range(n):
            out += [("ry", [q], [th[q]]), ("rz", [q], [ph[q]])]
        out += [("cx", [q, q + 1], []) for q in range(n - 1)]
        if family == "mcx":
            for _ in range(4):
                out.append(("mcx", [int(q) for q in rng.choice(n, 4, replace=False)], []))
    return out


def _circuit(n, gates):
    from blackwell_backend import QuantumCircuit
    qc = QuantumCircuit(n)
    for name, qs, ps in gates:
        if name == "unitary":
            qc.unitary(ps[0], qs)
        elif name == "mcx":
            qc.mcx(qs[:-1], qs[-1])
        else:
            getattr(qc, name)(*ps, *qs)
    return qc


def _state(n, seed, rhs=None):
    """Normalised random amplitudes, complex64."""
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    shape = (1 << n,) if rhs is None else (rhs, 1 << n)
    x = torch.view_as_complex(torch.randn(*shape, 2, generator=g, device=DEV))
    return x / torch.linalg.vector_norm(x, dim=-1, keepdim=True)


def _chain(n, seed):
    """[(label, coefficient)] of a Heisenberg chain with random couplings and
    transverse fields (label: rightmost character = qubit 0)."""
    rng = np.random.default_rng(seed)
    j, k, h = rng.uniform(-1, 1, n - 1), rng.uniform(-1, 1, n - 1), rng.uniform(-1, 1, n)

    def lab(ops):
        s = ["I"] * n
        for q, ch in ops:
            s[n - 1 - q] = ch
        return "".join(s)

    terms = []
    for i in range(n - 1):
        for ch, c in (("Z", j[i]), ("X", k[i]), ("Y", k[i])):
            terms.append((lab([(i, ch), (i + 1, ch)]), float(c)))
    return terms + [(lab([(i, "X")]), float(h[i])) for i in range(n)]


def _api_gates(n, shift, seed):
    """Calls of the kernel API: (function, matrix or phase or None, controls,
    targets), over in-register, in-wave and far targets; shift moves every
    qubit of the sequence up (mod n)."""
    rng = np.random.default_rng(seed)
    u4 = _haar(rng, 3)
    u2 = []
    for a, b, c in rng.uniform(0, 2 * math.pi, (4, 3)):
        u2.append(np.array([[math.cos(a), -np.exp(1j * b) * math.sin(a)],
                            [np.exp(1j * c) * math.sin(a), np.exp(1j * (b + c)) * math.cos(a)]]))
    ph = np.exp(1j * rng.uniform(0, 2 * math.pi, 3))
    m, t = n // 2, n - 1
    calls = [
        ("apply_gate", u2[0], [], [0]),
        ("apply_gate", u2[1], [], [m]),
        ("apply_gate", u2[2], [], [t]),
        ("apply_gate_2q", u4[0], [], [1, 4]),
        ("apply_gate_2q", u4[1], [], [3, m]),
        ("apply_gate_2q", u4[2], [], [m + 1, t]),
        ("apply_diagonal", ph[:2], [], [t - 1]),
        ("apply_diagonal_phase", ph[2], [], [m]),
        ("apply_mcx", None, [t - 2], [2]),
        ("apply_mcx", None, [4, t], [m]),
        ("apply_mcgate", u2[3], [m - 1], [t]),
        ("apply_mcswap", None, [], [4, t - 1]),
    ]
    return [(fn, mat, [(q + shift) % n for q in ctl], [(q + shift) % n for q in tg])
            for fn, mat, ctl, tg in calls]


def _serve_plan(case, seed):
    rng = np.random.default_rng(seed)
    span = np.arange(case["n_min"], case["n_max"] + 1)
    w = 0.75 ** (span - span[0])
    # the qubit counts of the stream stay those of the case; gates follow the seed
    ns = np.random.default_rng(case["count"]).choice(span, size=case["count"], p=w / w.sum())
    return [(int(n),) + _volume_arrays(int(n), int(n), rng) for n in ns]


def prepare(case, seed):
    kind = case["kind"]
    if kind == "gates":
        import blackwell_kernels as bk
        calls = []
        for fn, m, ctl, tg in _api_gates(case["n"], case["shift"], seed):
            if isinstance(m, np.ndarray):
                m = torch.from_numpy(m.astype(np.complex64)).to(DEV)
            calls.append((getattr(bk, fn), m, ctl, tg))
        return {"case": case, "state": _state(case["n"], seed), "calls": calls}
    if kind == "circuit":
        from blackwell_backend import BlackwellSimulator
        n = case["n"]
        sim = BlackwellSimulator(DEV)
        qc = _circuit(n, _gate_list(case, seed))
        if case["host"]:
            return {"case": case, "sim": sim, "qc": qc}
        cc = sim.compile(qc)
        return {"case": case, "cc": cc, "plan": cc.plan(cc.resolve_mode("auto", sim.device), sim.device),
                "state": torch.empty(1 << n, dtype=torch.complex64, device=DEV)}
    if kind in ("evolve", "observe"):
        from blackwell_backend import HamiltonianCSR, SparsePauliOp
        n = case["n"]
        spo = SparsePauliOp.from_list(_chain(n, seed))
        if kind == "observe":
            g = torch.Generator(device=DEV)
            g.manual_seed(seed + 1)
            u = torch.rand(case["shots"], dtype=torch.float64, device=DEV, generator=g)
            return {"case": case, "state": _state(n, seed), "op": spo, "u": u}
        return {"case": case, "ham": HamiltonianCSR.from_sparse_pauli_op(spo, DEV),
                "state": _state(n, seed, None if case["rhs"] == 1 else case["rhs"])}
    from blackwell_backend import BlackwellSimulator
    from blackwell_backend.serving import Request, Server
    reqs = [Request(i, 0.0, n, 0, i, gates=(pairs, us), keep_state=True)
            for i, (n, pairs, us) in enumerate(_serve_plan(case, seed))]
    return {"case": case, "server": Server(BlackwellSimulator(DEV)), "requests": reqs}


def run(state):
    kind = state["case"]["kind"]
    if kind == "gates":
        st = state["state"]
        for fn, m, ctl, tg in state["calls"]:
            if ctl or m is None:
                fn(st, ctl, *tg) if m is None else fn(st, m, ctl, *tg)
            else:
                fn(st, m, *tg)
        return st
    if kind == "circuit":
        if state["case"]["host"]:
            return state["sim"].run_statevector(state["qc"])[0]
        state["cc"].init_state(state["state"])
        return state["plan"].run(state["state"])
    if kind == "evolve":
        from blackwell_backend import chebyshev_evolve, chebyshev_evolve_batch
        fn = chebyshev_evolve if state["case"]["rhs"] == 1 else chebyshev_evolve_batch
        return fn(state["state"], state["ham"], state["case"]["t"])[0]
    if kind == "observe":
        import blackwell_kernels as bk
        from blackwell_backend.hamiltonian import expectation
        return {"energy": expectation(state["state"], state["op"]),
                "shots": bk.sample_with_uniforms(state["state"], state["u"])}
    state["server"].serve(state["requests"], realtime=False)
    return [r.state for r in state["requests"]]


# ------------------------------------------------------------------ least work
def _gate_flops(name, n):
    amps = float(1 << n)
    if name == "unitary":
        return 32 * amps
    if name in ("ry", "h"):
        return 14 * amps
    if name == "rz":
        return 6 * amps
    if name == "cp":
        return 1.5 * amps
    return 0.0


def work(case):
    kind = case["kind"]
    if kind == "gates":
        n, nbytes, flops = case["n"], 0.0, 0.0
        for fn, m, ctl, tg in _api_gates(n, case["shift"], 0):
            touched = 2.0 ** (n - len(ctl)) * (0.5 if fn in ("apply_mcswap", "apply_diagonal_phase") else 1.0)
            nbytes += 16 * touched
            flops += touched * {"apply_gate": 14, "apply_mcgate": 14, "apply_gate_2q": 30, "apply_diagonal": 6,
                                "apply_diagonal_phase": 6}.get(fn, 0)
        return {"bytes": nbytes, "flops": flops}
    if kind == "circuit":
        n = case["n"]
        gates = _gate_list(case, 0)
        return {"bytes": 8.0 * (1 << n) + 128.0 * len(gates), "flops": sum(_gate_flops(g, n) for g, _, _ in gates)}
    if kind == "evolve":
        # one read of the states, one write; per term each row sums one product
        # per entry (44 entries a row on a chain of 22)
        n, r = case["n"], case["rhs"]
        terms = case["t"] * 2.0 * n + 25
        return {"bytes": 16.0 * (1 << n) * r, "flops": terms * 8.0 * 2 * n * (1 << n) * r}
    if kind == "observe":
        n = case["n"]
        return {"bytes": 8.0 * (1 << n) + 16.0 * case["shots"], "flops": 4.0 * (4 * n - 3) * (1 << n)}
    ns = [n for n, _, _ in _serve_plan(case, 0)]
    return {"bytes": float(sum(8 << n for n in ns)), "flops": float(sum(32 * (n * (n // 2)) << n for n in ns))}


# ------------------------------------------------------------------ 64-bit results
def _split(n, qubits):
    """View shape that gives each of `qubits` an axis of its own, and those axes."""
    shape, axes, top = [], {}, n
    for q in sorted(qubits, reverse=True):
        shape.append(1 << (top - 1 - q))
        axes[q] = len(shape)
        shape.append(2)
        top = q
    shape.append(1 << top)
    return shape, axes


def _apply64(x, n, mat, targets, controls=()):
    """mat (row bit j <-> targets[j]) on targets where every control is 1."""
    shape, axes = _split(n, list(targets) + list(controls))
    v = x.view(shape)
    index = [slice(None)] * len(shape)
    for c in controls:
        index[axes[c]] = 1
    parts = []
    for r in range(1 << len(targets)):
        at = list(index)
        for j, t in enumerate(targets):
            at[axes[t]] = r >> j & 1
        parts.append(v[tuple(at)])
    mat = np.asarray(mat, dtype=np.complex128)
    if np.count_nonzero(mat - np.diag(np.diagonal(mat))) == 0:
        for r, p in enumerate(parts):
            if mat[r, r] != 1:
                p.mul_(complex(mat[r, r]))
        return
    old = [p.clone() for p in parts]
    for r, p in enumerate(parts):
        cols = [c for c in range(len(old)) if mat[r, c] != 0]
        p.copy_(old[cols[0]])
        if mat[r, cols[0]] != 1:
            p.mul_(complex(mat[r, cols[0]]))
        for c in cols[1:]:
            p.add_(old[c], alpha=complex(mat[r, c]))


_X = np.array([[0, 1], [1, 0]])
_SWAP = np.eye(4)[[0, 2, 1, 3]]


def _run64(n, gates):
    x = torch.zeros(1 << n, dtype=torch.complex128, device=DEV)
    x[0] = 1
    for name, qs, ps in gates:
        if name == "unitary":
            _apply64(x, n, ps[0], qs)
        elif name == "h":
            _apply64(x, n, np.array([[1, 1], [1, -1]]) / math.sqrt(2), qs)
        elif name == "ry":
            c, s = math.cos(ps[0] / 2), math.sin(ps[0] / 2)
            _apply64(x, n, [[c, -s], [s, c]], qs)
        elif name == "rz":
            _apply64(x, n, np.diag(np.exp([-0.5j * ps[0], 0.5j * ps[0]])), qs)
        elif name == "cp":
            _apply64(x, n, np.diag([1, np.exp(1j * ps[0])]), qs[1:], qs[:1])
        elif name == "swap":
            _apply64(x, n, _SWAP, qs)
        else:  # cx, mcx
            _apply64(x, n, _X, qs[-1:], qs[:-1])
    return x


def _signs(n, z):
    i = torch.arange(1 << n, device=DEV) & z
    for s in (16, 8, 4, 2, 1):
        i = i ^ (i >> s)
    return (1 - 2 * (i & 1)).to(torch.float64)


def _pauli_terms(terms, n):
    """[(x mask, z mask, coefficient i^y)] of labelled Pauli terms."""
    out = []
    for lab, c in terms:
        x = sum(1 << q for q, ch in enumerate(reversed(lab)) if ch in "XY")
        z = sum(1 << q for q, ch in enumerate(reversed(lab)) if ch in "ZY")
        out.append((x, z, c * 1j ** bin(x & z).count("1")))
    return out


def _groups64(terms, n):
    """x mask -> per-amplitude weight w: (H v)[i ^ x] = w[i] v[i], summed over x."""
    groups = {}
    for x, z, c in _pauli_terms(terms, n):
        w = _signs(n, z).to(torch.complex128) * complex(c)
        groups[x] = groups[x] + w if x in groups else w
    return groups


def _ham64(groups, v):
    out = torch.zeros_like(v)
    i = torch.arange(v.shape[-1], device=DEV)
    for x, w in groups.items():
        out += (v * w).index_select(-1, i ^ x)
    return out


def _evolve64(terms, n, v, t):
    bound = sum(abs(c) for _, c in terms)
    a = bound * t
    k = int(a + 40 + 2 * a ** (1 / 3))
    # Bessel coefficients by the periodic trapezoid rule of their integral
    tau = np.arange(4096) * (2 * math.pi / 4096)
    jk = np.array([np.mean(np.cos(m * tau - a * np.sin(tau))) for m in range(k + 1)])
    groups = {x: w / bound for x, w in _groups64(terms, n).items()}
    t0, t1 = v, _ham64(groups, v)
    out = jk[0] * t0 + (2 * (-1j) * jk[1]) * t1
    for m in range(2, k + 1):
        t0, t1 = t1, 2 * _ham64(groups, t1) - t0
        out += complex(2 * (-1j) ** (m % 4) * jk[m]) * t1
    return out


def exact(case, seed):
    kind = case["kind"]
    if kind == "circuit":
        x = _run64(case["n"], _gate_list(case, seed))
        return x.cpu().numpy() if case["host"] else x
    if kind == "gates":
        x = _state(case["n"], seed).to(torch.complex128)
        for fn, m, ctl, tg in _api_gates(case["n"], case["shift"], seed):
            if fn == "apply_gate_2q":
                # row index 2 * bit(larger qubit) + bit(smaller qubit)
                _apply64(x, case["n"], m, sorted(tg))
            elif fn == "apply_mcswap":
                _apply64(x, case["n"], _SWAP, tg, ctl)
            elif fn == "apply_mcx":
                _apply64(x, case["n"], _X, tg, ctl)
            elif fn == "apply_diagonal":
                _apply64(x, case["n"], np.diag(m), tg)
            elif fn == "apply_diagonal_phase":
                _apply64(x, case["n"], np.diag([1, m]), tg)
            else:
                _apply64(x, case["n"], m, tg, ctl)
        return x
    if kind == "evolve":
        n, r = case["n"], case["rhs"]
        x = _state(n, seed, None if r == 1 else r).to(torch.complex128)
        return _evolve64(_chain(n, seed), n, x, case["t"])
    if kind == "observe":
        n = case["n"]
        v = _state(n, seed).to(torch.complex128)
        i = torch.arange(1 << n, device=DEV)
        e = 0.0
        for x, z, c in _pauli_terms(_chain(n, seed), n):
            e += (complex(c) * torch.vdot(v, (v * _signs(n, z)).index_select(0, i ^ x))).real.item()
        return {"energy": e, "shots": None}
    return [_run64(n, [("unitary", [int(a), int(b)], [u]) for (a, b), u in zip(pairs, us)]).cpu().numpy()
            for n, pairs, us in _serve_plan(case, seed)]
