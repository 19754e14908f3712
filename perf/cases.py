"""The work this engine is used for, as cases that can be timed and checked.

A case is a circuit (or a batch of circuits, or an OpenQASM program) of a
stated family and size, run through the public Python binding as a program
would run it: rho reset to |0..0><0..0|, one run of the uploaded circuit, and
the results the program reads -- the whole rho where it is small, else the
outcome distribution, every <Z> and a set of entries gathered on the device
(4^n entries of a 14-qubit rho are 4.3 GB; programs do not copy that out).

Families
  mixed      gates uniform over H, X, Y, Z, S, T, RX, RY, RZ, U3, CX, CZ, SWAP
  brickwall  layers of Haar-random SU(4) on neighbours, then U3 and CX gates
  fusion     70 % U3, 30 % CX, RZZ, CU1 on random pairs
  hea        hardware-efficient ansatz: RY, RZ on every qubit, a CX ladder
  uccsd      exponentials of Pauli strings: basis changes, CX ladder, RZ, back
  structured basis state, QFT, CCX/C3X/C4X/CSWAP block, inverse QFT
`noise` > 0 adds a channel on each operand after every gate: depolarizing of
that probability after a gate on two qubits, amplitude damping after one on
a single qubit.
"""
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "dm-sim_amd"))

import costdata  # noqa: E402
import dmsim_amd as dm  # noqa: E402
import workloads as W  # noqa: E402

METHODS = {"plain": dm.METHOD_PLAIN, "plain_launch": dm.METHOD_PLAIN_LAUNCH,
           "fused": dm.METHOD_FUSED}
WHOLE_RHO = 9     # up to this many qubits a program reads all of rho
ENTRIES = 4096    # entries gathered above
SHOTS = 1000


def circuit(name, family, n, size, method="plain", learned=False, max_k=4, noise=0.0):
    """size: gates (mixed, fusion, brickwall's tail), layers (hea) or Pauli
    strings (uccsd); structured circuits have one size per n."""
    c = {"kind": "circuit", "family": family, "n": n, "size": size, "method": method,
         "learned": learned, "max_k": max_k, "noise": noise}
    return dict(c, name=name) if name else c


def batch(name, circuits, n_lo, n_hi, depth_lo, depth_hi):
    c = {"kind": "batch", "circuits": circuits, "n_lo": n_lo, "n_hi": n_hi,
         "depth_lo": depth_lo, "depth_hi": depth_hi}
    return dict(c, name=name) if name else c


def program(name, n, gates):
    c = {"kind": "program", "n": n, "gates": gates}
    return dict(c, name=name) if name else c


def listed():
    return [
        # A small circuit on a new user's settings (the default method): the
        # smallest call, all latency.
        circuit("plain_mixed_n6", "mixed", 6, 200),
        # A chemistry ansatz through the default method, the size of the
        # VQE-UCCSD circuits people first try.
        circuit("plain_uccsd_n8", "uccsd", 8, 60),
        # The default method at an odd middle size and near the largest that
        # is run gate by gate.
        circuit("plain_mixed_n11", "mixed", 11, 600),
        circuit("plain_brickwall_n13", "brickwall", 13, 120),
        # A .qasm file from text to shots, planning included: what qasm_run.py
        # does for one program.
        program("program_n9", 9, 20),
        # The same ansatz through the fused method with the shipped model: one
        # evaluation of a VQE loop.
        circuit("fused_uccsd_n8", "uccsd", 8, 60, "fused", True),
        # A middle-sized unitary circuit with the fused method's own settings.
        circuit("fused_mixed_n11", "mixed", 11, 601, "fused"),
        # Device-noise studies, what a density matrix is for: a small
        # variational circuit, and a random circuit at a size that fills the
        # GPU, a channel after every gate.
        circuit("noisy_hea_n8", "hea", 8, 6, "fused", False, 4, 0.01),
        circuit("noisy_brickwall_n12", "brickwall", 12, 40, "fused", True, 4, 0.002),
        # The benchmark's circuit: 20 layers of SU(4) and 2000 U3/CX gates.
        circuit("fused_brickwall_n14", "brickwall", 14, 2000, "fused", True),
        # An arithmetic circuit with five-qubit gates at the largest size that
        # several simulations share a GPU with.
        circuit("structured_n15", "structured", 15, 0, "fused", True, 5),
        # A variational sweep: many ansatz circuits of uneven width and depth
        # and their Pauli energies.
        batch("batch_hea_6_11", 96, 6, 11, 10, 40),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["plain", "plain", "fused", "fused", "noisy", "noisy", "batch", "program"])
    if kind == "program":
        return program(None, rng.randint(5, 11), _log_int(rng, 5, 60))
    if kind == "batch":
        lo = rng.randint(5, 8)
        return batch(None, _log_int(rng, 6, 96), lo, rng.randint(lo + 1, 11), rng.randint(3, 10),
                     rng.randint(11, 40))
    if kind == "plain":
        n = rng.randint(5, 13)
        family = rng.choice(["mixed", "brickwall", "fusion", "hea", "uccsd"])
        top = 1500 if n <= 9 else 600 if n <= 11 else 300 if n == 12 else 100
        gates, noise = _log_int(rng, 40, top), 0.0
    elif kind == "fused":
        n = rng.randint(5, 15)
        family = rng.choice(["mixed", "brickwall", "fusion", "hea", "uccsd", "structured"])
        if family == "structured":
            n = max(n, 6)
        gates, noise = _log_int(rng, 100, 2000 if n <= 13 else 1500 if n == 14 else 400), 0.0
    else:
        n = rng.randint(5, 12)
        family = rng.choice(["mixed", "brickwall", "hea", "uccsd"])
        gates, noise = _log_int(rng, 30, 400 if n <= 10 else 150), rng.choice([0.001, 0.004, 0.02])
    if family == "hea":
        size = max(1, gates // (3 * n))
    elif family == "uccsd":
        size = max(1, gates // (2 * n))
    else:
        size = gates
    fused = kind == "fused" or (kind == "noisy" and rng.random() < 0.8)
    return circuit(None, family, n, size, "fused" if fused else "plain",
                   fused and rng.random() < 0.5, 4, noise)


# ---- circuits --------------------------------------------------------------


def _uccsd(n, strings, rng):
    """exp(i theta P) for random Pauli strings P on 2 or 4 qubits (all of them
    between the first and the last carry the CX ladder, as in the
    Jordan-Wigner form)."""
    t = W.GateTable(n)
    for q in range(n // 2):
        t.add("X", [q])
    for _ in range(strings):
        k = 4 if n >= 4 and rng.uniform() < 0.7 else 2
        ends = sorted(int(q) for q in rng.choice(n, size=k, replace=False))
        span = sorted(set(ends) | set(range(ends[0], ends[1])) | set(range(ends[-2], ends[-1])))
        basis = [(q, "XY"[int(rng.integers(2))]) for q in ends]
        for q, b in basis:
            if b == "X":
                t.add("H", [q])
            else:
                t.add("RX", [q], [math.pi / 2])
        for a, b in zip(span, span[1:]):
            t.add("CX", [a, b])
        t.add("RZ", [span[-1]], [float(rng.uniform(-1, 1))])
        for a, b in reversed(list(zip(span, span[1:]))):
            t.add("CX", [a, b])
        for q, b in basis:
            if b == "X":
                t.add("H", [q])
            else:
                t.add("RX", [q], [-math.pi / 2])
    return t


def _table(case, seed):
    n, size, family = case["n"], case["size"], case["family"]
    if family == "mixed":
        return W.random_mixed(n, size, seed)
    if family == "brickwall":
        layers = 20 if size >= 1000 else 4
        return W.brickwall_su4(n=n, layers=layers, tail=size, seed=seed)
    if family == "fusion":
        return W.fusion_mix(n=n, n_gates=size, seed=seed)
    rng = np.random.default_rng(seed)
    if family == "hea":
        return W.hea_circuit(n, size, rng)
    if family == "uccsd":
        return _uccsd(n, size, rng)
    return W.structured(n=n, seed=seed)


def _steps(case, seed):
    """The circuit as its program appends it: ("gate", row) and
    ("kraus", qubit, operators) in order."""
    t = _table(case, seed)
    out = []
    for g in range(len(t)):
        out.append(("gate", g))
        if case["noise"] > 0:
            k = W.ARITY[W.OP_NAMES[t.ops[g]]]
            ops = (dm.depolarizing(case["noise"]) if k > 1 else
                   dm.amplitude_damping(case["noise"]))
            out += [("kraus", int(q), ops) for q in t.qbs[g][:k]]
    return t, out


def _qasm(case, seed):
    """A QFT-based arithmetic program as text."""
    n = case["n"]
    rng = np.random.default_rng(seed)
    lines = ['OPENQASM 2.0;', 'include "qelib1.inc";', f"qreg q[{n}];", f"creg c[{n}];"]
    lines += [f"x q[{q}];" for q in range(n) if rng.integers(2)]
    qft = []
    for j in range(n):
        qft.append(("h", j, 0, 0))
        qft += [("cu1", k, j, math.pi / (1 << (k - j))) for k in range(j + 1, n)]

    def emit(seq, sign):
        for op, a, b, ang in seq:
            lines.append(f"h q[{a}];" if op == "h" else
                         f"cu1({sign * ang!r}) q[{a}],q[{b}];")

    emit(qft, 1)
    for _ in range(case["gates"]):
        a, b, c = (int(x) for x in rng.choice(n, size=3, replace=False))
        r = rng.uniform()
        if r < 0.4:
            lines.append(f"rz({float(rng.uniform(-3, 3))!r}) q[{a}];")
        elif r < 0.6:
            lines.append(f"u3({float(rng.uniform(0, 3))!r},{float(rng.uniform(-3, 3))!r},"
                         f"{float(rng.uniform(-3, 3))!r}) q[{a}];")
        elif r < 0.8:
            lines.append(f"cx q[{a}],q[{b}];")
        else:
            lines.append(f"ccx q[{a}],q[{b}],q[{c}];")
    emit(list(reversed(qft)), -1)
    lines += [f"measure q[{q}] -> c[{q}];" for q in range(n)]
    return "\n".join(lines) + "\n"


def _batch(case, seed):
    return W.hea_batch(n_circuits=case["circuits"], seed=seed,
                       n_range=(case["n_lo"], case["n_hi"]),
                       depth_range=(case["depth_lo"], case["depth_hi"]))


def _entries(case, seed):
    return np.random.default_rng(seed + 77).integers(0, 4 ** case["n"], size=ENTRIES,
                                                     dtype=np.uint64)


_MODEL = []


def _model():
    """The shipped cost model, loaded once as a program does."""
    if not _MODEL:
        _MODEL.append(costdata.default_model())
    return _MODEL[0]


def prepare(case, seed):
    if case["kind"] == "program":
        return {"case": case, "source": _qasm(case, seed), "shot_seed": seed & 0xFFFF}
    if case["kind"] == "batch":
        b = dm.Batch()
        for circ, strings, weights in _batch(case, seed):
            b.add_circuit(circ, strings, weights)
        b.upload()
        return {"case": case, "batch": b}
    t, steps = _steps(case, seed)
    s = dm.Sim(case["n"])
    s.set_method(METHODS[case["method"]])
    if case["method"] == "fused":
        s.set_fusion_max_k(case["max_k"])
        if case["learned"]:
            s.set_cost_model(_model())
    if case["noise"] > 0:
        for st in steps:
            if st[0] == "gate":
                s.append_table(t.take([st[1]]))
            else:
                s.append_kraus(st[1], st[2])
    else:
        s.append_table(t)
    s.upload()
    return {"case": case, "sim": s, "entries": _entries(case, seed)}


def run(state):
    case = state["case"]
    if case["kind"] == "program":
        n, _, _, _ = dm.qasm_parse(state["source"])
        with dm.Sim(n) as s:
            s.set_method(dm.METHOD_FUSED)
            s.append_qasm(state["source"])
            s.upload()
            s.run()
            shots, total = s.measure(SHOTS, state["shot_seed"])
            return {"shots": shots, "total": total, "diag": s.get_diag()}
    if case["kind"] == "batch":
        state["batch"].run()
        return {"energies": state["batch"].energies()}
    s = state["sim"]
    s.reset_dm()
    s.run()
    if case["n"] <= WHOLE_RHO:
        re, im = s.get_dm()
        return {"re": re, "im": im, "z": s.expect_z()}
    return {"diag": s.get_diag(), "z": s.expect_z(), "entries": s.get_entries(state["entries"])}


# ---- the work and the values ------------------------------------------------


def _work(n, steps_k):
    """rho read once and written once; per gate the multiplications its matrix
    needs on both sides of one triangle of rho (a k-qubit dense matrix:
    2^k complex products an entry and side; X, CX, SWAP and the like move
    entries only)."""
    flops = 0.0
    for k in steps_k:
        flops += 2 * 0.5 * 4.0 ** n * 8 * (1 << k)
    return {"bytes": 32.0 * 4 ** n, "flops": flops}


_MOVES = {"X", "CX", "SWAP", "ID", "CCX", "CSWAP", "C3X"}


def _dense(table):
    return [min(W.ARITY[W.OP_NAMES[o]], 2) for o in table.ops if W.OP_NAMES[o] not in _MOVES]


def work(case):
    if case["kind"] == "program":
        n = case["n"]
        return _work(n, [1] * (2 * n) + [2] * (n * (n - 1)) + [1] * (case["gates"] * 6 // 10))
    if case["kind"] == "batch":
        total = {"bytes": 0.0, "flops": 0.0}
        for circ, strings, _ in _batch(case, 1):
            w = _work(circ.n_qubits, _dense(circ))
            total["bytes"] += w["bytes"]
            total["flops"] += w["flops"]
        return total
    t, steps = _steps(case, 1)
    w = _work(case["n"], _dense(t))
    channels = sum(1 for s in steps if s[0] == "kraus")
    w["flops"] += channels * 0.5 * 4.0 ** case["n"] * 8 * 4  # 4 x 4 on each quad
    return w


def _c(name):
    """Textbook 2x2 matrices by gate name."""
    s = 1 / math.sqrt(2)
    return {"H": [[s, s], [s, -s]], "X": [[0, 1], [1, 0]], "Y": [[0, -1j], [1j, 0]],
            "Z": [[1, 0], [0, -1]], "S": [[1, 0], [0, 1j]],
            "T": [[1, 0], [0, complex(s, s)]]}[name]


def _u3(th, ph, lam):
    c, s = math.cos(th / 2), math.sin(th / 2)
    e = lambda x: complex(math.cos(x), math.sin(x))
    return [[c, -e(lam) * s], [e(ph) * s, e(ph + lam) * c]]


def _phase(ang):
    return [[1, 0], [0, complex(math.cos(ang), math.sin(ang))]]


def _controlled(k, m):
    """m (2x2) on the lowest bit, k controls above it."""
    u = np.eye(2 << k, dtype=complex)
    u[-2:, -2:] = np.asarray(m)
    return u


def _gates_of(name, qb, prm, coef):
    """A gate as (qubits, matrix) pairs; qubits[0] is the matrix's high bit."""
    th, ph, lam = prm
    q = [int(x) for x in qb[:W.ARITY[name]]]
    if name in ("H", "X", "Y", "Z", "S", "T"):
        return [(q, _c(name))]
    if name in ("RX", "RY"):
        c, s = math.cos(th / 2), math.sin(th / 2)
        return [(q, [[c, -1j * s], [-1j * s, c]] if name == "RX" else [[c, -s], [s, c]])]
    if name == "RZ":
        return [(q, _phase(ph))]
    if name == "U3":
        return [(q, _u3(th, ph, lam))]
    if name == "CX":
        return [(q, _controlled(1, _c("X")))]
    if name == "CZ":
        return [(q, _controlled(1, _c("Z")))]
    if name == "SWAP":
        return [(q, np.eye(4)[[0, 2, 1, 3]])]
    if name == "CU1":
        return [(q, _controlled(1, _phase(lam)))]
    if name == "RZZ":
        e = complex(math.cos(th), math.sin(th))
        return [(q, np.diag([1, e, e, 1]))]
    if name == "CCX":
        return [(q, _controlled(2, _c("X")))]
    if name == "C3X":
        return [(q, _controlled(3, _c("X")))]
    if name == "CSWAP":  # the first operand is the control
        return [(q, np.kron([[1, 0], [0, 0]], np.eye(4)) +
                 np.kron([[0, 0], [0, 1]], np.eye(4)[[0, 2, 1, 3]]))]
    if name == "C4X":  # the sequence the gate set defines it by
        a, b, c, d, e = q
        h = lambda x: ([x], _c("H"))
        cu = lambda ang: ([d, e], _controlled(1, _phase(ang)))
        c3x = ([a, b, c, d], _controlled(3, _c("X")))
        return ([h(e), cu(-math.pi / 2), h(e), c3x, h(d), cu(math.pi / 4), h(d), c3x] +
                _root3(math.pi / 8, a, b, c, e))
    if name in ("C1", "C2"):
        d = 1 << len(q)
        return [(q, (coef[0:2 * d * d:2] + 1j * coef[1:2 * d * d:2]).reshape(d, d))]
    raise ValueError(name)


def _root3(ang, a, b, c, d):
    """The gate set's C3SQRTX: a ladder of seven controlled phases."""
    ctl, sgn = [a, b, b, c, c, c, c], [-1, 1, -1, 1, -1, 1, -1]
    cx = [(a, b), (a, b), (b, c), (a, c), (b, c), (a, c)]
    out = []
    for i in range(7):
        out += [([d], _c("H")), ([ctl[i], d], _controlled(1, _phase(sgn[i] * ang))),
                ([d], _c("H"))]
        if i < 6:
            out.append((list(cx[i]), _controlled(1, _c("X"))))
    return out


def _apply(v, n, qubits, m):
    """m on `qubits` of a state of n bits (numpy or torch); axis 0 of the
    reshaped state is bit n - 1."""
    k = len(qubits)
    axes = [n - 1 - q for q in qubits]
    if isinstance(v, np.ndarray):
        m = np.asarray(m, dtype=complex).reshape([2] * (2 * k))
        v = np.tensordot(m, v.reshape([2] * n), (list(range(k, 2 * k)), axes))
        return np.ascontiguousarray(np.moveaxis(v, list(range(k)), axes)).reshape(-1)
    m = torch.as_tensor(np.asarray(m, dtype=complex), device=v.device).reshape([2] * (2 * k))
    v = torch.tensordot(m, v.reshape([2] * n), (list(range(k, 2 * k)), axes))
    return torch.movedim(v, list(range(k)), axes).reshape(-1)


def _gates(t):
    for g in range(len(t)):
        yield from _gates_of(W.OP_NAMES[t.ops[g]], t.qbs[g], t.prms[g], t.coefs[g])


def _state(t):
    v = np.zeros(1 << t.n_qubits, dtype=complex)
    v[0] = 1
    for q, m in _gates(t):
        v = _apply(v, t.n_qubits, q, m)
    return v


def _density(case, seed):
    """rho of a noisy circuit as a state of 2n bits: row bits n.., column bits 0.."""
    t, steps = _steps(case, seed)
    n = case["n"]
    v = torch.zeros(4 ** n, dtype=torch.complex128,
                    device="cuda" if torch.cuda.is_available() else "cpu")
    v[0] = 1
    for st in steps:
        if st[0] == "gate":
            g = st[1]
            for q, m in _gates_of(W.OP_NAMES[t.ops[g]], t.qbs[g], t.prms[g], t.coefs[g]):
                m = np.asarray(m, dtype=complex)
                v = _apply(v, 2 * n, [x + n for x in q], m)
                v = _apply(v, 2 * n, list(q), m.conj())
        else:
            sup = sum(np.kron(np.asarray(k, dtype=complex), np.asarray(k, dtype=complex).conj())
                      for k in st[2])
            v = _apply(v, 2 * n, [st[1] + n, st[1]], sup)
    return v


def _z(diag, n):
    i = np.arange(1 << n)
    return np.array([np.sum(np.where((i >> q) & 1, -diag, diag)) for q in range(n)])


def _program_state(case, seed):
    """The program's gates read back from its text (one statement a line)."""
    n = case["n"]
    v = np.zeros(1 << n, dtype=complex)
    v[0] = 1
    for line in _qasm(case, seed).splitlines():
        op, _, rest = line.rstrip(";").partition(" ")
        name, _, args = op.partition("(")
        if name not in ("x", "h", "cu1", "rz", "u3", "cx", "ccx"):
            continue
        p = [float(x) for x in args.rstrip(")").split(",")] if args else []
        q = [int(x[2:-1]) for x in rest.split(",")]
        m = {"x": lambda: _c("X"), "h": lambda: _c("H"), "rz": lambda: _phase(p[0]),
             "cu1": lambda: _controlled(1, _phase(p[0])), "u3": lambda: _u3(*p),
             "cx": lambda: _controlled(1, _c("X")), "ccx": lambda: _controlled(2, _c("X"))}[name]()
        v = _apply(v, n, q, m)
    return v


def exact(case, seed):
    if case["kind"] == "program":
        p = np.abs(_program_state(case, seed)) ** 2
        return {"shots": None, "total": 1.0, "diag": p}
    if case["kind"] == "batch":
        out = []
        for circ, strings, weights in _batch(case, seed):
            v, e = _state(circ), 0.0
            for s, w in zip(strings, weights):
                u = v
                for q, ch in enumerate(s):
                    if ch != "I":
                        u = _apply(u, circ.n_qubits, [q], _c(ch))
                e += w * np.vdot(v, u).real
            out.append(e)
        return {"energies": np.array(out)}
    n = case["n"]
    dim = 1 << n
    # the engine holds conj(rho)
    if case["noise"] > 0:
        rho = np.conj(_density(case, seed).cpu().numpy())
        diag = rho[:: dim + 1].real.copy()
        at = lambda i: rho[i]
    else:
        v = _state(_table(case, seed))
        diag = np.abs(v) ** 2
        at = lambda i: np.conj(v[i // dim]) * v[i % dim]
    if n <= WHOLE_RHO:
        rho = at(np.arange(dim * dim))
        return {"re": rho.real.copy(), "im": rho.imag.copy(), "z": _z(diag, n)}
    return {"diag": diag, "z": _z(diag, n), "entries": at(_entries(case, seed).astype(np.int64))}
