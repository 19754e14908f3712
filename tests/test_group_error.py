"""Rounding of one stage of a group sweep (csrc/group.hip) on a dense rho, against 80-bit
arithmetic.  A complex product can be four real ones, three combined after their sums, or three
chained through one sum; each is emulated here on the same operands, with fused
multiply-adds as the matrix cores do.  The block sweeps take three for unitaries and four
for channels, and a stage may be no further off than halfway from that form to the next
worse one (on random operands, RMS relative: 16 x 16 unitaries, both sides, 2.7e-16, 3.0e-16 and
3.5e-16; 32 x 32 3.8e-16, 4.1e-16 and 4.7e-16; a superoperator 1.4e-16, 2.0e-16 and 2.4e-16).
"""
import numpy as np
import pytest

import workloads as W

pytestmark = pytest.mark.gpu


def _unitary(rng, d):
    q, r = np.linalg.qr(rng.normal(size=(d, d)) + 1j * rng.normal(size=(d, d)))
    return q * (np.diag(r) / np.abs(np.diag(r)))


def _exact(rng):
    """A two-qubit unitary of entries +-1/2, +-i/2: products of such and of the channel
    below are exact in double precision."""
    h = np.array([[1, 1], [1, -1]])
    return np.diag(1j ** rng.integers(0, 4, size=4)) @ np.kron(h, h) / 2


def _chain(a, b, c):
    for k in range(a.shape[-1]):
        c = (a[..., :, k, None].astype(np.longdouble) * b[..., k, None, :] + c).astype(float)
    return c


def _product(form, a, b):
    """a b in double precision, as `form` takes it."""
    ar, ai, br, bi = a.real.copy(), a.imag.copy(), b.real.copy(), b.imag.copy()
    zero = np.zeros(np.broadcast_shapes(a.shape[:-2], b.shape[:-2]) + (a.shape[-2], b.shape[-1]))
    if form == "four":
        return _chain(-ai, bi, _chain(ar, br, zero)) + 1j * _chain(ai, br, _chain(ar, bi, zero))
    if form == "three":
        p, q, t = _chain(ar, br, zero), _chain(ai, bi, zero), _chain(ar + ai, br + bi, zero)
        return (p - q) + 1j * ((t - p) - q)
    t = _chain(ar, br + bi, zero)
    return _chain(-(ar + ai), bi, t) + 1j * _chain(ai - ar, br, t)


def _off(got, want):
    return float(np.linalg.norm(got.astype(np.clongdouble) - want) / np.linalg.norm(want))


FLIP = [np.eye(2) / 2] * 3 + [np.diag([0.5, -0.5])]  # phase flip of probability 1/4


# qubits of the gate, channels on; the wide gates are arbitrary
@pytest.mark.parametrize("n,qubits,noisy", [(12, [7, 2], [7, 2]), (12, [9, 0, 4, 11], [6]),
                                            (13, [1, 12, 5, 8, 3], [])])
def test_one_stage(n, qubits, noisy):
    import dmsim_amd as dm
    k = len(qubits)
    rng = np.random.default_rng(n + k)
    s = dm.Sim(n)
    s.append_table(W.random_mixed(n, 60, 5, gate_set=["U3", "CX", "RYY", "H", "U3"]))
    for q in range(n):
        s.append(W.OP["U3"], [q], 0.4 + q, 0.3 * q, 1.1)
        s.append_kraus(q, dm.amplitude_damping(0.2))
    s.upload()
    s.run()
    s.clear_circuit()
    # the sub-blocks of rho on the stage's qubits, the others' bits fixed at random
    act = sorted(set(qubits) | set(noisy))
    rest = [q for q in range(n) if q not in act]
    local = sum(((np.arange(1 << len(act)) >> i) & 1) << q for i, q in enumerate(act))
    other = [sum(int(b) << q for q, b in zip(rest, rng.integers(0, 2, size=len(rest))))
             for _ in range(64)]
    # above the diagonal: below it a Hermitian sweep reads the mirrored entries
    idx = np.concatenate([((min(r, c) + local)[:, None] * (1 << n) + (max(r, c) + local)[None, :])
                          .ravel() for r, c in zip(other[::2], other[1::2])
                          if r != c]).astype(np.uint64)
    d = 1 << len(act)
    before = s.get_entries(idx).reshape(-1, d, d).astype(np.clongdouble).conj()  # held conjugated
    u = _exact(rng) if k == 2 else _unitary(rng, 1 << k)
    s.set_method(dm.METHOD_FUSED)
    s.set_fusion_max_k(5 if k == 5 else 4)
    s.append_matrix(qubits, u)
    for q in noisy:
        s.append_kraus(q, FLIP)
    s.upload()
    s.set_profiling(True)
    s.run()
    assert s.profile()["k_group"]["calls"] == 1
    after = s.get_entries(idx).reshape(-1, d, d).astype(np.clongdouble).conj()
    full = np.zeros((d, d), dtype=np.clongdouble)  # the gate on the local index
    pos = [act.index(q) for q in qubits]
    sub = [sum(((x >> (k - 1 - i)) & 1) << p for i, p in enumerate(pos)) for x in range(1 << k)]
    for base in range(d):
        if base & sum(1 << p for p in pos):
            continue
        for i in range(1 << k):
            for j in range(1 << k):
                full[base | sub[i], base | sub[j]] = u[i, j]
    want = full @ before @ full.conj().T
    for q in noisy:
        z = np.array([1 - 2 * ((x >> act.index(q)) & 1) for x in range(d)])
        want = want * np.where(np.outer(z, z) > 0, np.longdouble(1), np.longdouble(0.5))
    off, t = {}, before.astype(complex)
    for form in ("four", "three", "chained"):
        if k == 2:  # one product with the superoperator
            sup = np.kron(full, full.conj()).astype(complex)
            for q in noisy:
                z = np.array([1 - 2 * ((x >> act.index(q)) & 1) for x in range(d)])
                sup = np.where(np.outer(z, z) > 0, 1.0, 0.5).reshape(-1, 1) * sup
            got = _product(form, sup, t.reshape(-1, d * d).T).T.reshape(-1, d, d)
            off[form] = _off(got, want)
        else:
            m = full.astype(complex)
            got = _product(form, m, _product(form, t, m.conj().T))
            off[form] = _off(got, full @ before @ full.conj().T)
    limit = (off["four"] * off["three"] if k == 2 else off["three"] * off["chained"]) ** 0.5
    here = _off(after, want)
    print(f"{k} qubits: {here:.3g}, limit {limit:.3g}, forms {off}", flush=True)
    assert here <= limit
