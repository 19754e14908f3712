"""Group sweeps at the largest sizes they run at (csrc/group.hip)."""
import numpy as np
import pytest

import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [15, 16])
def test_noisy_product_state(n):
    """A rotation and a channel on every qubit and SWAPs between them, so that rho stays a
    product: sampled entries and the diagonal against the qubits' own 2 x 2 matrices.
    Entries are products of n factors, each rounded a few times: 1e-13 relative to the
    largest covers them many times over."""
    import dmsim_amd as dm
    rng = np.random.default_rng(n)
    s = dm.Sim(n)
    s.set_method(dm.METHOD_FUSED)
    rho = [np.diag([1.0 + 0j, 0.0])] * n
    channels = (dm.amplitude_damping(0.1), dm.depolarizing(0.05), dm.phase_damping(0.2))
    for layer in range(2):
        for q in rng.permutation(n):
            th, ph, lam = rng.uniform(0.2, 2.5, size=3)
            c, sn = np.cos(th / 2), np.sin(th / 2)
            u = np.array([[c, -np.exp(1j * lam) * sn],
                          [np.exp(1j * ph) * sn, np.exp(1j * (ph + lam)) * c]])
            ops = channels[int(rng.integers(3))]
            s.append_matrix([int(q)], u)
            s.append_kraus(int(q), ops)
            rho[q] = sum(k @ u @ rho[q] @ u.conj().T @ np.conj(k).T for k in ops)
        for _ in range(n // 3):
            a, b = (int(x) for x in rng.choice(n, size=2, replace=False))
            s.append(W.OP["SWAP"], [a, b])
            rho[a], rho[b] = rho[b], rho[a]
    s.upload()
    s.set_profiling(True)
    s.run()
    assert s.profile()["k_group"]["calls"] > 1
    idx = rng.integers(0, 4 ** n, size=1 << 16, dtype=np.uint64)
    want = np.ones(idx.size, dtype=complex)
    diag = np.ones(1 << n)
    for q in range(n):
        r = ((idx >> np.uint64(n + q)) & np.uint64(1)).astype(int)
        c = ((idx >> np.uint64(q)) & np.uint64(1)).astype(int)
        want *= np.conj(rho[q])[r, c]  # rho is held conjugated
        diag *= rho[q].diagonal().real[(np.arange(1 << n) >> q) & 1]
    biggest = diag.max()
    assert np.abs(s.get_entries(idx) - want).max() <= 1e-13 * biggest
    assert np.abs(s.get_diag() - diag).max() <= 1e-13 * biggest
    s.close()
