"""A batch's block sweeps, which dmx_batch_set_hermitian asks for: groups of circuits, waves
and graph replays on the paths that batches take without resident rows."""
import numpy as np
import pytest

import workloads as W

pytestmark = pytest.mark.gpu

BUDGETS = (0, 16 << 20, 32 << 20, 64 << 20, 128 << 20)


def _items(seed, widths, layers):
    rng = np.random.default_rng(seed)
    out = []
    for n in widths:
        strings, weights = W.random_paulis(n, 6, rng)
        out.append((W.hea_circuit(n, int(rng.integers(*layers)), rng), strings, weights))
    return out


def _batch(items, herm, budget=None, limit=0, graph=True):
    import dmsim_amd as dm
    b = dm.Batch()
    b.set_hermitian(herm)
    b.set_pool_limit(limit)
    if budget is not None:
        b.set_group_bytes(budget)
    for circ, strings, weights in items:
        b.add_circuit(circ, strings, weights)
    b.upload()
    b.set_graph(graph)
    b.run()
    return b


def _single_run(circ, herm):
    """rho of the circuit alone, as the batch runs it."""
    import dmsim_amd as dm
    s = dm.Sim(circ.n_qubits)
    s.set_method(dm.METHOD_FUSED)
    s.set_fusion_hermitian(2 if herm and circ.n_qubits >= 10 else 0)
    s.append_table(circ)
    s.upload()
    s.run()
    blocks = s.last_run_stats()["launches"]
    rho = s.get_dm()
    s.close()
    return blocks, rho


@pytest.mark.parametrize("herm", [False, True])
def test_groups_and_timed_schedule(herm):
    """Whole waves, groups of 1 MiB and the timed schedule: the same bits, with a launch per
    block step and width (the deepest circuit's blocks at least)."""
    items = _items(77, (6, 10, 8, 9, 10, 7, 10, 8, 6, 9), (4, 9))
    whole, grouped, timed = (_batch(items, herm, b) for b in (0, 1 << 20, None))
    deepest = max(_single_run(c, herm)[0] for c, _, _ in items)
    assert whole.stats()["launches"] >= deepest > 3
    assert whole.schedule() == {"group_bytes": 0, "groups": 1}
    assert grouped.schedule()["group_bytes"] == 1 << 20 and grouped.schedule()["groups"] > 4
    st = timed.schedule()
    groups, held = 1, 0  # consecutive circuits, the largest first, as many as fit
    for need in sorted((16 << 2 * c.n_qubits for c, _, _ in items), reverse=True):
        if st["group_bytes"] and held and held + need > st["group_bytes"]:
            groups, held = groups + 1, 0
        held += need
    assert st["group_bytes"] in BUDGETS and st["groups"] == groups
    widths = {n: timed.tile_bits(n) for n in (6, 7, 8, 9)}
    assert all(5 <= m <= min(8, n) for n, m in widths.items())
    for other in (grouped, timed):
        assert np.array_equal(whole.energies(), other.energies())
        for cid in range(len(items)):
            a, b = whole.get_dm(cid), other.get_dm(cid)
            assert np.array_equal(a[0], b[0]) and np.array_equal(a[1], b[1]), cid
    for b in (whole, grouped, timed):
        b.close()


@pytest.mark.parametrize("herm", [False, True])
def test_waves_and_replays(oracle, herm):
    """One wave, several by a pool limit, and eager launches: the same energies and
    diagonals over several replays with other work between; rho as alone."""
    import dmsim_amd as dm
    items = _items(1011, (10, 8, 11, 6, 10, 9, 11, 7, 4), (3, 8))
    one, many = _batch(items, herm), _batch(items, herm, limit=16 << 22)
    eager = _batch(items, herm, graph=False)
    assert one.waves() == 1 and many.waves() > 2
    for _ in range(3):
        for b in (many, eager):
            assert np.array_equal(one.energies(), b.energies())
            for cid, (circ, _, _) in enumerate(items):
                assert np.array_equal(one.get_diag(cid), b.get_diag(cid)), cid
        s = dm.Sim(5)
        s.append(W.OP["H"], [0])
        s.upload()
        s.run()
        s.get_dm()
        s.close()
        for b in (one, many, eager):
            b.run()
    for cid, (circ, _, _) in enumerate(items):
        psi = oracle.sv(circ.n_qubits, circ.arrays())
        assert np.max(np.abs(one.get_diag(cid) - np.abs(psi) ** 2)) <= 1e-10
        got, want = one.get_dm(cid), _single_run(circ, herm)[1]
        assert np.array_equal(got[0], want[0]) and np.array_equal(got[1], want[1]), cid
    for b in (one, many, eager):
        b.close()
