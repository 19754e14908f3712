"""Short circuits and short stretches of gates between channels: each runs the
cheaper of its forms, with the same results."""
import numpy as np
import pytest

import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 3, 6, 9, 10, 11, 13, 14])
def test_plain_segments_equal_one_launch_per_primitive(n):
    """The plain method on segments of one to twelve gates between channels, some on
    resident rows and some as sweeps, from both orientations, against one launch
    per primitive bit for bit."""
    import dmsim_amd as dm
    rng = np.random.default_rng(40 + n)
    names = [g for g in W.OP_NAMES if W.ARITY[g] <= min(n, 3)]
    sims = [dm.Sim(n) for _ in range(4)]
    for i, size in enumerate((1, 12, 1, 2, 1, 1, 12, 12, 3, 1)):
        t = W.random_mixed(n, size, 900 + 10 * n + i, gate_set=names)
        q = int(rng.integers(n))
        for s in sims:
            s.append_table(t)
            s.append_kraus(q, dm.amplitude_damping(0.07))
    idx = rng.integers(0, 4 ** n, size=4096, dtype=np.uint64)
    one, rows = dm.METHOD_PLAIN_LAUNCH, dm.METHOD_PLAIN
    for s, methods in zip(sims, ((rows, rows), (one, one), (one, rows), (rows, one))):
        s.upload()
        for m in methods:
            s.set_method(m)
            s.run()
    sims[0].set_profiling(True)
    sims[0].run()
    calls = sims[0].profile()
    assert "k_rows" in calls and any(c.startswith("k_sweep") for c in calls)
    sims[1].run()
    want = sims[1].get_entries(idx), sims[1].get_diag()
    assert np.array_equal(sims[0].get_entries(idx), want[0])
    assert np.array_equal(sims[0].get_diag(), want[1])
    for s in sims[2:]:
        s.run()  # the third run of each, in its last method
        assert np.array_equal(s.get_entries(idx), want[0])
        assert np.array_equal(s.get_diag(), want[1])


@pytest.mark.parametrize("n", [2, 9, 11, 13, 14])
def test_plain_short_segments_make_no_row_passes(n):
    """One dense gate, or two that touch half of the entries, as two launches a
    primitive; many gates on resident rows."""
    import dmsim_amd as dm
    for gates, launches in (([("H", [n - 1])], 2), ([("CX", [1, 0])], 2),
                            ([("T", [0]), ("CX", [0, n - 1])], 4), ([("H", [0])] * 12, 3)):
        t = W.GateTable(n)
        for name, q in gates:
            t.add(name, q)
        s = dm.Sim(n)
        s.append_table(t)
        s.upload()
        s.run()
        assert s.last_run_stats()["launches"] == launches, gates
        s.close()


@pytest.mark.parametrize("learned", [False, True])
@pytest.mark.parametrize("n", [5, 8, 9, 10, 11])
def test_fused_short_unitary_circuits_run_as_sweeps(n, learned):
    """A circuit of one or two blocks makes a sweep a block and keeps rho's orientation;
    deeper ones run on resident rows."""
    import costdata
    import dmsim_amd as dm
    model = costdata.default_model() if learned else None
    for gates, brief in ((1, True), (4, True), (200, False)):
        t = W.random_mixed(4, gates, 50 + n, gate_set=["H", "U3", "CX", "RZ"]) if brief else \
            W.random_mixed(n, gates, 50 + n, gate_set=["H", "U3", "CX", "RZ"])
        s, ref = dm.Sim(n), dm.Sim(n)
        for x in (s, ref):
            x.append_table(t)
        s.set_method(dm.METHOD_FUSED)
        if model is not None:
            s.set_cost_model(model)
        s.upload()
        ref.upload()
        s.set_profiling(True)
        for _ in range(2):
            s.run()
            ref.run()
            assert ("k_resident" in s.profile()) != brief, gates
            assert s.last_run_stats()["launches"] <= 3
            got, want = s.get_dm(), ref.get_dm()
            assert max(np.abs(got[i] - want[i]).max() for i in (0, 1)) <= 1e-12, gates
        if brief:
            info = s.plan_info()
            assert info["fused_blocks"] + info["plain_blocks"] == 1
            assert info["plain_blocks"] or s.last_run_stats()["launches"] == 1
        s.close()
        ref.close()
    if model is not None:
        model.close()


@pytest.mark.parametrize("n,gate,kernel", [(8, None, "k_quad"), (11, None, "k_quad"), (12, None, "k_quad"),
                                           (14, None, "k_quad"), (14, "C4X", "k_fused5")])
def test_a_lone_channel_or_wide_gate_runs_in_place(n, gate, kernel):
    """One launch in place, without a block or a group sweep around it."""
    import dmsim_amd as dm
    t = W.GateTable(n)
    for q in range(n):
        t.add("U3", [q], (0.3 + q, 0.2 * q, 0.7))
    ref, s = dm.Sim(n), dm.Sim(n)
    for x in (ref, s):  # a state first, then the circuit
        x.append_table(t)
        x.upload()
        x.run()
        x.clear_circuit()
        if gate:
            x.append(W.OP[gate], [0, 3, 5, 7, n - 1])
        else:
            x.append_kraus(n // 2, dm.amplitude_damping(0.3))
    s.set_method(dm.METHOD_FUSED)
    s.set_profiling(True)
    idx = np.random.default_rng(n).integers(0, 4 ** n, size=4096, dtype=np.uint64)
    for x in (ref, s):
        x.upload()
        x.run()
    assert list(s.profile()) == [kernel] and s.last_run_stats()["launches"] == 1
    assert np.abs(s.get_entries(idx) - ref.get_entries(idx)).max() <= 1e-12
    assert np.abs(s.get_diag() - ref.get_diag()).max() <= 1e-12


@pytest.mark.parametrize("n", [5, 6, 7, 8, 9])
def test_batched_column_passes_equal_single_runs(n):
    """Column passes of several columns to a chunk (7 to 9 qubits), more circuits than one,
    of uneven depth and beside other widths: bit for bit the circuits' own runs."""
    import dmsim_amd as dm
    rng = np.random.default_rng(n)
    widths = [n, n, 6, n, 8, n]
    circuits = [W.random_mixed(w, int(rng.integers(60, 300)), 20 * n + i,
                               gate_set=["H", "U3", "CX", "SWAP", "X", "RZZ", "CCX"])
                for i, w in enumerate(widths)]
    b = dm.Batch()
    for t in circuits:
        b.add_circuit(t)
    b.upload()
    for _ in range(2):
        b.run()
    for i, t in enumerate(circuits):
        s = dm.Sim(t.n_qubits)
        s.set_method(dm.METHOD_FUSED)
        s.append_table(t)
        s.upload()
        s.run()
        got, want = b.get_dm(i), s.get_dm()
        assert np.array_equal(got[0], want[0]) and np.array_equal(got[1], want[1]), i
        s.close()
    b.close()


def test_batched_short_circuits_equal_single_runs():
    """Circuits of one or two blocks beside deeper ones, 4 to 11 qubits, in one wave and in
    several: bit for bit the circuits' own runs, without a second pool of planes."""
    import dmsim_amd as dm
    rng = np.random.default_rng(8)
    circuits = []
    for n in range(4, 12):
        circuits.append(W.GateTable(n).add("RY", [n - 1], (0.7, 0, 0)))
        circuits.append(W.random_mixed(min(n, 6), 12, 60 + n, gate_set=["H", "CX", "U3", "SWAP", "X"]))
        circuits[-1].n_qubits = n
        circuits.append(W.hea_circuit(n, 5, rng))
    want = []
    for t in circuits:
        s = dm.Sim(t.n_qubits)
        s.set_method(dm.METHOD_FUSED)
        s.append_table(t)
        s.upload()
        s.run()
        want.append((s.get_diag(), *s.get_dm()))
        s.close()
    for limit in (0, 16 << 22):
        b = dm.Batch()
        b.set_pool_limit(limit)
        for t in circuits:
            b.add_circuit(t)
        b.upload()
        assert limit == 0 or b.waves() > 1
        for _ in range(3):
            b.run()
        for i, (diag, re, im) in enumerate(want):
            assert np.array_equal(b.get_diag(i), diag), i
            if limit == 0 and circuits[i].n_qubits < 10:
                got = b.get_dm(i)
                assert np.array_equal(got[0], re) and np.array_equal(got[1], im), i
        b.close()


@pytest.mark.parametrize("n", [9, 11])
def test_plan_info_counts_resident_blocks_once(n):
    """With a cost model, a block of one cheap gate counts as the fused block it runs as, and
    the predicted time is that of the blocks as fused sweeps."""
    import costdata
    import dmsim_amd as dm
    model = costdata.default_model()
    t = W.GateTable(n)
    for a in (0, 4):
        for g in W.random_mixed(4, 40, 3 + a, gate_set=["U3", "CX"]).qbs:
            t.add("U3", [a + g[0]], (0.3, 0.2, 0.1)) if g[0] == g[1] or g[1] >= 4 else \
                t.add("RYY", [a + g[0], a + g[1]], (0.4,))
    t.add("T", [8])
    s = dm.Sim(n)
    s.set_method(dm.METHOD_FUSED)
    s.set_cost_model(model)
    s.append_table(t)
    s.upload()
    s.set_profiling(True)
    s.run()
    assert s.profile()["k_resident"]["calls"] == 2
    info = s.plan_info()
    print(info, flush=True)
    assert info["plain_blocks"] == 0 and info["fused_blocks"] == 3
    assert sum(info["tiles"].values()) == info["fused_blocks"]
    model.close()
