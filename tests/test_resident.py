"""Fused blocks on resident rows of rho (csrc/resident.hpp, resident.hip)."""
import os
import shutil
import subprocess

import numpy as np
import pytest

import workloads as W
from conftest import ROOT

TOL = 1e-12


def test_resident_records(tmp_path):
    """Places and permutations of every block on the CPU, n = 4..11
    (tests/cpp/resident_places.cpp)."""
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("hipcc not found")
    exe = os.path.join(str(tmp_path), "resident_places")
    pkg = os.path.join(ROOT, "dm-sim_amd")
    r = subprocess.run([hipcc, "-std=c++17", "-O2", "-I", os.path.join(pkg, "csrc"),
                        os.path.join(ROOT, "tests", "cpp", "resident_places.cpp"), "-L", pkg,
                        "-ldmsim_amd", f"-Wl,-rpath,{pkg}", "-o", exe],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout.strip() == "24 cases OK", r.stdout


@pytest.mark.gpu
@pytest.mark.parametrize("n", list(range(4, 12)))
@pytest.mark.parametrize("first", [0, 1])
def test_resident_runs_match_plain(n, first):
    """Against the plain method: a first run, graph replays (from 10 qubits rho's
    orientation alternates), and, first = 1, from the orientation the launches
    of one primitive each leave."""
    import dmsim_amd as dm
    t = W.random_mixed(n, 150, 300 + n, gate_set=[g for g in W.OP_NAMES if W.ARITY[g] <= 4
                                                  and g not in ("SRN", "R")])
    ref, s = dm.Sim(n), dm.Sim(n)
    for x in (ref, s):
        x.append_table(t)
        x.set_method(1)
        x.upload()
        if first:
            x.run()
    s.set_method(dm.METHOD_FUSED)
    idx = np.random.default_rng(n).integers(0, 4 ** n, size=512, dtype=np.uint64)
    for step in range(3):
        ref.run()
        s.run()
        assert s.last_run_stats()["launches"] <= 3
        want, got = ref.get_entries(idx), s.get_entries(idx)
        assert max(np.abs(got[i] - want[i]).max() for i in (0, 1)) <= TOL, step
        assert np.abs(s.get_diag() - ref.get_diag()).max() <= TOL, step
        if step == 1:  # returns rho to the reference's orientation
            want, got = ref.get_dm(), s.get_dm()
            assert max(np.abs(got[i] - want[i]).max() for i in (0, 1)) <= TOL
    s.set_profiling(True)
    s.run()
    assert s.profile()["k_resident"]["calls"] == 2


@pytest.mark.gpu
def test_resident_batch_equals_single_runs():
    """Batched circuits of uneven width and depth against each circuit's own
    run (its result in the same orientation), bit for bit, in one wave and, by a pool
    limit, in several."""
    import dmsim_amd as dm
    rng = np.random.default_rng(5)
    items = []
    for n in (4, 11, 6, 8, 9, 10, 7, 5, 9, 11):
        strings, weights = W.random_paulis(n, 4, rng)
        items.append((W.hea_circuit(n, int(rng.integers(1, 9)), rng), strings, weights))
    diags = []
    for limit in (0, 16 << 22):
        b = dm.Batch()
        b.set_pool_limit(limit)
        for circ, strings, weights in items:
            b.add_circuit(circ, strings, weights)
        b.upload()
        b.run()
        b.run()
        diags.append([b.get_diag(i) for i in range(len(items))] + [b.energies()])
        if limit == 0:
            assert b.stats()["launches"] < 20
            for cid, (circ, _, _) in enumerate(items):
                s = dm.Sim(circ.n_qubits)
                s.set_method(dm.METHOD_FUSED)
                s.append_table(circ)
                s.upload()
                s.run()
                re, im = s.get_dm()
                bre, bim = b.get_dm(cid)
                if circ.n_qubits > 9:  # the batch leaves rho conj-transposed
                    d = 1 << circ.n_qubits
                    bre, bim = bre.reshape(d, d).T.ravel(), -bim.reshape(d, d).T.ravel()
                assert np.array_equal(re, bre) and np.array_equal(im, bim), cid
        b.close()
    for x, y in zip(*diags):
        assert np.array_equal(x, y)
