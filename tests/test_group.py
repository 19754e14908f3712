"""Hermitian group sweeps: several blocks on six qubits per sweep of rho
(csrc/group.hpp, group.hip, fuse.cpp build_group_plan)."""
import os
import shutil
import subprocess

import numpy as np
import pytest

import workloads as W
from conftest import ROOT


def test_group_maps_on_the_cpu(tmp_path):
    """Plans, schedules and index maps thread by thread against gate-by-gate
    application (tests/cpp/group_maps.cpp)."""
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("hipcc not found")
    exe = os.path.join(str(tmp_path), "group_maps")
    pkg = os.path.join(ROOT, "dm-sim_amd")
    r = subprocess.run([hipcc, "-std=c++17", "-O2", "-I", os.path.join(pkg, "csrc"), "-I",
                        os.path.join(ROOT, "include"),
                        os.path.join(ROOT, "tests", "cpp", "group_maps.cpp"), "-L", pkg,
                        "-ldmsim_amd", f"-Wl,-rpath,{pkg}", "-o", exe],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout.strip() == "10 cases OK", r.stdout


# Stage kinds: four-qubit unitaries, five-qubit ones (C4X), superoperators of
# pairs, and their mixtures; matrices past what LDS holds (many stages, or
# five-qubit ones); one gate; trailing index maps (X, CX, SWAP).  Sums of at most
# 1e3 products of unit-norm values per entry on values <= 1: 1e-12 is far above
# their rounding, the repository's 1e-10 bound is kept.
@pytest.mark.gpu
@pytest.mark.parametrize("n,gates,wide,noise", [(12, 60, False, 0.6), (12, 1, False, 1.0),
                                                (12, 60, True, 0.6), (13, 1, True, 0.0),
                                                (13, 80, True, 0.0), (13, 40, True, 0.3),
                                                (14, 30, True, 0.0), (14, 20, False, 0.5)])
def test_group_sweeps_match_plain(n, gates, wide, noise):
    """Against the plain method: two runs, the second after sweeps that leave rho
    conj-transposed."""
    import dmsim_amd as dm
    names = ["H", "X", "U3", "CX", "CX", "SWAP", "RZZ", "CCX", "C3X", "C2", "CU1"]
    t = W.random_mixed(n, gates, 800 + n + gates,
                       gate_set=["C4X"] if wide and gates == 1 else names + ["C4X"] * wide)

    def load(s):
        r = np.random.default_rng(n)
        for g in range(len(t)):
            s.append_table(t.take([g]))
            k = W.ARITY[W.OP_NAMES[t.ops[g]]]
            for q in t.qbs[g][:k]:
                if r.uniform() < noise:
                    s.append_kraus(int(q), [dm.depolarizing(0.05), dm.amplitude_damping(0.1),
                                            dm.phase_damping(0.2)][int(r.integers(3))])
        s.upload()

    ref, got = dm.Sim(n), dm.Sim(n)
    got.set_method(dm.METHOD_FUSED)
    got.set_profiling(True)
    load(ref)
    load(got)
    idx = np.random.default_rng(n).integers(0, 4 ** n, size=8192, dtype=np.uint64)
    for step in range(2):
        if step:
            for s in (ref, got):
                s.set_method(dm.METHOD_PLAIN_LAUNCH)
                s.run()
            ref.set_method(dm.METHOD_PLAIN)
            got.set_method(dm.METHOD_FUSED)
        ref.run()
        got.run()
        assert got.profile()["k_group"]["calls"] > 0
        assert np.max(np.abs(got.get_entries(idx) - ref.get_entries(idx))) <= 1e-10
        assert np.max(np.abs(got.get_diag() - ref.get_diag())) <= 1e-10
        assert abs(got.get_diag().sum() - 1) <= 1e-12
