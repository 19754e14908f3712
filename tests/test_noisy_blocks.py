"""Noise channels folded into block sweeps: a block's gates and channels run as
stages inside one sweep (csrc/fused.hpp FusedStage, fuse.cpp build_stages)."""
import os
import shutil
import subprocess

import numpy as np
import pytest

import workloads as W
from conftest import ROOT


def test_noisy_blocks_on_the_cpu(tmp_path):
    """Stage records and trailing maps against gate-by-gate application
    (tests/cpp/noisy_blocks.cpp)."""
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("hipcc not found")
    exe = os.path.join(str(tmp_path), "noisy_blocks")
    pkg = os.path.join(ROOT, "dm-sim_amd")
    r = subprocess.run([hipcc, "-std=c++17", "-O2", "-I", os.path.join(pkg, "csrc"), "-I",
                        os.path.join(ROOT, "include"),
                        os.path.join(ROOT, "tests", "cpp", "noisy_blocks.cpp"), "-L", pkg,
                        "-ldmsim_amd", f"-Wl,-rpath,{pkg}", "-o", exe],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout.strip() == "48 cases OK", r.stdout


@pytest.mark.gpu
@pytest.mark.parametrize("n,herm,permute,m", [(7, 0, True, 0), (7, 0, False, 4), (8, 0, True, 5),
                                             (8, 0, False, 6), (8, 2, True, 0), (9, 0, True, 7),
                                             (10, 2, True, 0), (12, 1, True, 0), (12, 0, True, 0),
                                             (12, 0, False, 0)])
def test_folded_channels_match_plain(n, herm, permute, m):
    """Fused plans with channels inside blocks (every tile width, in place, out
    of place and Hermitian sweeps) against the plain method, two runs, the
    second after sweeps that leave rho conj-transposed."""
    import dmsim_amd as dm
    rng = np.random.default_rng(70 + n)
    t = W.random_mixed(n, 60, 7000 + n, gate_set=["H", "X", "U3", "CX", "CX", "SWAP", "RZZ", "CCX",
                                                  "C3X", "C2", "CU1"])

    def load(s):
        r = np.random.default_rng(n)
        for g in range(len(t)):
            s.append_table(t.take([g]))
            k = W.ARITY[W.OP_NAMES[t.ops[g]]]
            for q in t.qbs[g][:k]:
                if r.uniform() < 0.6:
                    s.append_kraus(int(q), [dm.depolarizing(0.05), dm.amplitude_damping(0.1),
                                            dm.phase_damping(0.2)][int(r.integers(3))])
        s.upload()

    ref, got = dm.Sim(n), dm.Sim(n)
    got.set_method(dm.METHOD_FUSED)
    got.set_fusion_hermitian(herm)
    got.set_fusion_permute(permute)
    got.set_tile_bits(m)
    load(ref)
    load(got)
    idx = rng.integers(0, 4 ** n, size=8192, dtype=np.uint64)
    for step in range(2):
        if step:
            for s in (ref, got):
                s.set_method(dm.METHOD_PLAIN_LAUNCH)
                s.run()
            ref.set_method(dm.METHOD_PLAIN)
            got.set_method(dm.METHOD_FUSED)
        ref.run()
        got.run()
        assert np.max(np.abs(got.get_entries(idx) - ref.get_entries(idx))) <= 1e-10
        assert np.max(np.abs(got.get_diag() - ref.get_diag())) <= 1e-10
        assert abs(got.get_diag().sum() - 1) <= 1e-12
    assert got.last_run_stats()["launches"] < len(t)  # no sweep per channel
