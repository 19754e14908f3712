"""The plain method with whole rows of rho on chip (csrc/rows.hpp, rows.hip)."""
import os
import shutil
import subprocess

import numpy as np
import pytest

import workloads as W
from conftest import ROOT


def test_row_programs(tmp_path):
    """Every program's LDS places and arithmetic on the CPU, n = 1..14
    (tests/cpp/row_programs.cpp)."""
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("hipcc not found")
    exe = os.path.join(str(tmp_path), "row_programs")
    pkg = os.path.join(ROOT, "dm-sim_amd")
    r = subprocess.run([hipcc, "-std=c++17", "-O2", "-ffp-contract=off", "-I",
                        os.path.join(pkg, "csrc"), os.path.join(ROOT, "tests", "cpp",
                                                                "row_programs.cpp"),
                        "-L", pkg, "-ldmsim_amd", f"-Wl,-rpath,{pkg}", "-o", exe],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout.strip() == "42 cases OK", r.stdout


@pytest.mark.gpu
@pytest.mark.parametrize("n", list(range(1, 15)))
def test_rows_equal_one_launch_per_primitive(n):
    """Every row shape (one wave or many rows a workgroup, n = 14 with the
    planes in turn) against the sweeps of one primitive each, bit for bit:
    a continued run, and a run that starts from the conj-transposed
    orientation those sweeps leave."""
    import dmsim_amd as dm
    t = W.random_mixed(n, 40 if n > 11 else 120, 60 + n,
                       gate_set=[g for g in W.OP_NAMES if W.ARITY[g] <= n])
    sims = [dm.Sim(n) for _ in range(3)]
    idx = np.random.default_rng(n).integers(0, 4 ** n, size=4096, dtype=np.uint64)
    for s, methods in zip(sims, ((0, 0), (1, 1), (1, 0))):
        s.append_table(t)
        s.upload()
        for m in methods:
            s.set_method(m)
            s.run()
    if n <= 12:
        want = sims[1].get_dm()
        for s in (sims[0], sims[2]):
            got = s.get_dm()
            assert np.array_equal(got[0], want[0]) and np.array_equal(got[1], want[1])
    else:
        want = sims[1].get_entries(idx), sims[1].get_diag()
        for s in (sims[0], sims[2]):
            assert np.array_equal(s.get_entries(idx), want[0])
            assert np.array_equal(s.get_diag(), want[1])
