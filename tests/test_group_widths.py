"""The fusion width in group plans (csrc/fuse.cpp build_group_plan)."""
import os
import shutil
import subprocess

import pytest

from conftest import ROOT


def test_stages_keep_the_fusion_width(tmp_path):
    """Widths 1..5 with noise and with five-qubit gates, on the CPU
    (tests/cpp/group_widths.cpp)."""
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("hipcc not found")
    exe = os.path.join(str(tmp_path), "group_widths")
    pkg = os.path.join(ROOT, "dm-sim_amd")
    r = subprocess.run([hipcc, "-std=c++17", "-O2", "-I", os.path.join(pkg, "csrc"), "-I",
                        os.path.join(ROOT, "include"),
                        os.path.join(ROOT, "tests", "cpp", "group_widths.cpp"), "-L", pkg,
                        "-ldmsim_amd", f"-Wl,-rpath,{pkg}", "-o", exe],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout.strip() == "15 cases OK", r.stdout
