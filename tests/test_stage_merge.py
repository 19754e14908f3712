"""Which stages a block with channels takes (csrc/fuse.cpp build_stages)."""
import os
import shutil
import subprocess

import pytest

from conftest import ROOT


def test_channel_free_stages_merge(tmp_path):
    """tests/cpp/stage_merge.cpp, on the CPU."""
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("hipcc not found")
    exe = os.path.join(str(tmp_path), "stage_merge")
    pkg = os.path.join(ROOT, "dm-sim_amd")
    r = subprocess.run([hipcc, "-std=c++17", "-O2", "-I", os.path.join(pkg, "csrc"), "-I",
                        os.path.join(ROOT, "include"),
                        os.path.join(ROOT, "tests", "cpp", "stage_merge.cpp"), "-L", pkg,
                        "-ldmsim_amd", f"-Wl,-rpath,{pkg}", "-o", exe],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout.strip() == "OK", r.stdout
