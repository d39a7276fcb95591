"""Uploads and downloads where helper threads cannot be started, for want of threads or of memory (tests/hostcopy_check.cpp,
on the host): the threads that are there move the whole state, and no exception reaches the C entry points."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"


def test_lanes_without_threads(tmp_path):
    if not os.path.exists(HIPCC):
        pytest.skip("hipcc not found")
    exe = str(tmp_path / "hostcopy_check")
    subprocess.run([HIPCC, "-x", "hip", "-O1", "-std=c++17", "--offload-arch=gfx950", "-Xclang", "-target-feature",
                    "-Xclang", "-packed-fp32-ops", os.path.join(HERE, "hostcopy_check.cpp"),
                    os.path.join(HERE, "..", "fenice_amd", "csrc", "fvg_transfer.hip"), "-o", exe],
                   check=True, capture_output=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout.count("ok") == 12, r.stdout + r.stderr
