"""The co-residency cache of the launch plans (plh::capacity_key) keeps different kernels apart: a host program linked
to the library walks the geometries (CPU only)."""
from __future__ import annotations

import os
import shutil
import subprocess

import pytest

from persistent_lstm_hip_amd.extension import LIB_PATH

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.skipif(shutil.which("hipcc") is None, reason="hipcc not found")
def test_geometries_with_one_key_run_the_same_kernels(tmp_path):
    exe = str(tmp_path / "capacity_key_check")
    lib = os.path.dirname(LIB_PATH)
    cmd = ["hipcc", "-x", "hip", "--cuda-host-only", "-O1", "-std=c++17", "-w",
           "-I", os.path.join(ROOT, "persistent_lstm_hip_amd", "csrc"),
           os.path.join(ROOT, "tests", "capacity_key_check.cpp"), "-o", exe,
           "-L" + lib, "-lpersistent_lstm_hip", "-Wl,-rpath," + lib]
    subprocess.run(cmd, check=True, capture_output=True, text=True, timeout=300)
    out = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert out.returncode == 0, out.stdout + out.stderr
    assert " 0 mismatches" in out.stdout
