"""The grouped GEMM tiles' ring loads stay inside their operands, checked on the CPU."""

from __future__ import annotations

import os
import shutil
import subprocess
from pathlib import Path

ROOT = Path(__file__).resolve().parent.parent


def test_ring_loads_stay_in_range(tmp_path):
    """Every stage's loads are in range and at their stage, padding rows' and past-the-end
    loads are out of range, under every form of the buffer range check."""
    cxx = os.environ.get("CXX") or shutil.which("g++") or shutil.which("c++")
    assert cxx, "a host C++ compiler is needed"
    exe = tmp_path / "tile_range_check"
    subprocess.run([cxx, "-std=c++17", "-O2", "-Wall", "-I", str(ROOT / "fusion_amd" / "csrc"),
                    "-o", str(exe), str(ROOT / "tests" / "tile_range_check.cpp")], check=True)
    run = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert run.returncode == 0, run.stdout
