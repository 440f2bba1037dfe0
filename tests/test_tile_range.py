"""The grouped GEMM tiles' loads stay inside their operands, checked on the CPU."""

from __future__ import annotations

import os
import shutil
import subprocess
from pathlib import Path

import pytest
import torch

from fusion_amd import _lib

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


P = 1 << 20  # an aligned address that nothing reads: no launch succeeds here


@pytest.mark.skipif(torch.cuda.is_available(), reason="launches with made-up addresses")
@pytest.mark.parametrize("bm", [64, 128, 256])
@pytest.mark.parametrize("gated", [False, True])
def test_row_major_weight_span_is_checked(bm, gated):
    """Row-major W whose rows reach past the tiles' 32-bit offsets: refused by the tiles (a
    forced mapping and the atomic merge report it), left to the 64-bit mapping at 64 and 128
    tokens.  A launch that is not refused reports the missing device."""
    N, K, T = 512, 512, 64
    n_out = N // 2 if gated else N
    last = ((0xfffffff0 // 2 - K) // (N - 1)) // 8 * 8  # the largest row stride that fits
    lib = _lib.lib()

    def gemm(swn, variant):
        return lib.glm52_moe_gemm(P, K, 1, P, K, swn, n_out if gated else 0, P, n_out, None, P, P, P,
                                  4 * bm, bm, T, n_out, K, int(gated), variant, None)

    def merge(swn):
        return lib.glm52_moe_down_merge(P, K, P, K, swn, None, P, N, P, P, P, P, 4 * bm, bm, T, 8, N,
                                        K, None)

    assert gemm(last, 5) > 0 and merge(last) > 0
    assert gemm(last + 8, 5) == -2 and merge(last + 8) == -2
    assert gemm(1 << 40, 5) == -2
    auto = gemm(last + 8, 0)
    assert auto == -2 if bm == 256 else auto > 0
