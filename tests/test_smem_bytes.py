"""The LDS sizes the launcher modules report for the prefill tiles, against the kernel's ring:
a stage is (W rows + tokens) x 64 bytes, and the ring as many stages as 160 KB hold."""

from __future__ import annotations

import pytest

from fusion_amd.kernels import moe_down_merge as KD
from fusion_amd.kernels import moe_gateup as KG


@pytest.mark.parametrize("bm,stages,want", [(64, 8, 163840), (128, 6, 147456), (256, 5, 163840)])
def test_tiles_on_weights_in_place(bm, stages, want):
    assert stages * (256 + bm) * 64 == want
    for cfg in ({"BLOCK_M": bm}, {"BLOCK_M": bm, "variant": "auto"},
                {"BLOCK_M": bm, "variant": "w512"}):
        assert KG.smem_bytes(cfg, True) == KG.smem_bytes(cfg, False) == want
        assert KD.smem_bytes(cfg) == want


@pytest.mark.parametrize("bm,stages,want", [(64, 4, 147456), (128, 4, 163840)])
def test_atomic_merge_on_packed_weights(bm, stages, want):
    assert stages * (512 + bm) * 64 == want
    assert KD.smem_bytes({"BLOCK_M": bm, "w2_packed": object()}) == want
    assert KD.smem_bytes({"BLOCK_M": 256, "w2_packed": object()}) == 163840
