"""The prefill tile launches' item counters, through the host launch path on a machine without
a GPU: the set a launch deals from is drawn before the launch itself, which then reports the
missing device."""

from __future__ import annotations

import pytest
import torch

from fusion_amd import _lib

P = 1 << 20  # an aligned address that nothing reads: no launch succeeds here
T, K, N = 64, 512, 512


def _gemm(bm, gated, weighted, packed):
    tail = (P if weighted else None, P, P, P, 4 * bm, bm, T, N, K, int(gated))
    if packed:
        return _lib.lib().glm52_moe_gemm_packed(P, K, 1, P, P, N, *tail, None)
    return _lib.lib().glm52_moe_gemm(P, K, 1, P, 2 * N * K, K, N if gated else 0, P, N, *tail, 5,
                                     None)


def _down_merge(bm, packed):
    return _lib.lib().glm52_moe_down_merge(P, K, P, N * K, K, P if packed else None, P, N, P, P, P,
                                           P, 4 * bm, bm, T, 8, N, K, None)


def _launches():
    """The instances of each source file, which share its counters."""
    for bm in (64, 128, 256):
        for gated in (True, False):
            yield [(f"bm {bm} gated {gated} weighted {w} packed {p}",
                    lambda bm=bm, gated=gated, w=w, p=p: _gemm(bm, gated, w, p))
                   for w in (False, True) for p in (False, True)]
        yield [(f"bm {bm} atomic merge packed {p}", lambda bm=bm, p=p: _down_merge(bm, p))
               for p in (False, True)]


@pytest.mark.skipif(torch.cuda.is_available(), reason="launches with made-up addresses")
def test_instances_of_one_source_draw_different_sets():
    for group in _launches():
        seen = {}
        for turn in range(3):
            for name, launch in group:
                assert launch() > 0, f"{name}: a launch without a GPU must report a HIP error"
                s = _lib.query("glm52_debug_item_set")
                assert 0 <= s < 1024, f"{name}: an uncaptured launch took set {s}"
                assert s not in seen, f"{name} took set {s} of {seen[s]}"
                seen[s] = f"{name}, turn {turn}"
