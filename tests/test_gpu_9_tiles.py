"""The grouped GEMM tiles (block sizes 64, 128, 256) at their edges, against fp32 torch.

Row counts at the edges of a 16-row group, of a wave's share and of a block; the fewest
stages and an odd number of ring turns; row blocks of one expert past the groups they are
ordered in and past the 64 expert ids one look-up loads.
"""

from __future__ import annotations

import pytest
import torch

from fusion_amd import _lib
from fusion_amd.dispatch import moe_align_block_size
from fusion_amd.kernels import moe_down_merge as KD
from fusion_amd.kernels import moe_gateup as KG
from fusion_amd.kernels import oproj_resadd as KO

pytestmark = pytest.mark.gpu

BF16 = torch.bfloat16


def _close(got, want, K):
    """bf16 rounding of the result (2^-8 of it, both half-ulps), and K fp32 sums of products
    whose magnitudes are at most 4 here: K * 4 * 2^-22 covers any order of adds."""
    err = (got.float() - want).abs()
    tol = want.abs() * 2.0 ** -8 + K * 4 * 2.0 ** -22
    assert bool((err <= tol).all()), f"max excess {(err - tol).max().item()}"


@pytest.mark.parametrize("bm", [64, 128, 256])
@pytest.mark.parametrize("rows,K", [((1, 16, 17, 32), 256), ((33, 64, 65, 96), 256),
                                    ((127, 128, 129, 192), 768), ((193, 255, 256, 257), 256),
                                    ((1290, 2, 511, 513), 256), ((48, 80, 97, 112), 256),
                                    ((160, 161, 224, 225), 256), ((33 * 256 + 5, 3, 0, 1), 256)])
def test_tile_edges(gpu, rows, K, bm):
    print(f"tile bm={bm} rows={rows} K={K}", flush=True)
    g = torch.Generator(device=gpu).manual_seed(sum(rows) + K)
    E, N, T = len(rows), 512, sum(rows)
    ids = torch.cat([torch.full((n,), e, dtype=torch.int32) for e, n in enumerate(rows)])
    ids = ids[torch.randperm(T, generator=torch.Generator().manual_seed(K))].to(gpu)
    a = torch.empty(T, K, dtype=BF16, device=gpu).normal_(0, 1, generator=g).clamp_(-2, 2)
    w = torch.empty(E, N, K, dtype=BF16, device=gpu).normal_(0, 1, generator=g).clamp_(-2, 2)
    tw = torch.rand(T, generator=g, device=gpu)
    sti, eids, ntp = moe_align_block_size(ids.view(T, 1), bm, E)
    cfg = {"BLOCK_M": bm}
    full = torch.empty(T, N, device=gpu)
    for e in range(E):
        m = (ids == e).nonzero().view(-1)
        full[m] = a[m].float() @ w[e].float().t()

    def out(n):
        return torch.full((T, n), float("nan"), dtype=BF16, device=gpu)

    y, y_p, yw = out(N), out(N), out(N)
    wp = KG.pack_w512(w, N, 0, False)
    KG.moe_gemm(a, 1, w, y, None, sti, eids, ntp, T, N, 0, False, cfg)
    KG.moe_gemm_packed(a, 1, wp, y_p, None, sti, eids, ntp, T, N, False, cfg)
    KG.moe_gemm_packed(a, 1, wp, yw, tw, sti, eids, ntp, T, N, False, cfg)
    act, act_p = out(N // 2), out(N // 2)
    KG.moe_gemm(a, 1, w, act, None, sti, eids, ntp, T, N // 2, N // 2, True, cfg)
    KG.moe_gemm_packed(a, 1, KG.pack_w512(w, N // 2, N // 2, True), act_p, None, sti, eids, ntp,
                       T, N // 2, True, cfg)
    assert torch.equal(y, y_p) and torch.equal(act, act_p)
    _close(y, full, K)
    _close(yw, full * tw[:, None], K)
    gate, up = full[:, :N // 2], full[:, N // 2:]
    want = torch.nn.functional.silu(gate) * up
    # silu's slope is at most 1.1: the sums' errors reach the product through both factors
    err = (act.float() - want).abs()
    tol = want.abs() * 2.0 ** -7 + (gate.abs() + 1.1 * up.abs() + 1) * K * 4 * 2.0 ** -22
    assert bool((err <= tol).all())


@pytest.mark.parametrize("M,K,N", [(17, 64, 512), (64, 2048, 512), (65, 1024, 1536),
                                   (200, 4160, 512), (256, 64, 512), (257, 1024, 1024), (700, 2112, 512),
                                   (2300, 512, 1536),
                                   # 256-row tiles: one K slice, and four (N = 6144)
                                   (1281, 64, 6144), (2300, 128, 6144), (257, 4096, 6144),
                                   (383, 4096, 6144), (512, 4096, 6144),
                                   # 128-row tiles past 256 rows, two K slices; 256-row tiles again
                                   (513, 2048, 6144), (640, 2048, 6144), (641, 2048, 6144)])
def test_oproj_tile_edges(gpu, M, K, N):
    """o_proj from 17 rows: every epilogue, K slices or none, ragged last blocks, and row
    blocks past one order group."""
    print(f"oproj tile M={M} K={K} N={N}", flush=True)
    g = torch.Generator(device=gpu).manual_seed(M + K)
    a = torch.empty(M, K, dtype=BF16, device=gpu).normal_(0, 1, generator=g).clamp_(-2, 2)
    b = torch.empty(K, N, dtype=BF16, device=gpu).normal_(0, 1, generator=g).clamp_(-2, 2)
    r = torch.empty(M, N, dtype=BF16, device=gpu).normal_(0, 1, generator=g)
    want = a.float() @ b.float()
    for res in (None, r):
        c = torch.full((M, N), float("nan"), dtype=BF16, device=gpu)
        KO.gemm_launch(a, b, c, res, {}, res is not None, False)
        _close(c, want if res is None else want + r.float(), K)
        acc = torch.ones(M, N, device=gpu)
        KO.gemm_launch(a, b, acc, res, {}, res is not None, True)
        _close(acc, 1 + (want if res is None else want + r.float()), K)


def _side_by_side(pairs):
    """Each pair of launches first in order, then at once on two streams, their outputs filled
    with NaN: the same bits, from different sets of item counters."""
    gate, s1, s2 = torch.cuda.Stream(), torch.cuda.Stream(), torch.cuda.Stream()
    for name, (run_a, out_a), (run_b, out_b) in pairs:
        print(f"two streams: {name}", flush=True)
        want = []
        for run, out in ((run_a, out_a), (run_b, out_b)):
            out.fill_(float("nan"))
            run()
            torch.cuda.synchronize()
            want.append(out.clone())
            assert not bool(out.isnan().any()), name
        for _ in range(3):
            out_a.fill_(float("nan"))
            out_b.fill_(float("nan"))
            torch.cuda.synchronize()
            sets = []
            with torch.cuda.stream(gate):
                torch.cuda._sleep(1_000_000)  # both launches wait for it, then start together
                go = gate.record_event()
            for s, run in ((s1, run_a), (s2, run_b)):
                with torch.cuda.stream(s):
                    s.wait_event(go)
                    run()
                    sets.append(_lib.query("glm52_debug_item_set"))
            torch.cuda.synchronize()
            assert torch.equal(out_a, want[0]) and torch.equal(out_b, want[1]), name
            assert sets[0] != sets[1], (name, sets)


@pytest.mark.parametrize("bm", [64, 128, 256])
def test_two_streams_expert_gemms(gpu, bm):
    """Instances that share a counter array, at once: packed unweighted and packed weighted,
    and packed and in place."""
    g = torch.Generator(device=gpu).manual_seed(bm)
    E, N, K, T = 8, 1024, 1024, 2000
    ids = torch.randint(0, E, (T, 1), generator=g, dtype=torch.int32, device=gpu)
    a = torch.empty(T, K, dtype=BF16, device=gpu).normal_(0, 1, generator=g)
    w = torch.empty(E, N, K, dtype=BF16, device=gpu).normal_(0, 0.02, generator=g)
    wp, tw = KG.pack_w512(w, N, 0, False), torch.rand(T, generator=g, device=gpu)
    sti, eids, ntp = moe_align_block_size(ids, bm, E)
    o = [torch.empty(T, N, dtype=BF16, device=gpu) for _ in range(2)]
    cfg = {"BLOCK_M": bm}

    def packed(out, weights):
        return lambda: KG.moe_gemm_packed(a, 1, wp, out, weights, sti, eids, ntp, T, N, False, cfg)

    def in_place(out):
        return lambda: KG.moe_gemm(a, 1, w, out, None, sti, eids, ntp, T, N, 0, False, cfg)

    _side_by_side([("unweighted, weighted", (packed(o[0], None), o[0]), (packed(o[1], tw), o[1])),
                   ("packed, in place", (packed(o[0], None), o[0]), (in_place(o[1]), o[1]))])


def test_two_streams_oproj(gpu):
    """o_proj with K slices (epilogue 3) beside o_proj without (epilogue 1, and 2 into fp32)."""
    K, N = 4096, 1536
    g = torch.Generator(device=gpu).manual_seed(3)
    b = torch.empty(K, N, dtype=BF16, device=gpu).normal_(0, 0.02, generator=g)
    assert _lib.query("glm52_oproj_splits", 256, N, K) > 1
    assert _lib.query("glm52_oproj_splits", 12288, N, K) == 1

    def chain(M, f32):
        a = torch.empty(M, K, dtype=BF16, device=gpu).normal_(0, 1, generator=g)
        r = torch.empty(M, N, dtype=BF16, device=gpu).normal_(0, 1, generator=g)
        c = torch.empty(M, N, dtype=torch.float32 if f32 else BF16, device=gpu)

        def run():
            if f32:
                c.zero_()
            KO.gemm_launch(a, b, c, r, {}, True, f32)

        return run, c

    sliced, whole, whole32 = chain(256, False), chain(12288, False), chain(12288, True)
    _side_by_side([("K slices, whole K", sliced, whole), ("whole K, K slices", whole, sliced),
                   ("whole K, whole K into fp32", whole, whole32)])


def test_captured_launches_keep_sets_of_their_own(gpu):
    """A captured launch's counters are not among those that eager launches take in turn, so
    replays run beside any number of eager launches; every replay gives the eager bits."""
    g = torch.Generator(device=gpu).manual_seed(5)
    E, N, K, T, bm = 4, 512, 256, 300, 64
    ids = torch.randint(0, E, (T, 1), generator=g, dtype=torch.int32, device=gpu)
    a = torch.empty(T, K, dtype=BF16, device=gpu).normal_(0, 1, generator=g)
    wp = KG.pack_w512(torch.empty(E, N, K, dtype=BF16, device=gpu).normal_(0, 0.02, generator=g),
                      N, 0, False)
    lay = moe_align_block_size(ids, bm, E)
    out, eager = (torch.empty(T, N, dtype=BF16, device=gpu) for _ in range(2))

    def run(c):
        KG.moe_gemm_packed(a, 1, wp, c, None, *lay, T, N, False, {"BLOCK_M": bm})
        return _lib.query("glm52_debug_item_set")

    assert run(eager) < 1024
    torch.cuda.synchronize()
    want = eager.clone()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        sets = [run(out), run(out)]
    assert min(sets) >= 1024 and sets[0] != sets[1]
    side = torch.cuda.Stream()
    for i in range(4):
        out.fill_(float("nan"))
        eager.fill_(float("nan"))
        torch.cuda.synchronize()
        with torch.cuda.stream(side):
            for _ in range(300):  # 1200 in all: every eager set is taken
                assert run(eager) < 1024
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want) and torch.equal(eager, want), f"replay {i}"


@pytest.mark.parametrize("gated", [False, True])
def test_weight_rows_past_4_gib(gpu, gated):
    """Row-major W as a view with a row pitch of 8 MB, one expert spanning more than 2^32 bytes:
    64- and 128-token blocks give the rows' results, 256-token blocks and the atomic merge
    refuse it; a span just inside runs the tiles with the contiguous copy's bits."""
    E, N, K, T = 2, 512, 256, 200
    inside = ((0xfffffff0 // 2 - K) // (N - 1)) // 8 * 8
    pitch = inside + 8
    g = torch.Generator(device=gpu).manual_seed(9)
    vals = torch.empty(E, N, K, dtype=BF16, device=gpu).normal_(0, 1, generator=g).clamp_(-2, 2)
    big = torch.empty(N * pitch, dtype=BF16, device=gpu)
    ids = torch.randint(0, E, (T, 1), generator=g, dtype=torch.int32, device=gpu)
    a = torch.empty(T, K, dtype=BF16, device=gpu).normal_(0, 1, generator=g).clamp_(-2, 2)
    full = torch.stack([vals[int(e)].float() @ x.float() for e, x in zip(ids.view(-1), a)])
    n_out = N // 2 if gated else N
    want = torch.nn.functional.silu(full[:, :n_out]) * full[:, n_out:] if gated else full
    for bm in (64, 128, 256):
        print(f"weight span bm={bm} gated={gated}", flush=True)
        lay = moe_align_block_size(ids, bm, E)

        def run(w):
            c = torch.full((T, n_out), float("nan"), dtype=BF16, device=gpu)
            KG.moe_gemm(a, 1, w, c, None, *lay, T, n_out, n_out if gated else 0, gated,
                        {"BLOCK_M": bm})
            return c

        ref = run(vals)
        w_in = big.as_strided((E, N, K), (K, inside, 1))
        w_in.copy_(vals)
        assert torch.equal(run(w_in), ref)
        w_past = big.as_strided((E, N, K), (K, pitch, 1))
        w_past.copy_(vals)
        if bm == 256:
            with pytest.raises(RuntimeError, match="unsupported"):
                run(w_past)
        elif gated:  # silu's slope is at most 1.1: the sums' errors reach the product twice
            err = (run(w_past).float() - want).abs()
            tol = want.abs() * 2.0 ** -7 + (full[:, :n_out].abs() + 1.1 * full[:, n_out:].abs()
                                            + 1) * K * 4 * 2.0 ** -22
            assert bool((err <= tol).all())
        else:
            _close(run(w_past), full, K)
            out = torch.zeros(T, N, dtype=BF16, device=gpu)
            with pytest.raises(RuntimeError, match="unsupported"):
                KD.launch_down(a, w_past, out, torch.ones(T, device=gpu), *lay, T, 1,
                               {"BLOCK_M": bm}, True)


@pytest.mark.parametrize("bm", [64, 128, 256])
def test_nan_outputs(gpu, bm):
    """A NaN of either sign in a token row or a weight row reaches that row's or column's
    outputs and no other, in every bf16 store of the tiles."""
    g = torch.Generator(device=gpu).manual_seed(bm)
    E, N, K, T = 2, 512, 256, 300
    ids = (torch.arange(T, device=gpu) % E).to(torch.int32).view(T, 1)
    a = torch.empty(T, K, dtype=BF16, device=gpu).normal_(0, 1, generator=g)
    w = torch.empty(E, N, K, dtype=BF16, device=gpu).normal_(0, 1, generator=g)
    a.view(torch.int16)[[7, 130, 290], [3, 255, 64]] = torch.tensor(
        [0x7F81, -1, 0x7FC0], dtype=torch.int16, device=gpu)
    w.view(torch.int16)[1, [11, 300], 5] = torch.tensor([-63, 0x7FFF], dtype=torch.int16, device=gpu)
    nan = torch.zeros(T, N, dtype=torch.bool, device=gpu)
    nan[[7, 130, 290]] = True
    nan[1::2, 11] = nan[1::2, 300] = True
    lay = moe_align_block_size(ids, bm, E)
    cfg, tw = {"BLOCK_M": bm}, torch.rand(T, generator=g, device=gpu)
    for weights in (None, tw):
        for packed in (False, True):
            out = torch.zeros(T, N, dtype=BF16, device=gpu)
            if packed:
                KG.moe_gemm_packed(a, 1, KG.pack_w512(w, N, 0, False), out, weights, *lay, T, N,
                                   False, cfg)
            else:
                KG.moe_gemm(a, 1, w, out, weights, *lay, T, N, 0, False, cfg)
            assert torch.equal(out.isnan(), nan)
    act = torch.zeros(T, N // 2, dtype=BF16, device=gpu)
    KG.moe_gemm(a, 1, w, act, None, *lay, T, N // 2, N // 2, True, cfg)
    assert torch.equal(act.isnan(), nan[:, :N // 2] | nan[:, N // 2:])


@pytest.mark.parametrize("M", [40, 100, 1300])
def test_oproj_nan_outputs(gpu, M):
    """The same for o_proj without and with the residual (64-, 128- and 256-row tiles)."""
    K, N = 256, 6144
    g = torch.Generator(device=gpu).manual_seed(M)
    a = torch.empty(M, K, dtype=BF16, device=gpu).normal_(0, 1, generator=g)
    b = torch.empty(K, N, dtype=BF16, device=gpu).normal_(0, 1, generator=g)
    r = torch.empty(M, N, dtype=BF16, device=gpu).normal_(0, 1, generator=g)
    a.view(torch.int16)[[3, M - 1], [7, 200]] = torch.tensor([-1, 0x7F81], dtype=torch.int16,
                                                             device=gpu)
    r.view(torch.int16)[5, 77] = -63
    nan = torch.zeros(M, N, dtype=torch.bool, device=gpu)
    nan[[3, M - 1]] = True
    out = torch.zeros(M, N, dtype=BF16, device=gpu)
    KO.gemm_launch(a, b, out, None, {}, False, False)
    assert torch.equal(out.isnan(), nan)
    nan[5, 77] = True
    KO.gemm_launch(a, b, out, r, {}, True, False)
    assert torch.equal(out.isnan(), nan)
