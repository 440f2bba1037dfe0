"""Performance cases of the GLM-5.2 MoE FFN layer: what a serving program runs per layer.

Three kinds of case, each through public entry points:

* `block`: the composed layer, `MoEBlock(T, ...)(x, r)`, on the packed expert weights;
* `oproj`: the attention output projection with its residual add,
  `oproj_resadd.make_fused_chain`;
* `launchers`: the same layer as `block`, composed from the drop-in launchers on the
  row-major weights (w13 [E, 2I, H], w2 [E, H, I]), as a program written against the
  reference's launcher API runs it.

Sizes are the model's (256 experts, top 8, H = 6144, I = 2048) at the token counts of the
layer harness and the benchmark (1, 256, 512, 2048, 8192) and at ragged ones.
"""

from __future__ import annotations

import math

import torch

from fusion_amd import config as C
from fusion_amd.block import (MoEBlock, PackedExperts, default_block_m, default_shared_block_m,
                              shared_layout)
from fusion_amd.dispatch import moe_align_block_size
from fusion_amd.kernels import add_rmsnorm, moe_down_merge, moe_gateup, norm_router, oproj_resadd

H, I, E, K8 = C.H, C.I, C.E, C.TOPK
BF16 = torch.bfloat16
OPROJ_K_DECODE = 32768  # absorbed MLA: 64 heads x 512
OPROJ_K_PREFILL = 16384  # 64 heads x 256


def listed():
    return [
        # one sequence decoding: latency and launches count
        {"name": "block_t1", "kind": "block", "T": 1, "bias": "normal"},
        # a small serving batch, odd
        {"name": "block_t13", "kind": "block", "T": 13, "bias": "normal"},
        # a ragged decode batch: most experts hit, a few rows each
        {"name": "block_t100", "kind": "block", "T": 100, "bias": "normal"},
        # a full decode batch
        {"name": "block_t256", "kind": "block", "T": 256, "bias": "normal"},
        # a large decode batch, or a short prompt's prefill
        {"name": "block_t512", "kind": "block", "T": 512, "bias": "normal"},
        # a ragged prefill chunk between the usual powers of two
        {"name": "block_t1333", "kind": "block", "T": 1333, "bias": "normal"},
        # a prefill chunk
        {"name": "block_t2048", "kind": "block", "T": 2048, "bias": "normal"},
        # a long prompt's prefill with skewed expert load
        {"name": "block_t8192_zipf", "kind": "block", "T": 8192, "bias": "zipf"},
        # the output projection of one decoded token, of a decode batch, of a long prompt
        {"name": "oproj_m1", "kind": "oproj", "T": 1, "K": OPROJ_K_DECODE},
        {"name": "oproj_m256", "kind": "oproj", "T": 256, "K": OPROJ_K_DECODE},
        {"name": "oproj_m8192", "kind": "oproj", "T": 8192, "K": OPROJ_K_PREFILL},
        # a prefill chunk of a program that keeps the reference's weight layout
        {"name": "launchers_t2048", "kind": "launchers", "T": 2048, "bias": "normal"},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng):
    kind = rng.choices(("block", "oproj", "launchers"), (7, 3, 2))[0]
    if kind == "oproj":
        T = _log_int(rng, 1, 8192)
        return {"kind": kind, "T": T, "K": OPROJ_K_DECODE if T <= 1024 else OPROJ_K_PREFILL}
    T = _log_int(rng, 1, 8192 if kind == "block" else 2048)
    return {"kind": kind, "T": T, "bias": rng.choice(("normal", "zipf"))}


def _rng(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _normal(shape, std, g):
    return torch.empty(shape, dtype=BF16, device="cuda").normal_(0.0, std, generator=g)


def _front_inputs(case, g):
    """x, r, the norm weight, the gate [E, H] and the selection bias of one layer."""
    T = case["T"]
    x, r = _normal((T, H), 1.0, g), _normal((T, H), 1.0, g)
    w_norm = (1.0 + 0.02 * torch.randn(H, generator=g, device="cuda")).to(BF16)
    gate = _normal((E, H), H ** -0.5, g)
    if case["bias"] == "zipf":
        bias = 0.5 * torch.arange(1, E + 1, dtype=torch.float64, device="cuda") ** -1.1
    else:
        bias = 0.01 * torch.randn(E, generator=g, device="cuda")
    return x, r, w_norm, gate, bias.float()


def _expert_inputs(g):
    """w13, w2 of the routed experts, then of the shared one, each expert drawn alone."""
    out = []
    for n, rows, cols in ((E, 2 * I, H), (E, H, I), (1, 2 * I, H), (1, H, I)):
        w = torch.empty(n, rows, cols, dtype=BF16, device="cuda")
        for e in range(n):
            w[e].normal_(0.0, 0.02, generator=g)
        out.append(w)
    return out


def _oproj_inputs(case, g):
    T, K = case["T"], case["K"]
    return _normal((T, K), 1.0, g), _normal((K, H), 0.02, g), _normal((T, H), 1.0, g)


class _Launchers:
    """The layer from the drop-in launchers: the row-major weights and the buffers that a
    program allocates once."""

    def __init__(self, T, x, r, w_norm, gate, bias, w13, w2, w13s, w2s):
        def buf(*shape, dtype=BF16):
            return torch.empty(*shape, dtype=dtype, device="cuda")

        self.T, self.x, self.r, self.w_norm, self.wgt = T, x, r, w_norm, gate.t().contiguous()
        self.w13, self.w2, self.w13s, self.w2s = w13, w2, w13s, w2s
        self.bm, sbm = default_block_m(T), default_shared_block_m(T)
        self.cfg, self.cfg_s = {"BLOCK_M": self.bm}, {"BLOCK_M": sbm}
        self.cfg_topk = {"correction_bias": bias}
        self.shared = shared_layout(T, sbm, x.device)
        self.ones = torch.ones(T, device="cuda")
        self.h, self.y, self.routed, self.out = (buf(T, H) for _ in range(4))
        self.logits = buf(T, E, dtype=torch.float32)
        self.topw = buf(T, K8, dtype=torch.float32)
        self.topi = buf(T, K8, dtype=torch.int32)
        self.act, self.rows = buf(T * K8, I), buf(T * K8, H)
        self.act_s, self.rows_s = buf(T, I), buf(T, H)

    def __call__(self):
        T = self.T
        add_rmsnorm.fused_add_rmsnorm(self.x, self.r, self.w_norm, self.h, self.y, {})
        norm_router.router_gemm(self.y, self.wgt, self.logits, {})
        norm_router.topk_only(self.logits, self.topw, self.topi, self.cfg_topk)
        layout = moe_align_block_size(self.topi, self.bm, E)
        moe_gateup.launch_gateup(self.y, self.w13, self.act, *layout, T * K8, K8, I, self.cfg,
                                 True)
        moe_down_merge.launch_down(self.act, self.w2, self.rows, self.topw.view(-1), *layout,
                                   T * K8, K8, self.cfg, False)
        moe_down_merge.launch_moe_sum(self.rows, self.routed, self.h, K8, {}, True)
        moe_gateup.launch_gateup(self.y, self.w13s, self.act_s, *self.shared, T, 1, I,
                                 self.cfg_s, True)
        moe_down_merge.launch_down(self.act_s, self.w2s, self.rows_s, self.ones, *self.shared,
                                   T, 1, self.cfg_s, False)
        moe_down_merge.launch_resadd(self.routed, self.rows_s, self.out, {})


def prepare(case, seed):
    g = _rng(seed)
    if case["kind"] == "oproj":
        a, b, r = _oproj_inputs(case, g)
        out = torch.empty(case["T"], H, dtype=BF16, device="cuda")
        return {"kind": "oproj", "a": a, "b": b, "r": r, "out": out,
                "chain": oproj_resadd.make_fused_chain(a, b, r, out, None, {})}
    x, r, w_norm, gate, bias = _front_inputs(case, g)
    weights = _expert_inputs(g)
    if case["kind"] == "launchers":
        return {"kind": "launchers",
                "layer": _Launchers(case["T"], x, r, w_norm, gate, bias, *weights)}
    experts = PackedExperts(*weights)
    return {"kind": "block", "x": x, "r": r,
            "layer": MoEBlock(case["T"], w_norm, gate.t().contiguous(), bias, experts)}


def run(state):
    if state["kind"] == "oproj":
        for launch in state["chain"]:
            launch()
        return {"h1": state["out"]}
    layer = state["layer"]
    if state["kind"] == "launchers":
        layer()
    else:
        layer(state["x"], state["r"])
    return {"h": layer.h, "out": layer.out, "topi": layer.topi, "topw": layer.topw}


def work(case):
    T = case["T"]
    if case["kind"] == "oproj":
        K = case["K"]
        return {"bytes": 2.0 * (K * H + T * K + 2 * T * H), "flops": 2.0 * T * K * H}
    # distinct experts hit: the expectation under a flat load
    hit = E * (1.0 - (1.0 - K8 / E) ** T)
    weights = 2.0 * (3 * H * I * (hit + 1) + E * H)
    flops = 2.0 * T * (3 * H * I * (K8 + 1) + E * H)
    # x and r in; h, out and the routing back
    return {"bytes": weights + T * (2.0 * 4 * H + 8 * K8), "flops": flops}


def tolerance(case):
    # bf16 outputs of fp32 sums: half a bf16 ulp each side, and in the layer one rounding per
    # expert row before the merge
    if case["kind"] == "oproj":
        return {"rel": 7e-3, "max": 3e-2}
    return {"rel": 8e-3, "max": 5e-2}


def _exact_oproj(case, g):
    a, b, r = _oproj_inputs(case, g)
    return {"h1": torch.addmm(r.double(), a.double(), b.double())}


def _exact_layer(case, g):
    """The layer in 64 bits from its stored 16-bit states h and y, which define the routing."""
    x, r, w_norm, gate, bias = _front_inputs(case, g)
    w13, w2, w13s, w2s = _expert_inputs(g)
    h = (x.double() + r.double()).to(BF16)
    hd = h.double()
    rstd = 1.0 / torch.sqrt(hd.square().mean(1, keepdim=True) + C.RMS_NORM_EPS)
    y = ((h.float() * rstd.float()).to(BF16).float() * w_norm.float()).to(BF16).double()

    logits = (y @ gate.double().t()).float()
    s = torch.sigmoid(logits.double()).float()
    order = torch.sort(s + bias, dim=1, descending=True, stable=True).indices
    topi = order[:, :K8].contiguous()
    picked = s.gather(1, topi).double()
    topw = picked / picked.sum(1, keepdim=True) * C.ROUTED_SCALING_FACTOR

    def mlp(rows, up, down):
        gu = rows @ up.double().t()
        return (torch.nn.functional.silu(gu[:, :I]) * gu[:, I:]) @ down.double().t()

    out = hd + mlp(y, w13s[0], w2s[0])
    for e in range(E):
        t, k = (topi == e).nonzero(as_tuple=True)
        if t.numel():
            out.index_add_(0, t, topw[t, k, None] * mlp(y[t], w13[e], w2[e]))
    return {"h": h, "out": out, "topi": topi.int(), "topw": topw}


def exact(case, seed):
    g = _rng(seed)
    return _exact_oproj(case, g) if case["kind"] == "oproj" else _exact_layer(case, g)
