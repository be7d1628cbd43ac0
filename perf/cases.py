"""The work that users of this framework have it do, as cases that a timing program can run one pass at a time.

Four kinds of call, each through the public entry points as a model's forward (or its loader) makes them:

  moe     one routed MoE layer: the router (`moe.route.route_step`, as R9kTopKRouter calls it) and the experts
          (`R9700Mxfp4Experts.apply`), from decode batches to long prompts. Widths: the 288-expert layer of the decode
          and prefill benchmarks, the 384-expert layer with Zipf-skewed routing, and one tensor-parallel rank's share
          of a 512-expert layer (intermediate 320, not a multiple of the kernels' 128-wide K-tiles).
  shared  the gated shared expert beside every routed layer (`torch.ops.r9700.shared_expert`).
  dense   one dense linear: MXFP4 weights (`linear.mxfp4.apply_dense`) or a checkpoint's NVFP4 weights kept exactly
          (`quant.nvfp4.native_dense_forward`, the default for dense NVFP4 linears).
  load    one NVFP4 linear's load: conversion to MXFP4 with searched block exponents and the kernels' weight layout.

`listed()` names the cases, `draw(rng)` gives others of the same ranges, `prepare` / `run` are a state and one pass over
it, `work` the bytes and operations a pass cannot do without, `exact` the outputs in 64 bits without this package's
code, and `tolerance` how far another implementation of the same precision may be off.
"""
import math
import os
import sys
from types import SimpleNamespace

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "r9700-stack_amd"))

from r9700_vllm.kernels import moe as K                        # noqa: E402
from r9700_vllm.linear import mxfp4 as LX                      # noqa: E402
from r9700_vllm.moe import route, shared                       # noqa: E402
from r9700_vllm.moe.experts import R9700Mxfp4Experts           # noqa: E402
from r9700_vllm.quant import nvfp4 as NV                       # noqa: E402

# routed layers: experts, hidden, intermediate, top-k, Zipf exponent of the expert popularity (0: uniform), e8m0 range
LAYERS = {
    "e288": dict(E=288, H=2048, I=512, topk=8, zipf=0.0, lo=118, hi=126),
    "e384_skew": dict(E=384, H=4096, I=2048, topk=8, zipf=1.1, lo=116, hi=126),
    "e512_rank": dict(E=512, H=2560, I=320, topk=10, zipf=0.0, lo=118, hi=126),
}
# dense linears [N, K]: the benchmark's widest, the launch table's widths, one rank's odd widths
DENSE = [(17408, 5120), (4096, 4096), (2048, 5120), (1024, 2048), (640, 2560), (2560, 320)]
NATIVE = [(17408, 5120), (4096, 4096), (2048, 5120), (1024, 2048)]


def listed():
    big = dict(N=17408, K=5120)
    return [
        # one user's decode step: routing, two small GEMMs, all latency
        dict(name="moe_t1", kind="moe", layer="e288", T=1),
        # a busy decode batch: 240 of the 288 experts touched by one or two rows each
        dict(name="moe_t64", kind="moe", layer="e288", T=64),
        # a long prompt
        dict(name="moe_t8192", kind="moe", layer="e288", T=8192),
        # wide experts under skewed routing: a large decode batch, and a prompt chunk (the largest case)
        dict(name="moe_skew_t256", kind="moe", layer="e384_skew", T=256),
        dict(name="moe_skew_t4096", kind="moe", layer="e384_skew", T=4096),
        # one rank's share of a 512-expert layer on a ragged prompt chunk
        dict(name="moe_rank_t3001", kind="moe", layer="e512_rank", T=3001),
        # the shared expert at a decode batch: the smallest GEMMs of the path
        dict(name="shared_t16", kind="shared", H=2048, I=512, T=16),
        # a dense MXFP4 linear at a middling decode batch, and at a short prompt
        dict(name="dense_m37", kind="dense", fmt="mxfp4", M=37, **big),
        dict(name="dense_m333", kind="dense", fmt="mxfp4", M=333, **big),
        # a checkpoint's NVFP4 linear kept exactly: a small decode batch and a prompt chunk
        dict(name="nvfp4_m4", kind="dense", fmt="nvfp4", M=4, **big),
        dict(name="nvfp4_m2000", kind="dense", fmt="nvfp4", M=2000, **big),
        # loading one NVFP4 linear as MXFP4
        dict(name="load_nvfp4", kind="load", **big),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.49))))))


def draw(rng):
    kind = rng.choice(("moe", "moe", "moe", "dense", "dense", "dense", "shared", "load"))
    if kind == "moe":
        layer = rng.choice(sorted(LAYERS))
        return dict(kind=kind, layer=layer, T=_log_int(rng, 1, 8192 if layer == "e288" else 4096))
    if kind == "shared":
        return dict(kind=kind, H=2048, I=512, T=_log_int(rng, 1, 4096))
    if kind == "dense":
        fmt = rng.choice(("mxfp4", "nvfp4"))
        N, Kd = rng.choice(DENSE if fmt == "mxfp4" else NATIVE)
        M = _log_int(rng, 1, 4096)
        if fmt == "nvfp4" and 32 <= M < 128:                   # widths the NVFP4 linear does not serve at every K
            M = M // 4 if rng.random() < 0.5 else 4 * M
        return dict(kind=kind, fmt=fmt, M=M, N=N, K=Kd)
    return dict(kind=kind, N=16 * _log_int(rng, 32, 1088), K=32 * _log_int(rng, 16, 160))


# ------------------------------------------------------------------------------------------------- inputs
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(1_000_003 * (seed + 1))


def _bytes(g, shape, lo=0, hi=255):
    return torch.randint(lo, hi + 1, shape, generator=g, device="cuda", dtype=torch.uint8)


def _randn(g, *shape):
    return torch.randn(*shape, generator=g, device="cuda")


def _mxfp4_ckpt(g, E, N, Kd, lo, hi):
    """Checkpoint MXFP4 tensors: e2m1 codes two a byte, an e8m0 exponent per 32."""
    return _bytes(g, (E, N, Kd // 2)), _bytes(g, (E, N, Kd // 32), lo, hi)


def _nvfp4_ckpt(g, N, Kd):
    """Checkpoint NVFP4 tensors: e2m1 codes, an e4m3 scale per 16, one fp32 global divisor."""
    s16 = (_randn(g, N, Kd // 16).abs() * 0.05 * 448).clamp(2.0 ** -9, 448.0).to(torch.float8_e4m3fn)
    return _bytes(g, (N, Kd // 2)), s16, torch.full((1,), 448.0, device="cuda")


def _moe_inputs(case, seed):
    L, T, g = LAYERS[case["layer"]], case["T"], _gen(seed)
    w13 = _mxfp4_ckpt(g, L["E"], 2 * L["I"], L["H"], L["lo"], L["hi"])
    w2 = _mxfp4_ckpt(g, L["E"], L["H"], L["I"], L["lo"], L["hi"])
    x = _randn(g, T, L["H"]).to(torch.bfloat16)
    logits = _randn(g, T, L["E"])
    if L["zipf"]:
        rank = torch.rand(L["E"], generator=g, device="cuda").argsort().float() + 1
        logits = logits - L["zipf"] * torch.log(rank)
    return L, w13, w2, x, logits.to(torch.bfloat16)


def _shared_inputs(case, seed):
    g = _gen(seed)
    w1 = _mxfp4_ckpt(g, 1, 2 * case["I"], case["H"], 118, 126)
    w2 = _mxfp4_ckpt(g, 1, case["H"], case["I"], 118, 126)
    wg = (_randn(g, case["H"]) * case["H"] ** -0.5).to(torch.bfloat16)
    return w1, w2, wg, _randn(g, case["T"], case["H"]).to(torch.bfloat16)


def _dense_inputs(case, seed):
    g = _gen(seed)
    N, Kd = case["N"], case["K"]
    w = _nvfp4_ckpt(g, N, Kd) if case["fmt"] == "nvfp4" else _mxfp4_ckpt(g, 1, N, Kd, 118, 126)
    return w, _randn(g, case["M"], Kd).to(torch.bfloat16)


def prepare(case, seed):
    st = SimpleNamespace(kind=case["kind"])
    if st.kind == "moe":
        L, w13, w2, st.x, st.logits = _moe_inputs(case, seed)
        st.W13, st.W2 = K.prepare_mxfp4_weights(*w13), K.prepare_mxfp4_weights(*w2)
        st.E, st.topk = L["E"], L["topk"]
        st.layer = SimpleNamespace(_r9k_tables=None)           # what router and experts share
        st.bufs = route.RouteBuffers(st.x.device, st.E, st.topk)
        st.experts = R9700Mxfp4Experts.standalone(st.W13.wsr, st.W2.wsr)
        st.experts.r9k_layer = st.layer
    elif st.kind == "shared":
        shared.register()
        w1, w2, st.wg, st.x = _shared_inputs(case, seed)
        st.W1, st.W2 = K.prepare_mxfp4_weights(*w1), K.prepare_mxfp4_weights(*w2)
    elif st.kind == "dense":
        w, st.x = _dense_inputs(case, seed)
        st.layer = SimpleNamespace()
        if case["fmt"] == "nvfp4":
            st.layer.weight_packed, st.layer.weight_scale, st.layer.weight_global_scale = map(_data, w)
            st.layer.logical_widths = [case["N"]]
            NV.prepare_native_dense_layer(st.layer)
            st.forward = NV.native_dense_forward
        else:
            st.layer.weight, st.layer.weight_scale = _data(w[0][0]), _data(w[1][0])
            LX.prep_dense(st.layer)
            st.forward = LX.apply_dense
    else:
        st.ckpt = list(map(_data, _nvfp4_ckpt(_gen(seed), case["N"], case["K"])))
        st.widths = [case["N"]]
    return st


def _data(t):
    return torch.nn.Parameter(t, requires_grad=False)


def run(st):
    if st.kind == "moe":
        numel = st.x.shape[0] * st.topk
        r = route.route_step(st.logits, st.x, st.topk, True, st.E, st.bufs,
                             dual_blk=route.dual_wanted(st.layer, numel, st.E),
                             wide=route.split_planned(st.layer, numel, st.E))
        w, ids, st.layer._r9k_tables = r
        out = torch.empty_like(st.x)
        st.experts.apply(out, st.x, st.W13.wq, st.W2.wq, w, ids, "silu", st.E, None, None, None, None, None, None,
                         False)
        return out, w, ids
    if st.kind == "shared":
        W1, W2 = st.W1, st.W2
        return torch.ops.r9700.shared_expert(st.x, W1.wq, W1.wsr, W2.wq, W2.wsr, st.wg, W1.N, W1.K, W2.N, W2.K, False,
                                             False)
    if st.kind == "dense":
        return st.forward(st.layer, st.x)
    layer = SimpleNamespace(logical_widths=st.widths)
    layer.weight_packed, layer.weight_scale, layer.weight_global_scale = st.ckpt
    NV.convert_dense_layer(layer)
    LX.prep_dense(layer)
    return layer.weight, layer.weight_scale


# --------------------------------------------------------------------------------------------------- work
def _touched(L, T):
    """Distinct experts that T tokens reach, over one seeded routing."""
    g = torch.Generator().manual_seed(7)
    logits = torch.randn(T, L["E"], generator=g)
    if L["zipf"]:
        logits = logits - L["zipf"] * torch.log(torch.arange(1, L["E"] + 1).float())
    return int(logits.topk(L["topk"], dim=1).indices.unique().numel())


def _mx_bytes(N, Kd):
    return N * Kd // 2 + N * Kd // 32


def work(case):
    if case["kind"] == "moe":
        L, T = LAYERS[case["layer"]], case["T"]
        H, I = L["H"], L["I"]
        expert = _mx_bytes(2 * I, H) + _mx_bytes(H, I)
        io = T * (2 * H + 2 * L["E"] + 2 * H + 8 * L["topk"])   # x, logits, out, weights and ids
        return {"bytes": _touched(L, T) * expert + io, "flops": 6 * T * L["topk"] * H * I}
    if case["kind"] == "shared":
        H, I, T = case["H"], case["I"], case["T"]
        return {"bytes": _mx_bytes(2 * I, H) + _mx_bytes(H, I) + 2 * H + 4 * T * H, "flops": 6 * T * H * I}
    N, Kd = case["N"], case["K"]
    if case["kind"] == "dense":
        M = case["M"]
        w = _mx_bytes(N, Kd) if case["fmt"] == "mxfp4" else N * Kd // 2 + N * Kd // 16 + 4 * N
        return {"bytes": w + 2 * M * (N + Kd), "flops": 2 * M * N * Kd}
    return {"bytes": N * Kd // 2 + N * Kd // 16 + _mx_bytes(N, Kd) + N, "flops": 0}


def tolerance(case):
    """How far an implementation that sums in another order may be off: about four times what a torch restatement of
    the path's roundings (fp32 or fp64 sums) shows. A dense linear differs by flips of its one bf16 rounding (rel 1e-4,
    largest 2^-7). A layer rounds gate_up to bf16 and then to fp8: a bf16 flip now and then moves an fp8 code by a
    step, 1/16 to 1/8 of one value, which the down product carries into a row (rel 1e-3, largest 0.11 of the output's
    root mean square). Indices and codes are exact."""
    if case["kind"] == "load":
        return "exact"
    if case["kind"] == "dense":
        return {"rel": 5e-4, "max": 0.03}
    return {"rel": 4e-3, "max": 0.4, "differ": 0.0}


# -------------------------------------------------------------------------------------------------- exact
_E2M1 = (0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0, -0.0, -0.5, -1.0, -1.5, -2.0, -3.0, -4.0, -6.0)


def _codes(packed):
    lut = torch.tensor(_E2M1, device=packed.device, dtype=torch.float64)
    return lut[torch.stack((packed & 15, packed >> 4), dim=-1).reshape(packed.shape[0], -1).int()]


def _mxfp4(packed, e8):
    """Checkpoint tensors of one matrix -> fp64 [N, K]."""
    s = torch.pow(2.0, e8.double() - 127.0)
    return _codes(packed) * s.repeat_interleave(32, dim=1)


def _fp8_rows(x):
    """Rows through the path's activation format: e4m3 codes of x * 448 / amax, times amax / 448."""
    amax = x.abs().amax(dim=1, keepdim=True)
    one = torch.where(amax > 0, amax, torch.ones_like(amax))
    return (x * (448.0 / one)).to(torch.float8_e4m3fn).double() * (amax / 448.0)


def _mlp(xq, w1, w2):
    h = xq @ w1.t()
    g, u = h.chunk(2, dim=1)
    return _fp8_rows(g * torch.sigmoid(g) * u) @ w2.t()


def exact(case, seed):
    if case["kind"] == "moe":
        L, w13, w2, x, logits = _moe_inputs(case, seed)
        p = torch.softmax(logits.double(), dim=1)
        ids = logits.double().sort(dim=1, descending=True, stable=True).indices[:, :L["topk"]]
        w = p.gather(1, ids)
        w = w / w.sum(dim=1, keepdim=True)
        xq = _fp8_rows(x.double())
        out = torch.zeros_like(xq)
        order = ids.reshape(-1).sort(stable=True)
        ends = torch.bincount(order.values, minlength=L["E"]).cumsum(0).tolist()
        for e in range(L["E"]):
            rows = order.indices[(ends[e - 1] if e else 0):ends[e]]
            if rows.numel():
                t = rows // L["topk"]
                y = _mlp(xq[t], _mxfp4(w13[0][e], w13[1][e]), _mxfp4(w2[0][e], w2[1][e]))
                out.index_add_(0, t, y * w.reshape(-1)[rows].unsqueeze(1))
        return out, w, None
    if case["kind"] == "shared":
        w1, w2, wg, x = _shared_inputs(case, seed)
        xd = x.double()
        y = _mlp(_fp8_rows(xd), _mxfp4(w1[0][0], w1[1][0]), _mxfp4(w2[0][0], w2[1][0]))
        return y * torch.sigmoid(xd @ wg.double()).unsqueeze(1)
    if case["kind"] == "dense":
        w, x = _dense_inputs(case, seed)
        if case["fmt"] == "nvfp4":
            W = _codes(w[0]) * w[1].double().repeat_interleave(16, dim=1) / w[2].double()
        else:
            W = _mxfp4(w[0][0], w[1][0])
        return _fp8_rows(x.double()) @ W.t()
    return None
