"""What a user of mxfp8gg has it do, as measurable cases.

Each case is one pass of a program through the package's public entry points:
an MoE layer being served or trained, a grouped linear layer, a weight
gradient, the casts of the expert weights, and the drop-in calls of the
reference's sweeps and of torchao's trainer.  Hidden size 7168, intermediate
size 2048 and 32 experts on one GPU are the DeepSeek-V3 layer of this
repository's benchmark; the rest are small, odd or generic sizes.

`exact` computes what a pass returns in 64 bits with plain torch: every GEMM
and the activation in float64.  The MXFP8 rounding of the operands and the
bf16 rounding of the tensors that are cast are part of what the ops define and
are kept; the outputs themselves are not rounded.
"""
import math
import sys
from pathlib import Path

import numpy as np
import torch

_PACKAGE = str(Path.cwd() / "mxfp8-grouped-gemm_amd")
if _PACKAGE not in sys.path:
    sys.path.insert(0, _PACKAGE)

import mxfp8gg  # noqa: E402
from mxfp8gg import workloads  # noqa: E402

DEV = "cuda"


def listed():
    return [
        # The smallest call: four experts, 320 tokens, a 256 -> 512 layer.
        # Latency of two launches and their host path.
        dict(name="linear_tiny", kind="linear", routing="dirichlet", tokens=320, experts=4, n=512,
             k=256),
        # Gate+up projection of a forward pass over a large batch, ragged groups.
        dict(name="linear_gate_up", kind="linear", routing="dirichlet", tokens=65536, experts=32,
             n=4096, k=7168),
        # Down projection of the same pass: short contraction, wide output.
        dict(name="linear_down", kind="linear", routing="dirichlet", tokens=65536, experts=32,
             n=7168, k=2048),
        # Weight gradient of gate+up with fp32 accumulation buffers, skewed
        # routing with two empty experts, from the bf16 tensors a trainer holds.
        dict(name="wgrad_fp32", kind="wgrad", routing="zipf", tokens=65536, experts=32, n=4096,
             k=7168),
        # Serving, decode: 64 sequences, one token each, weights cast at load.
        dict(name="serve_decode", kind="serve", tokens=64, topk=8, experts=32, hidden=7168,
             inter=2048),
        # Serving, prefill of a prompt of 1900 tokens: about 475 rows per expert.
        dict(name="serve_prefill", kind="serve", tokens=1900, topk=8, experts=32, hidden=7168,
             inter=2048),
        # The full training step of the layer, 16384 tokens x top-8, weights
        # cast in the step (they changed in the optimizer step before).
        dict(name="train_step", kind="train", tokens=16384, topk=8, experts=32, hidden=7168,
             inter=2048, cached=False),
        # A micro-batch of gradient accumulation: 1000 tokens, the weights'
        # casts kept from the first micro-batch.
        dict(name="train_micro_batch", kind="train", tokens=1000, topk=8, experts=32, hidden=7168,
             inter=2048, cached=True),
        # A small differentiable grouped linear layer, odd group sizes:
        # forward and both gradients.
        dict(name="autograd_small", kind="autograd", routing="dirichlet", tokens=1537, experts=8,
             n=1024, k=1056),
        # The reference's sweep: unscaled e4m3 operands, equal groups, forward
        # and bf16 weight gradient.
        dict(name="unscaled_sweep", kind="unscaled", tokens=32768, experts=4, n=2048, k=7168),
        # torchao's trainer calls: FLOOR casts with row-major scales along both
        # axes, forward and fp32 weight gradient.
        dict(name="torchao_linear", kind="torchao", tokens=32768, experts=8, n=7168, k=2048),
        # After every optimizer step: both casts of the gate+up weights.
        dict(name="cast_weights", kind="weights", experts=32, n=4096, k=7168),
    ]


def _log(rng, lo, hi, step=1):
    """A multiple of `step` in [lo, hi], spread over the logarithm."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return max(lo, min(hi, int(round(v / step)) * step))


def draw(rng):
    """One more case of the listed kinds: sizes from the smallest to the largest
    listed ones, odd ones among them."""
    most = _cost(dict(kind="train", tokens=16384, topk=8, experts=32, hidden=7168, inter=2048,
                      cached=False))
    while True:
        kind = rng.choice(["linear", "linear", "wgrad", "serve", "serve", "train", "train",
                           "autograd", "unscaled", "torchao", "weights"])
        e = rng.choice([1, 2, 4, 8, 16, 24, 32, 48, 64])
        routing = rng.choice(["dirichlet", "zipf", "equal"])
        if kind in ("linear", "wgrad", "autograd"):
            c = dict(kind=kind, routing=routing, tokens=_log(rng, 64, 65536), experts=e,
                     n=_log(rng, 256, 7168, 32), k=_log(rng, 256, 7168, 32))
        elif kind in ("serve", "train"):
            topk = rng.choice([1, 2, 4, 6, 8])
            c = dict(kind=kind, tokens=_log(rng, 1, 16384), topk=topk, experts=max(e, topk),
                     hidden=_log(rng, 512, 7168, 32), inter=_log(rng, 256, 2048, 32))
            if kind == "train":
                c["cached"] = rng.random() < 0.5
                c["tokens"] = max(16, c["tokens"])
        elif kind in ("unscaled", "torchao"):
            per = _log(rng, 128, 16384, 32)
            c = dict(kind=kind, tokens=min(131072 // e // 32 * 32, per) * e, experts=e,
                     n=_log(rng, 256, 7168, 128), k=_log(rng, 256, 7168, 128))
        else:
            c = dict(kind=kind, experts=e, n=_log(rng, 256, 7168, 32),
                     k=_log(rng, 256, 7168, 32))
        if _cost(c) <= most:
            return c


# ---------------------------------------------------------------------------
# sizes and work
# ---------------------------------------------------------------------------
def _cost(case):
    """Seconds a pass cannot go below at nominal rates (for comparing cases)."""
    w = work(case)
    return max(w["bytes"] / 8e12, w["flops"] / 5e15)


def _sizes(case, seed):
    """Tokens of every expert."""
    m, e, how = case["tokens"], case["experts"], case.get("routing", "equal")
    if how == "dirichlet":
        return workloads.dirichlet_sizes(m, e, seed)
    if how == "zipf":
        return workloads.zipf_sizes(m, e, 1.2, seed, empty=2 if e >= 8 else 0)
    return np.full(e, m // e) + (np.arange(e) < m % e)


def _hit(case):
    """Experts that a routing of this many slots reaches, about."""
    e, slots = case["experts"], case["tokens"] * case["topk"]
    return e * (1.0 - (1.0 - 1.0 / e) ** slots)


def work(case):
    kind = case["kind"]
    if kind in ("serve", "train"):
        t, h, f = case["tokens"], case["hidden"], case["inter"]
        slots, e = t * case["topk"], _hit(case)
        gemm = 2 * slots * 3 * f * h
        wts = 3 * f * h
        if kind == "serve":
            # x and out in bf16, MXFP8 weights of the experts that are reached
            return {"bytes": 4 * t * h + e * wts * 33 / 32, "flops": gemm}
        # x, dout, out, dx in bf16; weights (bf16, or their two MXFP8 casts)
        # read, bf16 gradients of all experts written
        read = case["experts"] * wts * (2 * 33 / 32 if case["cached"] else 2)
        return {"bytes": 8 * t * h + read + case["experts"] * wts * 2, "flops": 3 * gemm}
    n, k, e = case["n"], case["k"], case["experts"]
    if kind == "weights":
        return {"bytes": e * n * k * (2 + 2 * 33 / 32), "flops": 0}
    m = case["tokens"]
    if kind == "linear":
        return {"bytes": m * (2 * k + 2 * n) + e * n * k * 33 / 32, "flops": 2 * m * n * k}
    if kind == "wgrad":
        return {"bytes": m * (2 * k + 2 * n) + e * n * k * 4, "flops": 2 * m * n * k}
    if kind == "autograd":
        return {"bytes": 4 * m * (k + n) + 4 * e * n * k, "flops": 6 * m * n * k}
    if kind == "unscaled":
        # forward: x, w read, y written; weight gradient: dy, x read, dw written
        return {"bytes": m * (2 * k + 3 * n) + e * n * k * 3, "flops": 4 * m * n * k}
    # torchao: x, dy, weights read, y and fp32 dw written
    return {"bytes": m * (2 * k + 4 * n) + e * n * k * (33 / 32 + 4), "flops": 4 * m * n * k}


def tolerance(case):
    """About four times what the path differs from `exact` by.

    Single layers: the bf16 rounding of the outputs (rel 1.7e-3, max 4.2e-3).
    The expert FFN: also h, the activation and their casts, each of which moves
    by a unit in the last place where a sum rounds the other way (rel 3.2e-3;
    max 0.03 for the output, 0.4 for weight gradients over few tokens).  fp32
    weight gradients: the matrix cores' accumulation (rel 1.5e-5, max 2.5e-4)."""
    kind = case["kind"]
    if kind == "weights":
        return "exact"
    if kind == "wgrad":
        return {"rel": 6e-5, "max": 1e-3}
    if kind == "serve":
        return {"rel": 1.3e-2, "max": 0.13}
    if kind == "train":
        return {"rel": 1.3e-2, "max": 0.9}
    return {"rel": 7e-3, "max": 1.7e-2}


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _bf16(gen, shape, scale=1.0):
    out = torch.empty(shape, dtype=torch.bfloat16, device=DEV)
    return out.normal_(0.0, scale, generator=gen)


def _ends(sizes):
    return torch.from_numpy(workloads.ends_of(sizes)).to(DEV)


def _activations(gen, m, k):
    """N(0, 1) with 1% of the values 20 times as large, as activations have."""
    x = _bf16(gen, (m, k), 0.5)
    return torch.where(torch.rand((m, k), generator=gen, device=DEV) < 0.01, x * 20, x)


def _routing(gen, case):
    """Distinct experts per token, popular experts drawn more often (Gumbel
    top-k over Zipf(1) preferences in a random order), softmax scores."""
    t, e, k = case["tokens"], case["experts"], case["topk"]
    pref = -torch.log(torch.arange(1, e + 1, device=DEV, dtype=torch.float32))
    pref = pref[torch.randperm(e, generator=gen, device=DEV)]
    u = torch.rand((t, e), generator=gen, device=DEV).clamp_(1e-7, 1 - 1e-7)
    idx = (pref - torch.log(-torch.log(u))).topk(k, dim=1).indices.to(torch.int32)
    scores = torch.randn((t, k), generator=gen, device=DEV).softmax(dim=1)
    return idx.contiguous(), scores


def prepare(case, seed):
    gen = torch.Generator(device=DEV).manual_seed(int(seed))
    kind = case["kind"]
    s = dict(kind=kind)
    if kind in ("serve", "train"):
        t, e, h, f = case["tokens"], case["experts"], case["hidden"], case["inter"]
        s["x"] = _bf16(gen, (t, h))
        s["idx"], s["scores"] = _routing(gen, case)
        s["w_gate_up"] = _bf16(gen, (e, 2 * f, h), 0.006 * math.sqrt(7168 / h))
        s["w_down"] = _bf16(gen, (e, h, f), 0.006 * math.sqrt(7168 / h))
        s["cache"] = None
        if kind == "train":
            s["dout"] = _bf16(gen, (t, h), 1e-3)
            for name in ("x", "scores", "w_gate_up", "w_down"):
                s[name].requires_grad_(True)
        if kind == "serve" or case["cached"]:
            s["cache"] = mxfp8gg.WeightCastCache()
            for name in ("w_gate_up", "w_down"):
                s["cache"].get(s[name])
        return s
    e, n, k = case["experts"], case["n"], case["k"]
    if kind == "weights":
        s["w"] = _bf16(gen, (e, n, k), 0.006)
        return s
    m = case["tokens"]
    sizes = _sizes(case, int(seed))
    s["offs"] = _ends(sizes)
    if kind == "linear":
        s["x"] = _activations(gen, m, k)
        s["w"], s["ws"] = mxfp8gg.to_mxfp8_dim0(_bf16(gen, (e, n, k), 0.006))
    elif kind == "wgrad":
        s["x"], s["dy"] = _bf16(gen, (m, k)), _bf16(gen, (m, n), 1e-3)
    elif kind == "autograd":
        s["x"] = _activations(gen, m, k).requires_grad_(True)
        s["w"] = _bf16(gen, (e, n, k), 0.02).requires_grad_(True)
        s["dy"] = _bf16(gen, (m, n), 1e-3)
    elif kind == "unscaled":
        s["x"] = _bf16(gen, (m, k)).to(torch.float8_e4m3fn)
        s["w"] = _bf16(gen, (e, n, k)).to(torch.float8_e4m3fn)
        s["go"] = _bf16(gen, (n, m)).to(torch.float8_e4m3fn)
        s["ia"] = _bf16(gen, (k, m)).to(torch.float8_e4m3fn)
    else:
        s["x"], s["dy"] = _activations(gen, m, k), _bf16(gen, (m, n), 1e-3)
        s["w"], s["ws"] = mxfp8gg.triton_to_mxfp8_dim0(_bf16(gen, (e, n, k), 0.006))
    return s


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def run(s):
    kind = s["kind"]
    if kind == "serve":
        with torch.no_grad():
            return mxfp8gg.moe_routed_ffn(s["x"], s["idx"], s["scores"], s["w_gate_up"],
                                          s["w_down"], weight_cache=s["cache"])
    if kind == "train":
        leaves = (s["x"], s["scores"], s["w_gate_up"], s["w_down"])
        out = mxfp8gg.moe_routed_ffn(s["x"], s["idx"], s["scores"], s["w_gate_up"], s["w_down"],
                                     weight_cache=s["cache"])
        dx, dscores, dwgu, dwd = torch.autograd.grad(out, leaves, s["dout"])
        return dict(out=out.detach(), dx=dx, dscores=dscores, dw_gate_up=dwgu, dw_down=dwd)
    if kind == "weights":
        (q, qs), (t, ts) = mxfp8gg.quant_weight_dual(s["w"])
        return dict(q=q.view(torch.uint8), qs=qs, t=t.view(torch.uint8), ts=ts)
    if kind == "linear":
        q, qs = mxfp8gg.to_mxfp8_dim0(s["x"])
        return mxfp8gg.fused_grouped_fwd(q, s["w"], s["offs"], qs, s["ws"])
    if kind == "wgrad":
        go, gos, pad = mxfp8gg.to_mxfp8_dim1(s["dy"], s["offs"])
        ia, ias, _ = mxfp8gg.to_mxfp8_dim1(s["x"], s["offs"])
        return mxfp8gg.wgrad_fused(go, ia, pad, gos, ias, out_dtype=torch.float32)
    if kind == "autograd":
        y = mxfp8gg.mxfp8_grouped_mm(s["x"], s["w"], s["offs"])
        dx, dw = torch.autograd.grad(y, (s["x"], s["w"]), s["dy"])
        return dict(y=y.detach(), dx=dx, dw=dw)
    if kind == "unscaled":
        return dict(y=mxfp8gg.fused_grouped_fwd(s["x"], s["w"], s["offs"]),
                    dw=mxfp8gg.wgrad_fused(s["go"], s["ia"], s["offs"], offs_kind="ends"))
    q, qs = mxfp8gg.triton_to_mxfp8_dim0(s["x"])
    y = mxfp8gg.triton_mxfp8_grouped_mm(q, s["w"], qs, s["ws"], s["offs"])
    go, gos = mxfp8gg.triton_to_mxfp8_dim1(s["dy"])
    ia, ias = mxfp8gg.triton_to_mxfp8_dim1(s["x"])
    return dict(y=y, dw=mxfp8gg.triton_mxfp8_wgrad(go.t(), gos, ia.t(), ias, s["offs"]))


# ---------------------------------------------------------------------------
# the same in 64 bits
# ---------------------------------------------------------------------------
def _mx(x, floor=False):
    """The MXFP8 value of finite bf16 x, 1x32 blocks along the last dimension, as
    float64: scale exponent ceil(log2(amax / 448)) (floor: floor(log2(amax)) - 8),
    payload rounded to e4m3."""
    b = x.reshape(-1, 32)
    amax = (b.view(torch.int16).to(torch.int32) & 0x7FFF).amax(dim=1, keepdim=True)
    e = (amax >> 7) - 8
    if not floor:
        e += ((amax & 0x7F) > 0x60).to(torch.int32)
    e = e.clamp_(1, 254)
    up = ((254 - e) << 23).view(torch.float32)
    back = ((e.to(torch.int64) - 127 + 1023) << 52).view(torch.float64)
    q = (b.float() * up).clamp_(-448, 448).to(torch.float8_e4m3fn)
    return (q.double() * back).reshape(x.shape)


def _mx_tokens(x, floor=False):
    """The token-axis cast of one expert's rows [m, C], padded to 32: [C, m32]."""
    m = x.shape[0]
    pad = torch.nn.functional.pad(x, (0, 0, 0, -m % 32))
    return _mx(pad.t().contiguous(), floor)


def _bounds(offs):
    ends = [0] + offs.tolist()
    return [(g, ends[g], ends[g + 1]) for g in range(len(ends) - 1)]


def _wide(*shape):
    return torch.zeros(shape, dtype=torch.float64, device=DEV)


def _bf(x):
    return x.to(torch.bfloat16)


def _exact_ffn(s, train):
    x, dev_w, dev_d = s["x"].detach(), s["w_gate_up"].detach(), s["w_down"].detach()
    scores = s["scores"].detach()
    (t, h), e, f, topk = x.shape, dev_w.shape[0], dev_d.shape[2], scores.shape[1]
    out = _wide(t, h)
    if train:
        dx, dscores = _wide(t, h), _wide(t * topk)
        dwgu, dwd = _wide(e, 2 * f, h), _wide(e, h, f)
    flat, sc = s["idx"].reshape(-1), scores.reshape(-1)
    for g in range(e):
        slots = (flat == g).nonzero()[:, 0]
        if not slots.numel():
            continue
        tok = slots // topk
        xr = x[tok]
        hid = _bf(_mx(xr) @ _mx(dev_w[g]).t()).double()
        gate, up = hid[:, :f], hid[:, f:]
        sig = 1 / (1 + torch.exp(-gate))
        act = _bf(gate * sig).double()
        a = _bf(act * up)
        y = _mx(a) @ _mx(dev_d[g]).t()
        out.index_add_(0, tok, y * sc[slots, None].double())
        if not train:
            continue
        dout = s["dout"][tok]
        dscores[slots] = (dout.double() * y).sum(dim=1)
        dy = _bf(dout.float() * sc[slots, None])
        da = _bf(_mx(dy) @ _mx(dev_d[g].t().contiguous()).t()).double()
        dact = _bf(da * up).double()
        dh = torch.cat([_bf(dact * sig * (1 + gate * (1 - sig))), _bf(da * act)], dim=1)
        dx.index_add_(0, tok, _mx(dh) @ _mx(dev_w[g].t().contiguous()).t())
        dwd[g] = _mx_tokens(dy) @ _mx_tokens(a).t()
        dwgu[g] = _mx_tokens(dh) @ _mx_tokens(xr).t()
    if not train:
        return out
    return dict(out=out, dx=dx, dscores=dscores.reshape(t, topk), dw_gate_up=dwgu, dw_down=dwd)


def exact(case, seed):
    kind = case["kind"]
    if kind == "weights":
        return None  # bytes
    s = prepare(dict(case, cached=False), seed)
    if kind in ("serve", "train"):
        return _exact_ffn(s, kind == "train")
    n, k, m, e = case["n"], case["k"], case["tokens"], case["experts"]
    groups = _bounds(s["offs"])
    if kind in ("linear", "wgrad", "autograd"):
        x = s["x"].detach()
        w = None
        if kind == "linear":  # the weights are given as MXFP8
            back = ((s["ws"].to(torch.int64) - 127 + 1023) << 52).view(torch.float64)
            w = s["w"].double() * back.repeat_interleave(32, dim=2)
        y = _wide(m, n) if kind != "wgrad" else None
        dx = _wide(m, k) if kind == "autograd" else None
        dw = _wide(e, n, k) if kind != "linear" else None
        for g, b, c in groups:
            if b == c:
                continue
            if kind == "linear":
                y[b:c] = _mx(x[b:c]) @ w[g].t()
                continue
            dw[g] = _mx_tokens(s["dy"][b:c]) @ _mx_tokens(x[b:c]).t()
            if kind == "autograd":
                wg = s["w"].detach()[g]
                y[b:c] = _mx(x[b:c]) @ _mx(wg).t()
                dx[b:c] = _mx(s["dy"][b:c]) @ _mx(wg.t().contiguous()).t()
        return y if kind == "linear" else dw if kind == "wgrad" else dict(y=y, dx=dx, dw=dw)
    y, dw = _wide(m, n), _wide(e, n, k)
    for g, b, c in groups:
        if kind == "unscaled":
            y[b:c] = s["x"][b:c].double() @ s["w"][g].double().t()
            dw[g] = s["go"][:, b:c].double() @ s["ia"][:, b:c].double().t()
        else:
            ws = s["ws"][g].contiguous().view(torch.uint8).to(torch.int64)
            back = ((ws - 127 + 1023) << 52).view(torch.float64).repeat_interleave(32, dim=1)
            y[b:c] = _mx(s["x"][b:c], True) @ (s["w"][g].double() * back).t()
            dw[g] = _mx_tokens(s["dy"][b:c], True) @ _mx_tokens(s["x"][b:c], True).t()
    return dict(y=y, dw=dw)
