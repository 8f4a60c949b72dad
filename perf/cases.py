"""The work the framework's speed is measured on: calls a user's program makes through the public entry points, over
the sizes, types and options they are used with.  Every case is a dict of plain values; `prepare` makes what the
program has in hand (module, weights, inputs), `run` is one pass, `exact` the same result in 64-bit torch.

Kinds:
  layer     MoESwiGLU under no_grad (sampling and evaluation of a denoiser block): output, routing ids and weights
  train     MoESwiGLU forward and backward (a training step of a denoiser block): the same, and every gradient
  block     PoziomkaMoE (the BailingMoeV2 block of the frozen text encoder): int8 experts, sigmoid group-limited gate,
            shared expert
  infer     moe_infer of a block fused with fuse_moe, routed by the model's own softmax gate: bf16, fp16 or int8 experts
  grouped   moe_triton.grouped_mm with its gather, row scale and scatter
"""
from __future__ import annotations

import math

import torch
import torch.nn as nn
import torch.nn.functional as F

DEV = "cuda"


def listed():
    return [
        # the smallest layer: 512 tokens of a small denoiser, where launches and latency count
        dict(name="layer_512", kind="layer", T=512, d=256, E=8, k=2, h=512, skew=False),
        # eight 256 px images
        dict(name="layer_2048", kind="layer", T=2048, d=1024, E=8, k=2, h=2048, skew=False),
        # about 16k tokens packed from images of several resolutions: skewed experts, two of them never routed
        dict(name="layer_16384_skew", kind="layer", T=16384, d=1536, E=16, k=2, h=4096, skew=True),
        # a training step on eight 256 px images
        dict(name="train_2048", kind="train", T=2048, d=1024, E=8, k=2, h=2048, skew=False, weights="bf16"),
        # a training step with fp32 master weights, an odd token count, top-3 and widths off the tile sizes
        dict(name="train_3001_fp32", kind="train", T=3001, d=760, E=12, k=3, h=1352, skew=True, weights="fp32"),
        # a training step on four 1024 px images: the largest
        dict(name="train_16384", kind="train", T=16384, d=1536, E=16, k=2, h=4096, skew=False, weights="bf16"),
        # the text encoder's block on one short prompt, on a batch of captions, and on a full packed call
        dict(name="block_64", kind="block", T=64, d=2048, E=128, k=8, h=320, n_group=8, topk_group=2, shared_h=320),
        dict(name="block_1500", kind="block", T=1500, d=2048, E=128, k=8, h=320, n_group=8, topk_group=2,
             shared_h=320),
        dict(name="block_8192", kind="block", T=8192, d=2048, E=128, k=8, h=320, n_group=8, topk_group=2,
             shared_h=320),
        # fused blocks of other checkpoints: a short prompt on int8 experts, a batch of captions in fp16
        dict(name="infer_24_int8", kind="infer", T=24, d=2048, E=64, k=6, h=1408, dtype="bf16", quant=True),
        dict(name="infer_777_fp16", kind="infer", T=777, d=1536, E=60, k=4, h=1024, dtype="fp16", quant=False),
        # the grouped product by itself, gathered, scaled and scattered, with widths off the tile sizes
        dict(name="grouped_6000", kind="grouped", T=2000, k=3, E=24, K=1000, N=1512, dtype="bf16", quant=False),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("layer", "layer", "train", "train", "block", "block", "infer", "infer", "grouped"))
    if kind in ("layer", "train"):
        E = rng.randint(4, 24)
        # (a step renormalises its routing weights: with top-1 they are constant and the router has no gradient)
        k = rng.randint(2 if kind == "train" else 1, min(4, E))
        d, h = 8 * rng.randint(32, 200), 8 * rng.randint(48, 520)
        T = _log_int(rng, 128, 16384)
        # no more work than the largest listed step
        T = max(64, min(T, int(16384 * 2 * 1536 * 4096 / (k * d * h))))
        c = dict(kind=kind, T=T, d=d, E=E, k=k, h=h, skew=rng.random() < 0.4)
        if kind == "train":
            c["weights"] = rng.choice(("bf16", "bf16", "fp32"))
        return c
    if kind == "block":
        T = _log_int(rng, 1, 8192)
        d = rng.choice((1024, 1536, 2048))
        E, h = rng.choice((64, 128)), 32 * rng.randint(6, 14)
        return dict(kind=kind, T=T, d=d, E=E, k=rng.choice((4, 6, 8)), h=h, n_group=8, topk_group=rng.choice((2, 4)),
                    shared_h=h)
    dtype, quant = rng.choice((("bf16", False), ("fp16", False), ("bf16", True), ("fp16", True)))
    if kind == "infer":
        E = rng.randint(16, 96)
        return dict(kind=kind, T=_log_int(rng, 1, 4096), d=16 * rng.randint(32, 128), E=E, k=rng.randint(2, 8),
                    h=16 * rng.randint(20, 90), dtype=dtype, quant=quant)
    return dict(kind=kind, T=_log_int(rng, 32, 8192), k=rng.randint(1, 4), E=rng.randint(2, 32),
                K=rng.choice((8 * rng.randint(16, 256), rng.randint(100, 2000))),
                N=rng.choice((16 * rng.randint(8, 128), rng.randint(100, 2000))), dtype=dtype, quant=quant)


# ---------------------------------------------------------------------------------------------------------------
# Inputs, and the state a program keeps
# ---------------------------------------------------------------------------------------------------------------
_DT = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}


class _Expert(nn.Module):
    """An expert of a DeepSeek / Bailing style block, as fuse_moe reads it."""

    def __init__(self, d, h, **f):
        super().__init__()
        self.gate_proj = nn.Linear(d, h, bias=False, **f)
        self.up_proj = nn.Linear(d, h, bias=False, **f)
        self.down_proj = nn.Linear(h, d, bias=False, **f)
        self.act_fn = nn.SiLU()


class _Block(nn.Module):
    def __init__(self, d, h, E, **f):
        super().__init__()
        self.experts = nn.ModuleList([_Expert(d, h, **f) for _ in range(E)])

    def moe_infer(self, x, topk_ids, topk_weight):
        raise NotImplementedError("replaced by fuse_moe")


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _randn(g, *shape, std=1.0, dtype=torch.bfloat16):
    return (torch.randn(*shape, generator=g, device=DEV) * std).to(dtype)


def _zipf_bias(E, g):
    """Router bias of skewed experts: -1.2 ln(rank) over a random order, the last two (of more than four) off."""
    b = torch.empty(E, device=DEV)
    order = torch.randperm(E, generator=g, device=DEV)
    b[order] = -1.2 * torch.log(torch.arange(1, E + 1, device=DEV, dtype=torch.float32))
    if E > 4:
        b[order[-2:]] = -math.inf
    return b


def _quant(w):
    """(E, K, N) -> int8 and its per-(expert, column) bf16 scale."""
    s = w.float().abs().amax(dim=1).clamp(min=1e-8) / 127
    return (w.float() / s.unsqueeze(1)).round().clamp(-127, 127).to(torch.int8), s.to(torch.bfloat16)


def prepare(case, seed):
    g = _gen(seed)
    kind = case["kind"]
    with torch.no_grad():
        if kind in ("layer", "train"):
            return _prepare_layer(case, g)
        if kind == "block":
            return _prepare_block(case, g)
        if kind == "infer":
            return _prepare_infer(case, g)
        return _prepare_grouped(case, g)


def _prepare_layer(c, g):
    from trenowanie_generatora_obrazkow_amd import MoESwiGLU
    train = c["kind"] == "train"
    m = MoESwiGLU(c["d"], c["h"], c["E"], c["k"], device=DEV, dtype=_DT[c.get("weights", "bf16")])
    for p, fan_in in ((m.router_weight, c["d"]), (m.w_gu, c["d"]), (m.w_d, c["h"])):
        p.normal_(0.0, fan_in ** -0.5, generator=g)
    if c["skew"]:
        m.logit_bias.copy_(_zipf_bias(c["E"], g))
    x = _randn(g, c["T"], c["d"])
    st = dict(case=c, m=m, x=x)
    if train:
        x.requires_grad_(True)
        st["dy"] = _randn(g, c["T"], c["d"])
    return st


def _prepare_block(c, g):
    from trenowanie_generatora_obrazkow_amd.poziomka import PoziomkaMoE
    d, E, h, sh = c["d"], c["E"], c["h"], c["shared_h"]
    with torch.device(DEV):
        m = PoziomkaMoE(d, h, E, c["k"], c["n_group"], c["topk_group"], 2.5, sh)
    m.gate.weight.normal_(0.0, d ** -0.5, generator=g)
    m.gate.expert_bias.normal_(0.0, 0.01, generator=g)
    s = m.shared_experts
    for lin in (s.gate_proj, s.up_proj, s.down_proj):
        lin.weight.normal_(0.0, lin.in_features ** -0.5, generator=g)
    for name, shape in (("_wgu", (E, d, 2 * h)), ("_wd", (E, h, d))):
        q, sc = _quant(_randn(g, *shape, std=shape[1] ** -0.5, dtype=torch.float32))
        getattr(m, name).copy_(q)
        getattr(m, name + "_s").copy_(sc)
    return dict(case=c, m=m.to(torch.bfloat16), x=_randn(g, c["T"], d))


def _prepare_infer(c, g):
    from trenowanie_generatora_obrazkow_amd.hf_compat import fuse_moe
    dt = _DT[c["dtype"]]
    model = nn.Sequential(_Block(c["d"], c["h"], c["E"], device="meta", dtype=dt)).to_empty(device=DEV)
    for p in model.parameters():
        p.normal_(0.0, p.shape[1] ** -0.5, generator=g)
    gate = _randn(g, c["E"], c["d"], std=c["d"] ** -0.5, dtype=torch.float32)
    x = _randn(g, c["T"], c["d"], dtype=dt)
    w, ids = (x.float() @ gate.t()).softmax(-1).topk(c["k"], dim=-1)
    fuse_moe(model, quant="int8" if c["quant"] else "")
    return dict(case=c, m=model[0], x=x, ids=ids, w=w / w.sum(-1, keepdim=True))


def _prepare_grouped(c, g):
    dt = _DT[c["dtype"]]
    T, k, E, K, N = c["T"], c["k"], c["E"], c["K"], c["N"]
    k = min(k, E)
    # ragged groups: the first third of the experts takes twice the load, the last one nothing
    load = torch.ones(E, device=DEV)
    load[: E // 3] = 2.0
    load[-1] = 0.0 if E > k else 1.0
    ids = torch.multinomial(load.expand(T, E), k, generator=g)
    order = ids.reshape(-1).argsort(stable=True)
    w = _randn(g, E, K, N, std=K ** -0.5, dtype=dt)
    w, ws = _quant(w) if c["quant"] else (w, None)
    return dict(case=c, a=_randn(g, T, K, dtype=dt), w=w, w_scale=ws,
                counts=torch.bincount(ids.reshape(-1), minlength=E), a_idx=(order // k).to(torch.int32),
                y_idx=order.to(torch.int32), scale=torch.rand(T * k, generator=g, device=DEV).to(dt))


# ---------------------------------------------------------------------------------------------------------------
# One pass
# ---------------------------------------------------------------------------------------------------------------
def run(st):
    kind = st["case"]["kind"]
    if kind == "layer":
        m = st["m"]
        with torch.no_grad():
            y = m(st["x"])
        return [y, m.last_topk_ids, m.last_topk_weight]
    if kind == "train":
        m, x = st["m"], st["x"]
        m.zero_grad(set_to_none=True)
        x.grad = None
        y = m(x)
        y.backward(st["dy"])
        return [y.detach(), m.last_topk_ids, m.last_topk_weight.detach(), x.grad, m.router_weight.grad, m.w_gu.grad,
                m.w_d.grad]
    if kind == "block":
        return st["m"](st["x"])
    if kind == "infer":
        return st["m"].moe_infer(st["x"], st["ids"], st["w"])
    from trenowanie_generatora_obrazkow_amd.moe_triton import grouped_mm, make_schedule
    return grouped_mm(st["a"], st["w"], st["counts"], make_schedule(st["counts"], st["a_idx"].numel()),
                      a_idx=st["a_idx"], y_idx=st["y_idx"], scale=st["scale"], w_scale=st["w_scale"])


# ---------------------------------------------------------------------------------------------------------------
# What a pass cannot do without
# ---------------------------------------------------------------------------------------------------------------
def _experts_hit(T, k, E):
    """Experts with at least one row when T tokens pick k of E evenly (whose weights have to be read)."""
    return E * (1.0 - (1.0 - min(k, E) / E) ** T)


def work(case):
    c = case
    kind, T, k, E = c["kind"], c["T"], c["k"], c["E"]
    hit = _experts_hit(T, k, E)
    if kind == "grouped":
        k = min(k, E)
        K, N, M = c["K"], c["N"], T * k
        b = 2 * T * K + hit * K * N * (1 if c["quant"] else 2) + 2 * M * N + 12 * M
        return dict(bytes=int(b), flops=2 * M * K * N)
    d, h, M = c["d"], c["h"], T * k
    flops = 6 * M * d * h
    act = 4 * T * d  # x read, the output written
    if kind == "layer":
        return dict(bytes=int(act + 2 * E * d + hit * 6 * d * h + 8 * M), flops=flops + 2 * T * E * d)
    if kind == "train":
        ws = 4 if c["weights"] == "fp32" else 2
        # weights read for the forward and the backward and their gradients written, x and dy read, y and dx written
        return dict(bytes=int(2 * act + ws * 2 * E * d + ws * 6 * hit * d * h + 8 * M),
                    flops=3 * (flops + 2 * T * E * d))
    if kind == "block":
        b = act + 2 * E * d + hit * 3 * d * h + hit * 2 * (2 * h + d) + 6 * d * c["shared_h"]
        return dict(bytes=int(b), flops=flops + 2 * T * E * d + 6 * T * d * c["shared_h"])
    b = act + hit * 3 * d * h * (1 if c["quant"] else 2) + 12 * M
    return dict(bytes=int(b), flops=flops)


# Four times the difference seen against the 64-bit results, which round nothing on the way: here the routed
# activations, each expert's output row and, in a step, the gradients at the same places are rounded to 16 bits (seen:
# 4.6e-3 in bf16 and 5.7e-4 in fp16; the single product, rounded once, 1.7e-3 and 2.1e-4).  "differ": routing ids of
# near ties.
def tolerance(case):
    fp16 = case.get("dtype") == "fp16"
    if case["kind"] == "grouped":
        return dict(rel=8.5e-4 if fp16 else 7e-3)
    tol = dict(rel=2.3e-3 if fp16 else 1.8e-2)
    if case["kind"] in ("layer", "train"):
        tol["differ"] = 1e-3
    return tol


# ---------------------------------------------------------------------------------------------------------------
# The same in 64 bits
# ---------------------------------------------------------------------------------------------------------------
def _experts64(x, ids, w, wgu_of, wd_of, E):
    """sum over a token's slots of w * (silu(x Wg) * (x Wu)) Wd, an expert at a time."""
    out = torch.zeros_like(x)
    for e in range(E):
        rows, slot = (ids == e).nonzero(as_tuple=True)
        if rows.numel() == 0:
            continue
        g, u = (x[rows] @ wgu_of(e)).chunk(2, dim=-1)
        out = out.index_add(0, rows, ((F.silu(g) * u) @ wd_of(e)) * w[rows, slot, None])
    return out


def exact(case, seed):
    st = prepare(case, seed)
    kind = case["kind"]
    if kind in ("layer", "train"):
        return _exact_layer(st, case)
    with torch.no_grad():
        if kind == "block":
            return _exact_block(st, case)
        if kind == "infer":
            m = st["m"]
            return _experts64(st["x"].double(), st["ids"], st["w"].double(), _stack64(m._wgu, m._wgu_s),
                              _stack64(m._wd, m._wd_s), case["E"])
        w = _stack64(st["w"], st["w_scale"])
        a, y_idx, scale = st["a"].double(), st["y_idx"].long(), st["scale"].double()
        y = torch.empty(y_idx.numel(), case["N"], device=DEV, dtype=torch.float64)
        r0 = 0
        for e, n in enumerate(st["counts"].tolist()):
            r = slice(r0, r0 + n)
            y[y_idx[r]] = (a[st["a_idx"][r].long()] @ w(e)) * scale[r, None]
            r0 += n
        return y


def _stack64(w, s):
    return lambda e: w[e].double() if s is None else w[e].double() * s[e].double()


def _exact_layer(st, c):
    m = st["m"]
    train = c["kind"] == "train"
    with torch.set_grad_enabled(train):
        x, wr = (t.detach().bfloat16().double().requires_grad_(train) for t in (st["x"], m.router_weight))
        # one 64-bit leaf per expert; fp32 master weights enter the products rounded to bf16
        wgu, wd = ([w[e].detach().bfloat16().double().requires_grad_(train) for e in range(c["E"])]
                   for w in (m.w_gu, m.w_d))
        p = (x @ wr.t() + m.logit_bias.double()).softmax(-1)
        w, ids = p.topk(c["k"], dim=-1)
        w = w / w.sum(-1, keepdim=True)
        y = _experts64(x, ids, w, wgu.__getitem__, wd.__getitem__, c["E"])
        out = [y.detach(), ids.to(torch.int32), w.detach()]
        if train:
            y.backward(st["dy"].double())
            grads = [torch.stack([t.grad if t.grad is not None else torch.zeros_like(t) for t in ts])
                     for ts in (wgu, wd)]
            out += [x.grad, wr.grad, *grads]
    return out


def _exact_block(st, c):
    m, x = st["m"], st["x"].double()
    T, E, ng = c["T"], c["E"], c["n_group"]
    scores = torch.sigmoid(x @ m.gate.weight.double().t())
    routing = scores + m.gate.expert_bias.double()
    group = routing.view(T, ng, -1).topk(2, dim=-1)[0].sum(-1)
    keep = torch.zeros_like(group).scatter_(1, group.topk(c["topk_group"], dim=-1)[1], 1.0).bool()
    keep = keep.unsqueeze(-1).expand(T, ng, E // ng).reshape(T, E)
    ids = routing.masked_fill(~keep, -math.inf).topk(c["k"], dim=-1)[1]
    w = scores.gather(1, ids)
    w = w / (w.sum(-1, keepdim=True) + 1e-20) * m.scaling
    y = _experts64(x, ids, w, _stack64(m._wgu, m._wgu_s), _stack64(m._wd, m._wd_s), E)
    s = m.shared_experts
    gate, up, down = (lin.weight.double().t() for lin in (s.gate_proj, s.up_proj, s.down_proj))
    return y + (F.silu(x @ gate) * (x @ up)) @ down
