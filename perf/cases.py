"""What is measured: the fused fp8 MoE layer as a serving program calls it, and
the packing of its weights when a model is loaded.

A layer case is one call of the public Python entry points on a buffer that
the program keeps (``get_symm_buffer_for_mega_moe``): ``fp8_mega_moe``,
``bf16_fp8_mega_moe``, or ``fp8_mega_moe_compute`` + ``fp8_mega_moe_reduce``.
A load case is one call of ``transform_weights_for_mega_moe``.

A case's fields:
  kind     "layer" or "load"
  E, K, H, I   experts, experts per token, hidden and intermediate size
  T, cap   tokens of the call, and tokens the kept buffer was made for
  x        "fp8" (quantised by the caller) or "bf16" (folded inside the layer)
  scaled   UE8M0 block scales, or raw e4m3 operands
  zipf     exponent of a Zipf router bias (0: none)
  mfma     "bf16" (default arithmetic) or "fp8" (the opt-in fp8 MFMA path)
  split    compute and reduce as two calls

Inputs are made with plain torch from the seed alone: x ~ N(0, 1), weights ~
N(0, 0.02), softmax top-k router on N(0, 1) logits.
"""
from __future__ import annotations

import math

import torch

import mini_mega_amd as mm


def _layer(name, T, cap, E=256, K=8, H=6144, I=2048, x="fp8", scaled=True, zipf=0.0, mfma="bf16",
           split=False):
    return {"name": name, "kind": "layer", "E": E, "K": K, "H": H, "I": I, "T": T, "cap": cap,
            "x": x, "scaled": scaled, "zipf": zipf, "mfma": mfma, "split": split}


def listed():
    return [
        # one user's next token: eight experts' weights, launches and latency
        _layer("token-1", T=1, cap=512),
        # a handful of users: most pairs alone on their expert
        _layer("decode-13", T=13, cap=512),
        # a decode batch with an uneven router; most experts hold 1 to 8 rows
        _layer("decode-96-skew", T=96, cap=512, zipf=1.1),
        # bf16 activations and raw e4m3 weights, as a checkpoint without block
        # scales is served
        _layer("decode-203-bf16-raw", T=203, cap=512, x="bf16", scaled=False),
        # the benchmark's decode batch: 16 rows per expert
        _layer("decode-512", T=512, cap=512),
        # a prefill chunk, 64 rows per expert
        _layer("chunk-2048", T=2048, cap=8192),
        # the same with a skewed router, compute and reduce called apart
        _layer("chunk-2048-skew", T=2048, cap=8192, zipf=1.1, split=True),
        # the benchmark's largest prefill: 256 rows per expert
        _layer("prefill-8192", T=8192, cap=8192),
        # the same on the opt-in fp8 MFMA path, at a ragged length
        _layer("prefill-7001-fp8mfma", T=7001, cap=8192, mfma="fp8"),
        # smaller models of the tests' shapes: a few MB to 0.3 GB of weights
        _layer("small-200", T=200, cap=200, E=32, H=1024, I=512),
        _layer("medium-777", T=777, cap=1024, E=64, K=4, H=2048, I=768, x="bf16"),
        # loading one layer of an expert-parallel eighth of the model
        {"name": "load-32-experts", "kind": "load", "E": 32, "K": 8, "H": 6144, "I": 2048,
         "T": 0, "cap": 0, "x": "fp8", "scaled": True, "zipf": 0.0, "mfma": "bf16",
         "split": False},
    ]


def draw(rng):
    """One more case: token counts from 1 to 8192 over their logarithm, the
    full model half of the time and otherwise layers down to a few MB, every
    input type, scale mode and routing of the listed cases."""
    if rng.random() < 0.1:
        return {"kind": "load", "E": rng.randint(2, 32), "K": 8, "H": 256 * rng.randint(4, 24),
                "I": 256 * rng.randint(1, 8), "T": 0, "cap": 0, "x": "fp8",
                "scaled": rng.random() < 0.7, "zipf": 0.0, "mfma": "bf16", "split": False}
    T = max(1, min(8192, int(round(math.exp(rng.uniform(0.0, math.log(8192.0)))))))
    if rng.random() < 0.5:
        E, K, H, I = 256, 8, 6144, 2048
    else:
        E, K = rng.choice([16, 32, 64, 128]), rng.choice([2, 4, 6, 8])
        H, I = 256 * rng.randint(4, 24), rng.choice([128, 256, 512, 768, 1024, 1280, 1536, 2048])
    c = _layer("", T=T, cap=max(T, rng.choice([512, 2048, 8192])), E=E, K=K, H=H, I=I,
               x="bf16" if rng.random() < 0.3 else "fp8", scaled=rng.random() < 0.75,
               zipf=1.1 if rng.random() < 0.35 else 0.0,
               mfma="fp8" if T >= 1024 and rng.random() < 0.3 else "bf16",
               split=rng.random() < 0.2)
    del c["name"]
    return c


# ------------------------------------------------------------------ inputs --
def _gen(seed, stream):
    g = torch.Generator(device="cuda")
    g.manual_seed((int(seed) * 1000003 + stream) % (1 << 62))
    return g


def _pow2_scale(amax):
    """The power of two >= amax.clamp(1e-4) / 448, and its UE8M0 byte."""
    bits = (amax.float().clamp(min=1e-4) / 448.0).view(torch.int32)
    e = ((bits >> 23) & 0xFF) + ((bits & 0x7FFFFF) != 0).to(torch.int32)
    e = e.clamp(1, 254)
    return (e << 23).view(torch.float32), e.to(torch.uint8)


def _quant_rows(v):
    """[n, 128 m] -> e4m3 with one UE8M0 scale per row and 128 columns."""
    n, k = v.shape
    b = v.view(n, k // 128, 128)
    s, byte = _pow2_scale(b.abs().amax(dim=2))
    q = (b / s.unsqueeze(2).to(v.dtype)).float().to(torch.float8_e4m3fn)
    return q.view(n, k), byte


def _quant_blocks(w):
    """[n, k] -> e4m3 with one UE8M0 scale per 128 x 128 block."""
    n, k = w.shape
    b = w.view(n // 128, 128, k // 128, 128)
    s, byte = _pow2_scale(b.abs().amax(dim=3).amax(dim=1))
    q = (b / s.view(n // 128, 1, k // 128, 1)).to(torch.float8_e4m3fn)
    return q.view(n, k), byte


W2_RAW_SCALE = 4096.0   # raw W2 is stored times this power of two, undone in the top-k weights


def _expert(case, g):
    """The next expert's weights: (W1 [2I, H], its scales, W2 [H, I], scales)."""
    H, I = case["H"], case["I"]
    w1 = torch.randn((2 * I, H), generator=g, device="cuda").mul_(0.02)
    w2 = torch.randn((H, I), generator=g, device="cuda").mul_(0.02)
    if case["scaled"]:
        return _quant_blocks(w1) + _quant_blocks(w2)
    return (w1.to(torch.float8_e4m3fn), None,
            w2.mul_(W2_RAW_SCALE).clamp_(-448.0, 448.0).to(torch.float8_e4m3fn), None)


def _weights(case, seed):
    """All experts' logical weights: ((W1, scales), (W2, scales))."""
    E, H, I = case["E"], case["H"], case["I"]
    w1 = torch.empty((E, 2 * I, H), dtype=torch.float8_e4m3fn, device="cuda")
    w2 = torch.empty((E, H, I), dtype=torch.float8_e4m3fn, device="cuda")
    s1 = torch.empty((E, 2 * I // 128, H // 128), dtype=torch.uint8, device="cuda")
    s2 = torch.empty((E, H // 128, I // 128), dtype=torch.uint8, device="cuda")
    g = _gen(seed, 1)
    for e in range(E):
        a, sa, b, sb = _expert(case, g)
        w1[e].copy_(a)
        w2[e].copy_(b)
        if case["scaled"]:
            s1[e].copy_(sa)
            s2[e].copy_(sb)
    return ((w1, s1), (w2, s2)) if case["scaled"] else (w1, w2)


def _route(case, g, device):
    """Softmax top-k router: experts int64 [T, K], their weights fp32 [T, K]."""
    T, E, K = case["T"], case["E"], case["K"]
    logits = torch.randn((T, E), generator=g, device=device, dtype=torch.float64)
    if case["zipf"]:
        rank = torch.randperm(E, generator=g, device=device).double() + 1.0
        bias = -0.4 * case["zipf"] * rank.log()
        bias[rank > E - E // 16] = -math.inf
        logits = logits + bias
    p, idx = logits.softmax(dim=1).topk(K, dim=1)
    return idx, (p / p.sum(dim=1, keepdim=True)).float()


def _tokens(case, seed):
    """x bf16 [T, H], the routes int64 [T, K] and their weights fp32 [T, K]."""
    x = torch.randn((case["T"], case["H"]), generator=_gen(seed, 2), device="cuda").to(torch.bfloat16)
    idx, w = _route(case, _gen(seed, 3), "cuda")
    if not case["scaled"]:
        w = w / W2_RAW_SCALE
    return x, idx.contiguous(), w.contiguous()


def _x_fp8(case, x):
    if case["scaled"]:
        return _quant_rows(x.float())
    return x.float().clamp(-448.0, 448.0).to(torch.float8_e4m3fn), None


def prepare(case, seed):
    if case["kind"] == "load":
        l1, l2 = _weights(case, seed)
        return {"kind": "load", "l1": l1, "l2": l2}
    T = case["T"]
    l1, l2 = mm.transform_weights_for_mega_moe(*_weights(case, seed))
    buf = mm.get_symm_buffer_for_mega_moe(
        None, case["E"], case["cap"], case["K"], case["H"], case["I"],
        mma_type="bf16xfp8" if case["x"] == "bf16" else "fp8xfp8")
    buf.mfma_fp8 = case["mfma"] == "fp8"
    x, idx, w = _tokens(case, seed)
    if case["x"] == "bf16":
        buf.x[:T].copy_(x)
    else:
        q, sf = _x_fp8(case, x)
        buf.x.view(torch.uint8)[:T].copy_(q.view(torch.uint8))
        if sf is not None:
            buf.x_sf[:T].copy_(sf)
    buf.topk_idx[:T].copy_(idx)
    buf.topk_weights[:T].copy_(w)
    y = torch.empty((T, case["H"]), dtype=torch.bfloat16, device="cuda")
    kind = "split" if case["split"] else case["x"]
    return {"kind": kind, "T": T, "l1": l1, "l2": l2, "buf": buf, "y": y, "counts": buf.counts()}


def run(state):
    kind = state["kind"]
    if kind == "load":
        (w1, s1), (w2, s2) = _pairs(mm.transform_weights_for_mega_moe(state["l1"], state["l2"]))
        return {"w1": w1, "s1": s1, "w2": w2, "s2": s2}
    y, buf = state["y"], state["buf"]
    if kind == "split":
        mm.fp8_mega_moe_compute(state["l1"], state["l2"], buf, state["T"])
        mm.fp8_mega_moe_reduce(y, buf)
    elif kind == "bf16":
        mm.bf16_fp8_mega_moe(y, state["l1"], state["l2"], buf)
    else:
        mm.fp8_mega_moe(y, state["l1"], state["l2"], buf)
    return {"y": y, "counts": state["counts"]}


def _pairs(packed):
    return tuple(p if isinstance(p, tuple) else (p, None) for p in packed)


# ------------------------------------------------------- work and tolerance --
def work(case):
    E, K, H, I, T = (case[k] for k in ("E", "K", "H", "I", "T"))
    expert = 3 * H * I
    if case["scaled"]:
        expert += 3 * (H // 128) * (I // 128)
    if case["kind"] == "load":
        return {"bytes": 2 * E * expert, "flops": 0}
    # experts that get a token, counted on one routing of these sizes
    g = torch.Generator().manual_seed(5)
    active = int(_route(case, g, "cpu")[0].unique().numel())
    xb = 2 * H if case["x"] == "bf16" else H + (H // 128 if case["scaled"] else 0)
    return {"bytes": active * expert + T * (xb + 2 * H + 12 * K), "flops": 6 * H * I * T * K}


def tolerance(case):
    """Packing moves bytes.  The layer rounds its intermediate to e4m3 and its
    expert rows and result to bf16, so another order of its fp32 sums flips
    single roundings."""
    if case["kind"] == "load":
        return "exact"
    if case["mfma"] == "fp8":
        return {"rel": 1.5e-2, "max": 0.2}
    return {"rel": 1e-2, "max": 0.1}


# -------------------------------------------------------------- in 64 bits --
def _dequant_blocks(q, s):
    w = q.double()
    if s is None:
        return w
    f = torch.exp2(s.double() - 127.0)
    n, k = q.shape
    return (w.view(n // 128, 128, k // 128, 128) * f.view(n // 128, 1, k // 128, 1)).view(n, k)


def _dequant_rows(q, s):
    v = q.double()
    if s is None:
        return v
    n, k = q.shape
    f = torch.exp2(s.double() - 127.0)
    return (v.view(n, k // 128, 128) * f.unsqueeze(2)).view(n, k)


def exact(case, seed):
    """The layer with the operands' and the intermediate's declared e4m3
    formats and every product and sum in 64 bits."""
    if case["kind"] == "load":
        return None
    I = case["I"]
    x, idx, w = _tokens(case, seed)
    xd = _dequant_rows(*_x_fp8(case, x))
    y = torch.zeros((case["T"], case["H"]), dtype=torch.float64, device="cuda")
    g = _gen(seed, 1)
    for e in range(case["E"]):
        w1, s1, w2, s2 = _expert(case, g)
        tok, k = (idx == e).nonzero(as_tuple=True)
        if tok.numel() == 0:
            continue
        gu = torch.mm(xd[tok], _dequant_blocks(w1, s1).t())
        gate, up = gu[:, :I], gu[:, I:]
        h = gate * torch.sigmoid(gate) * up
        if case["scaled"]:
            h = _dequant_rows(*_quant_rows(h.contiguous()))
        else:
            h = h.clamp(-448.0, 448.0).float().to(torch.float8_e4m3fn).double()
        o = torch.mm(h, _dequant_blocks(w2, s2).t())
        y.index_add_(0, tok, o * w[tok, k].double().unsqueeze(1))
    return {"y": y, "counts": None}
