"""The calls whose speed this framework is held to: attention, one transformer
block and the cocktail-party head, over the sizes, masks, types and options
that its configurations, tests and training step use.

``listed()`` gives the fixed cases and ``draw(rng)`` further ones of the same
ranges.  ``prepare`` makes on the GPU what a caller holds before the call
(inputs, metadata, the module with its weights), ``run`` is one call through
the public entry points, ``exact`` the same outputs in 64-bit torch,
``work`` the bytes and operations the call cannot do without, and
``tolerance`` how far another correct implementation at the same precision may
be from it.
"""
from __future__ import annotations

import math

import torch

from kerneldev_amd import flash_attention
from kerneldev_amd.attention import AttentionPlan, build_plan, build_plan_from_tokens
from kerneldev_amd.gpt import Block
from kerneldev_amd.span_head import span_scores
from kerneldev_amd.synth import CONFIG3_LAYOUT, CONFIG4_LAYOUT, CocktailLayout, cocktail_batch

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
DEVICE = "cuda:0"


# ------------------------------------------------------------------- cases
def _attention(name, B, H, T, d, **opts):
    """One flash_attention call: forward, and with ``backward`` the gradients too."""
    case = dict(name=name, kind="attention", B=B, H=H, T=T, d=d, dtype="bf16", mask="causal", precision="tf32",
                qk_dtype="bf16", hadamard=False, outliers=False, backward=True, lens=False, strided=False)
    case.update(opts)
    return case


def listed():
    return [
        # the fp32 golden configuration: the smallest training call, all launches and latency
        _attention("fp32_small", 2, 4, 256, 64, dtype="fp32", precision="ieee"),
        # causal language-model training at head dim 64
        _attention("causal_train", 8, 16, 2048, 64),
        # cocktail-party training batches at head dim 64, the mask from the collate's metadata tensors
        _attention("cocktail_train", 16, 12, 1024, 64, mask="cocktail"),
        # long cocktail-party sequences with outlier channels, rotated Q and K: the headline benchmark
        _attention("cocktail_long", 2, 32, 8192, 128, mask="cocktail", hadamard=True, outliers=True),
        # the same with fp8 scores
        _attention("cocktail_long_fp8", 2, 32, 8192, 128, mask="cocktail", hadamard=True, outliers=True,
                   qk_dtype="fp8_e4m3"),
        # scoring one prompt: forward only, the plan from the tokens, projections' strided views, odd length
        _attention("score_one", 1, 12, 1531, 64, mask="tokens", backward=False, strided=True),
        # fine-tuning on one long sequence: few heads, odd length
        _attention("one_sequence", 1, 8, 4095, 128),
        # the largest head dim
        _attention("causal_d256", 2, 8, 4096, 256),
        # fp32 training, where the products run in full precision
        _attention("causal_fp32", 2, 8, 4096, 128, dtype="fp32"),
        # a small model on a padded batch: fp16, narrow heads, ragged lengths
        _attention("ragged_fp16", 4, 8, 777, 32, dtype="fp16", mask="cocktail", lens=True, strided=True),
        # one layer of the GPT model's training step at its specified size
        dict(name="gpt_block", kind="block", B=8, T=2048, dim=768, heads=12, hidden=2048, backward=True),
        # the cocktail-party head of that model: span scores and the gradient of the hidden state
        dict(name="span_head", kind="head", B=8, T=2048, dim=768, backward=True),
    ]


def _log_int(rng, lo, hi):
    """An integer in [lo, hi], spread over its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.49)))))))


def draw(rng):
    kind = rng.choices(("train", "score", "block", "head"), (12, 4, 2, 2))[0]
    if kind == "block":
        heads = rng.choice((4, 8, 12))
        return dict(kind="block", B=_log_int(rng, 1, 8), T=_log_int(rng, 128, 2048), dim=64 * heads, heads=heads,
                    hidden=rng.choice((1024, 1536, 2048)), backward=rng.random() < 0.7)
    if kind == "head":
        return dict(kind="head", B=_log_int(rng, 1, 16), T=_log_int(rng, 256, 4096), dim=rng.choice((256, 512, 768, 1024)),
                    backward=rng.random() < 0.7)
    dtype = rng.choices(("bf16", "fp16", "fp32"), (6, 2, 2))[0]
    d = rng.choices((16, 32, 64, 128, 256), (1, 2, 6, 5, 2))[0]
    T = _log_int(rng, 64, 8192)
    if rng.random() < 0.4:
        T = max(64, T // 64 * 64)
    # no dearer than the largest listed case of the type, and the tensors of a moderate size
    cells = (1 << 28) * 128 if dtype == "fp32" else (1 << 30) * 128
    most = max(1, min(512, cells // (T * T * d), (1 << 27) // (T * d)))
    BH = _log_int(rng, 1, most)
    B = max(b for b in (1, 2, 4, 8, 16) if b <= max(1, min(BH, _log_int(rng, 1, 16))))
    H = max(1, min(64, BH // B))
    mask = rng.choices(("causal", "all", "cocktail", "tokens"), (4, 1, 5, 1))[0]
    if T < 128 and mask in ("cocktail", "tokens"):
        mask = "causal"
    case = _attention("", B, H, T, d, dtype=dtype, mask=mask, backward=kind == "train", strided=rng.random() < 0.5,
                      lens=mask != "tokens" and rng.random() < 0.25,
                      precision=rng.choices(("tf32", "ieee", "bf16"), (7, 1, 1))[0])
    if dtype != "fp32":
        case["hadamard"] = d in (64, 128) and rng.random() < 0.3
        case["outliers"] = case["hadamard"]
        if dtype == "bf16" and d >= 64 and case["precision"] != "ieee" and rng.random() < 0.15:
            case["qk_dtype"] = "fp8_e4m3"
    del case["name"]
    return case


# ------------------------------------------------------------------ inputs
def _layout(T):
    """A cocktail-party layout for rows of T tokens: the configurations' own, or one in proportion."""
    if T == 8192:
        return CONFIG4_LAYOUT
    if 1024 <= T <= 2048:
        return CONFIG3_LAYOUT
    return CocktailLayout((max(2, T // 32), max(4, T // 10)), (max(8, T // 4), max(12, T // 2)), (4, 8),
                          (max(2, T // 64), max(4, T // 20)))


def _normal(shape, seed, dtype):
    g = torch.Generator(DEVICE).manual_seed(seed)
    return torch.randn(shape, generator=g, device=DEVICE, dtype=torch.float32).to(dtype)


def _inputs(case, seed):
    """Tensors of one case (all made from the seed), before any of them requires a gradient."""
    s = {}
    if case["kind"] == "attention":
        B, H, T, d = case["B"], case["H"], case["T"], case["d"]
        dt = DTYPES[case["dtype"]]
        g = torch.Generator("cpu").manual_seed(seed)
        for i, name in enumerate(("q", "k", "v", "do")):
            # strided: [B, H, T, d] views of [B, T, H, d] memory, as projections leave them
            x = _normal((B, T, H, d) if case["strided"] else (B, H, T, d), 8 * seed + i, torch.float32)
            x = x.transpose(1, 2) if case["strided"] else x
            if case["outliers"] and i < 3:  # 1% of the channels of every head, 20 times as large
                pick = torch.rand(H, d, generator=g).argsort(dim=1)[:, : math.ceil(0.01 * d)]
                mult = torch.ones(H, d).scatter_(1, pick, 20.0).to(DEVICE)
                x = x * mult[None, :, None, :]
            s[name] = x.to(dt)
        if case["mask"] in ("cocktail", "tokens"):
            tokens, in_span, span_id, is_prefix = cocktail_batch(B, T, _layout(T), seed)
            s["tokens"] = tokens.to(DEVICE)
            s["in_span"], s["span_id"], s["is_prefix"] = in_span.to(DEVICE), span_id.to(DEVICE), is_prefix.to(DEVICE)
        if case["lens"]:
            s["lens"] = torch.randint(max(1, T // 2), T + 1, (B,), generator=g, dtype=torch.int32).to(DEVICE)
    elif case["kind"] == "block":
        B, T, dim, hidden = case["B"], case["T"], case["dim"], case["hidden"]
        s["x"] = _normal((B, T, dim), 8 * seed, torch.bfloat16)
        s["dy"] = _normal((B, T, dim), 8 * seed + 1, torch.bfloat16)
        tokens, s["in_span"], s["span_id"], s["is_prefix"] = (
            x.to(DEVICE) for x in cocktail_batch(B, T, _layout(T), seed))
        shapes = dict(q=(dim, dim), k=(dim, dim), v=(dim, dim), o=(dim, dim), w1=(hidden, dim), w3=(hidden, dim),
                      w2=(dim, hidden))
        for i, (n, shape) in enumerate(shapes.items()):  # weights of a trained size: unit-variance projections
            s[n] = (_normal(shape, 8 * seed + 100 + i, torch.float32) / math.sqrt(shape[1])).to(torch.bfloat16)
    else:
        B, T, dim = case["B"], case["T"], case["dim"]
        lay = _layout(T)  # (always eight spans, so that the scores' shape is the case's and not the seed's)
        lay = CocktailLayout(lay.prefix_bytes, lay.context, (8, 8), lay.span_bytes)
        s["tokens"] = cocktail_batch(B, T, lay, seed)[0].to(DEVICE)
        s["h"] = _normal((B, T, dim), 8 * seed, torch.bfloat16)
        s["ds"] = _normal((B, 8), 8 * seed + 1, torch.float32)
    return s


def prepare(case, seed):
    s = _inputs(case, seed)
    s["case"] = case
    if case["kind"] == "attention":
        for n in ("q", "k", "v"):
            s[n].requires_grad_(case["backward"])
    elif case["kind"] == "block":
        blk = Block(case["dim"], case["heads"], case["hidden"]).to(DEVICE).to(torch.bfloat16)
        with torch.no_grad():
            for lin, n in _linears(blk):
                lin.weight.copy_(s.pop(n))
        s["block"] = blk
        s["x"].requires_grad_(case["backward"])
        d = case["dim"] // case["heads"]
        # the model builds one plan per step and hands it to each of its layers
        s["plan"] = AttentionPlan(build_plan(case["B"], case["T"], d, s["x"].device, 0, s["in_span"], s["span_id"],
                                             s["is_prefix"]), case["B"], case["T"], d)
    else:
        s["h"].requires_grad_(case["backward"])
    return s


def _linears(blk):
    return ((blk.attn.q_proj, "q"), (blk.attn.k_proj, "k"), (blk.attn.v_proj, "v"), (blk.attn.o_proj, "o"),
            (blk.mlp.w1, "w1"), (blk.mlp.w3, "w3"), (blk.mlp.w2, "w2"))


# --------------------------------------------------------------------- run
def run(s):
    case = s["case"]
    if case["kind"] == "block":
        blk = s["block"]
        if not case["backward"]:
            with torch.no_grad():
                return blk(s["x"], None, None, None, s["plan"])
        y = blk(s["x"], None, None, None, s["plan"])
        weights = [lin.weight for lin, _ in _linears(blk)]
        return (y, *torch.autograd.grad(y, [s["x"], *weights], s["dy"]))
    if case["kind"] == "head":
        if not case["backward"]:
            with torch.no_grad():
                return span_scores(s["tokens"], s["h"])
        scores = span_scores(s["tokens"], s["h"])
        return (scores, *torch.autograd.grad(scores, s["h"], s["ds"]))
    opts = dict(causal=case["mask"] != "all", precision=case["precision"], qk_dtype=case["qk_dtype"],
                hadamard=case["hadamard"], out_layout="bthd" if case["strided"] else "bhtd")
    if case["mask"] == "tokens":
        opts["plan"] = build_plan_from_tokens(s["tokens"], case["d"], rule="fallback")
    elif case["mask"] == "cocktail":
        opts.update(in_span=s["in_span"], span_id=s["span_id"], is_prefix=s["is_prefix"])
    if case["lens"]:
        opts["lens"] = s["lens"]
    if not case["backward"]:
        with torch.no_grad():
            return flash_attention(s["q"], s["k"], s["v"], return_lse=True, **opts)
    o = flash_attention(s["q"], s["k"], s["v"], **opts)
    return (o, *torch.autograd.grad(o, (s["q"], s["k"], s["v"]), s["do"]))


# ------------------------------------------------------- the same in 64 bits
def _fallback_metadata(tokens):
    """in_span, span_id, is_prefix that a model derives from the tokens alone: a
    span from its [SPAN] (3) up to but not including its [ES] (4), the prefix
    through the first [CLS] (1), -1 at [MASKQ] (5)."""
    n_span, n_es = (tokens == 3).cumsum(1), (tokens == 4).cumsum(1)
    in_span = n_span > n_es
    span_id = torch.where(in_span, n_span, torch.zeros_like(n_span))
    span_id = torch.where(tokens == 5, torch.full_like(span_id, -1), span_id)
    cls = (tokens == 1).long()
    return in_span, span_id, ((cls.cumsum(1) - cls) == 0) & cls.any(1, keepdim=True)


def _dense_mask(case, s, b):
    """Which key j each query i of batch row b sees, bool [T, T]."""
    T = case["T"]
    i = torch.arange(T, device=DEVICE)
    order = i[:, None] >= i[None, :]
    if case["kind"] == "attention" and case["mask"] in ("causal", "all"):
        ok = order if case["mask"] == "causal" else torch.ones_like(order)
    else:
        if case["kind"] == "attention" and case["mask"] == "tokens":
            S, sid, P = (x[b] for x in _fallback_metadata(s["tokens"]))
        else:
            S, sid, P = s["in_span"][b], s["span_id"][b], s["is_prefix"][b]
        M = sid == -1
        C = ~(S | P | M)
        own = S & (sid > 0)
        ok = ((P | C | M)[:, None] & P[None, :]) | (S[:, None] & C[None, :]) | (M[:, None] & S[None, :])
        ok |= C[:, None] & C[None, :] & order
        ok |= own[:, None] & own[None, :] & (sid[:, None] == sid[None, :])
    if case.get("lens"):
        live = i < int(s["lens"][b])
        ok = ok & live[:, None] & live[None, :]
    return ok


def _softmax(S, ok):
    """Row softmax over the allowed keys (zeros on a row without any) and its base-2 log-sum."""
    S = S.masked_fill(~ok, -math.inf)
    m = S.amax(-1, keepdim=True)
    P = torch.exp(S - torch.where(m == -math.inf, torch.zeros_like(m), m))
    l = P.sum(-1, keepdim=True)
    lse = (m + torch.log(l)).squeeze(-1) * math.log2(math.e)
    return P / torch.where(l > 0, l, torch.ones_like(l)), lse


def _rotation(d):
    """diag(s) H_d / sqrt(d), with the signs of seed 0."""
    g = torch.Generator("cpu").manual_seed(0)
    signs = torch.randint(0, 2, (d,), generator=g, dtype=torch.int64).double() * 2 - 1
    Hd = torch.ones(1, 1, dtype=torch.float64)
    while Hd.shape[0] < d:
        Hd = torch.cat([torch.cat([Hd, Hd], 1), torch.cat([Hd, -Hd], 1)], 0)
    return (signs[:, None] * Hd / math.sqrt(d)).to(DEVICE)


def _fp8(x):
    """The values that per-head e4m3 scores see: x to 8 bits with its largest magnitude at 448."""
    amax = x.abs().max()
    scale = torch.where(amax > 0, amax, torch.full_like(amax, 448.0)) / 448.0
    return (x / scale).clamp(-448, 448).float().to(torch.float8_e4m3fn).double() * scale


def _exact_attention(case, s):
    B, H, T, d = case["B"], case["H"], case["T"], case["d"]
    f64 = dict(dtype=torch.float64, device=DEVICE)
    fp8 = case["qk_dtype"] != "bf16"
    outs = [torch.zeros(B, H, T, d, **f64) for _ in range(4 if case["backward"] else 1)]
    lse = torch.zeros(B, H, T, **f64)
    R = _rotation(d) if fp8 and case["hadamard"] else None
    sc = d ** -0.5
    for b in range(B):
        ok = _dense_mask(case, s, b)
        for h in range(H):
            q, k, v, do = (s[n][b, h].double() for n in ("q", "k", "v", "do"))
            if fp8:  # scores from 8-bit copies of the (rotated) operands; gradients straight through to those
                if R is not None:
                    q, k = ((x @ R).to(torch.bfloat16).double() for x in (q, k))
                else:
                    q, k = (x.to(torch.bfloat16).double() for x in (q, k))
                S = _fp8(q) @ _fp8(k).T * sc
            else:  # (a rotation of both operands leaves their products as they are)
                S = q @ k.T * sc
            P, lse[b, h] = _softmax(S, ok)
            o = P @ v
            outs[0][b, h] = o
            if case["backward"]:
                dS = P * (do @ v.T - (do * o).sum(-1, keepdim=True))
                dq, dk = dS @ k * sc, dS.T @ q * sc
                outs[1][b, h], outs[2][b, h] = (dq, dk) if R is None else (dq @ R.T, dk @ R.T)
                outs[3][b, h] = P.T @ do
    return tuple(outs) if case["backward"] else (outs[0], lse)


def _exact_block(case, s):
    B, T, dim, nh = case["B"], case["T"], case["dim"], case["heads"]
    w = {n: s[n].double().requires_grad_() for n in ("q", "k", "v", "o", "w1", "w3", "w2")}
    x = s["x"].double().requires_grad_()

    def norm(t):
        return t * torch.rsqrt(t.pow(2).mean(-1, keepdim=True) + 1e-6)

    total = [torch.zeros_like(t) for t in (x, *w.values())]
    ys = []
    for b in range(B):  # one batch row at a time: the [heads, T, T] scores in 64 bits
        ok = _dense_mask(case, s, b)
        xb = x[b]
        n1 = norm(xb)
        q, k, v = ((n1 @ w[n].T).view(T, nh, -1).transpose(0, 1) for n in ("q", "k", "v"))
        P = _softmax(q @ k.transpose(1, 2) * (dim // nh) ** -0.5, ok)[0]
        hmid = xb + (P @ v).transpose(0, 1).reshape(T, dim) @ w["o"].T
        n2 = norm(hmid)
        y = hmid + (torch.nn.functional.silu(n2 @ w["w1"].T) * (n2 @ w["w3"].T)) @ w["w2"].T
        ys.append(y.detach())
        if case["backward"]:
            for t, g in zip(total, torch.autograd.grad(y, [x, *w.values()], s["dy"][b].double())):
                t += g
    y = torch.stack(ys)
    return (y, *total) if case["backward"] else y


def _exact_head(case, s):
    tokens, h = s["tokens"], s["h"].double().requires_grad_()
    rows = []
    for b in range(case["B"]):
        st, ed = (tokens[b] == 3).nonzero().flatten().tolist(), (tokens[b] == 4).nonzero().flatten().tolist()
        ctx = h[b, int((tokens[b] == 2).nonzero()[0])]
        row = [h[b, i + 1:j].mean(0) @ ctx for i, j in zip(st, ed) if i + 1 < j]
        rows.append(torch.nn.functional.pad(torch.stack(row), (0, s["ds"].shape[1] - len(row))))
    scores = torch.stack(rows)
    if not case["backward"]:
        return scores.detach()
    return (scores.detach(), *torch.autograd.grad(scores, h, s["ds"].double()))


def exact(case, seed):
    s = _inputs(case, seed)
    return {"attention": _exact_attention, "block": _exact_block, "head": _exact_head}[case["kind"]](case, s)


# -------------------------------------------------------- work and tolerance
def _allowed(case):
    """Score entries of one head summed over the batch (of the layouts of seed 0; lens: three quarters of T)."""
    B, T = case["B"], case["T"]
    if case["kind"] == "attention" and case["mask"] in ("causal", "all"):
        t = T * 3 // 4 if case["lens"] else T
        return B * (t * (t + 1) // 2 if case["mask"] == "causal" else t * t)
    tokens, in_span, span_id, is_prefix = cocktail_batch(B, T, _layout(T), 0)
    n = 0
    for b in range(B):
        S, M, P = (int(x[b].sum()) for x in (in_span, span_id == -1, is_prefix))
        C = T - S - M - P
        own = span_id[b][in_span[b]].bincount().square().sum()
        n += (P + C + M) * P + C * (C + 1) // 2 + S * C + M * S + int(own)
    return n * 9 // 16 if case.get("lens") else n


def work(case):
    B, T = case["B"], case["T"]
    if case["kind"] == "head":  # the hidden state's span rows read; with the gradient, all of it written
        h = B * T * case["dim"] * 2
        return {"bytes": h + B * T * 8 + (h if case["backward"] else 0), "flops": B * T * case["dim"]}
    if case["kind"] == "block":
        dim, hidden = case["dim"], case["hidden"]
        weights = 4 * dim * dim + 3 * dim * hidden
        back = case["backward"]
        return {"bytes": 2 * ((4 if back else 2) * B * T * dim + (2 if back else 1) * weights),
                "flops": (6 if back else 2) * B * T * weights + (14 if back else 4) * dim * _allowed(case)}
    H, d = case["H"], case["d"]
    one = B * H * T * d * (4 if case["dtype"] == "fp32" else 2)
    return {"bytes": (8 if case["backward"] else 4) * one + (0 if case["backward"] else 4 * B * H * T),
            "flops": (14 if case["backward"] else 4) * d * H * _allowed(case)}


def tolerance(case):
    """About four times the measured distance from ``exact`` (where the harness's bound allows it)."""
    if case["kind"] == "block":  # bf16 activations between the block's layers: 0.004 to 0.011 measured
        return {"rel": 0.03, "max": 0.3}
    if case["kind"] == "head":  # fp32 scores, a bf16 gradient: 0.0017
        return {"rel": 7e-3, "max": 0.05}
    if case["dtype"] == "fp32":
        # fp32 throughout: 0.2e-6 to 2e-6; narrow heads at "tf32" carry 16 bits
        return {"rel": 1e-4 if case["d"] <= 32 and case["precision"] == "tf32" else 1e-5}
    if case["qk_dtype"] != "bf16":  # scores from 8-bit operands, whose rounding the order of the rotation's sums decides
        return {"rel": 0.03, "max": 0.8}
    if case["hadamard"]:  # the rotated operands are rounded to 16 bits before the scores: 0.02 with outlier channels
        return {"rel": 0.03, "max": 0.8}
    if case["dtype"] == "fp16":  # rounding of the outputs (2e-4), and of P and dS at "bf16"
        return {"rel": 1e-3 if case["precision"] != "bf16" else 3e-3, "max": 0.05}
    return {"rel": 7e-3 if case["precision"] != "bf16" else 0.02, "max": 0.1 if case["precision"] != "bf16" else 0.3}
