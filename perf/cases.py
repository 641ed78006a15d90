"""Workloads of the attention and norm ops, for timing and for comparing two builds.

Each case is one call (or one training step) as a model's layer makes it, through the
public entry points: ``F.scaled_dot_product_attention``, ``kohakutt_amd.sdpa`` (key
lengths), ``kohakutt_amd.sdpa_varlen``, ``F.layer_norm`` and ``F.rms_norm``.

* ``listed()`` -- the fixed cases; ``draw(rng)`` -- one more case of the same ranges.
* ``prepare(case, seed)`` -- the inputs a program holds before the call, on the GPU.
* ``run(state)`` -- one call (``train``: the forward and the gradients of every input).
* ``exact(case, seed)`` -- the same outputs in float64, in plain torch.
* ``work(case)`` -- bytes and FLOPs the call cannot do without; ``tolerance(case)``.
"""

import math
import os
import sys

import torch
import torch.nn.functional as F

# The package of the tree the process runs in (its root is the working folder).
_PACKAGE_ROOT = os.path.abspath("kohaku-tt_amd")
if _PACKAGE_ROOT not in sys.path:
    sys.path.insert(0, _PACKAGE_ROOT)

import kohakutt_amd  # noqa: E402

_DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}


def _attn(name, kind="dense", **kw):
    case = {
        "name": name,
        "op": "attention",
        "kind": kind,  # dense | lengths (key counts per batch entry) | varlen (packed)
        "batch": 1,  # dense: batch entries; varlen: sequences
        "heads_q": 1,
        "heads_kv": 1,
        "seq_q": 1,  # varlen: the longest sequence; the others are drawn from [seq_min, seq_q]
        "seq_k": 1,
        "seq_min": 1,
        "dim": 64,
        "causal": False,
        "mask": "none",  # none | pad (bool [B, 1, 1, Sk]) | additive ([1, 1, Sq, Sk], q's dtype)
        "layout": "heads",  # heads: dense [B, H, S, D]; rows: views of [B, S, H * D] projections
        "dtype": "bf16",
        "train": False,
    }
    case.update(kw)
    return case


def _norm(name, kind, rows, width, dtype="bf16", train=False):
    return {"name": name, "op": "norm", "kind": kind, "rows": rows, "width": width, "dtype": dtype, "train": train}


def listed():
    return [
        # One token of a decoding batch through an RMSNorm: nothing but launch latency.
        _norm("rms_decode_8x2048", "rms", 8, 2048),
        # The input norm of a 640-wide image transformer block, one training step.
        _norm("ln_train_8192x640", "layer", 8192, 640, train=True),
        # A ViT-B/16 batch: 197 tokens (odd), q / k / v views of the projections.
        _attn("vit_32x12x197x64", batch=32, heads_q=12, heads_kv=12, seq_q=197, seq_k=197, layout="rows"),
        # Prefill of a small GQA language model (14 query heads over 2 K/V heads).
        _attn("prefill_gqa_14_2x2048x64", heads_q=14, heads_kv=2, seq_q=2048, seq_k=2048, causal=True),
        # Self-attention of a 1024-pixel diffusion UNet's 640-wide block, both CFG halves.
        _attn("unet_self_2x10x4096x64", batch=2, heads_q=10, heads_kv=10, seq_q=4096, seq_k=4096, layout="rows"),
        # The same block's cross-attention over 77 text tokens.
        _attn("unet_cross_2x10x4096_77x64", batch=2, heads_q=10, heads_kv=10, seq_q=4096, seq_k=77, layout="rows"),
        # Joint attention of a diffusion transformer at head dim 128: 4096 image tokens
        # and 300 text tokens (not a whole number of tiles).
        _attn("joint_24x4396x128", heads_q=24, heads_kv=24, seq_q=4396, seq_k=4396, dim=128),
        # Prefill with a full additive mask (a prefix / document mask).
        _attn("masked_16x2048x64", heads_q=16, heads_kv=16, seq_q=2048, seq_k=2048, mask="additive"),
        # A training step of the small GQA model's attention.
        _attn("train_gqa_14_2x2048x64", heads_q=14, heads_kv=2, seq_q=2048, seq_k=2048, causal=True, train=True),
        # A packed training batch of ragged sequences, GQA at head dim 128.
        _attn("varlen_train_8x1024_16_8x128", kind="varlen", batch=8, heads_q=16, heads_kv=8, seq_q=1024, seq_k=1024,
              seq_min=64, dim=128, causal=True, train=True),
        # One decoding step over a K/V cache with a padding mask.
        _attn("decode_mask_8x16_2x4096x128", batch=8, heads_q=16, heads_kv=2, seq_q=1, seq_k=4096, dim=128, mask="pad"),
        # One decoding step of a large serving batch, cache lengths as a tensor.
        _attn("decode_lengths_64x16_2x8192x128", kind="lengths", batch=64, heads_q=16, heads_kv=2, seq_q=1, seq_k=8192,
              dim=128),
    ]


# What a drawn attention case may cost: the largest listed one's FLOPs (forward plus the
# backward's 2.5 times).
_MOST_FLOPS = 4.0 * 128 * 24 * 4396 * 4396
_HEADS = [(14, 2), (12, 12), (16, 8), (16, 2), (10, 10), (24, 24), (32, 8), (8, 2), (16, 16), (6, 3)]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    """One more case.  Sequence lengths, batches, rows and widths are spread over the
    logarithm of their ranges, odd ones included."""
    what = rng.choice(["prefill", "prefill", "cross", "train", "train", "varlen", "decode", "decode", "norm", "norm"])
    if what == "norm":
        dtype = rng.choice(["bf16", "bf16", "bf16", "f16", "f32"])
        width = _log(rng, 64, 8192)
        if rng.random() < 0.8:
            width = max(64, width // 8 * 8)
        rows = min(_log(rng, 1, 16384), (1 << 26) // width)
        case = _norm("", rng.choice(["rms", "layer"]), rows, width, dtype, rng.random() < 0.5)
        del case["name"]
        return case
    dtype = rng.choice(["bf16", "bf16", "bf16", "f16"])
    heads_q, heads_kv = rng.choice(_HEADS)
    dim = rng.choice([64, 64, 64, 128, 128, 128, 80, 96, 40, 256])
    if what == "decode":
        kind = rng.choice(["dense", "lengths"])
        case = _attn("", kind=kind, batch=_log(rng, 1, 64), heads_q=heads_q, heads_kv=heads_kv, seq_q=1,
                     seq_k=_log(rng, 16, 8192), dim=rng.choice([64, 128]),
                     mask=rng.choice(["none", "pad"]) if kind == "dense" else "none", dtype=dtype)
        limit = 64 * 2 * 8192 * 128
        while case["batch"] > 1 and case["batch"] * heads_kv * case["seq_k"] * case["dim"] > limit:
            case["batch"] //= 2
        while case["batch"] * heads_kv * case["seq_k"] * case["dim"] > limit:
            case["seq_k"] //= 2
    elif what == "varlen":
        longest = _log(rng, 16, 2048)
        case = _attn("", kind="varlen", batch=rng.randint(1, 16), heads_q=heads_q, heads_kv=heads_kv, seq_q=longest,
                     seq_k=longest, seq_min=max(1, longest // rng.choice([1, 4, 16])), dim=dim,
                     causal=rng.random() < 0.7, dtype=dtype, train=rng.random() < 0.5)
    elif what == "cross":
        case = _attn("", batch=rng.randint(1, 4), heads_q=heads_q, heads_kv=heads_kv, seq_q=_log(rng, 64, 4096),
                     seq_k=_log(rng, 1, 512), dim=dim, layout=rng.choice(["heads", "rows"]), dtype=dtype,
                     train=rng.random() < 0.3)
    else:
        seq = _log(rng, 32, 4396)
        case = _attn("", batch=_log(rng, 1, 32), heads_q=heads_q, heads_kv=heads_kv, seq_q=seq, seq_k=seq, dim=dim,
                     layout=rng.choice(["heads", "rows"]), dtype=dtype, train=what == "train")
        option = rng.choice(["causal", "causal", "plain", "plain", "pad", "additive"])
        case["causal"] = option == "causal"
        case["mask"] = option if option in ("pad", "additive") else "none"
    while case["batch"] > 1 and work(case)["flops"] > _MOST_FLOPS:
        case["batch"] = max(1, case["batch"] // 2)
    while work(case)["flops"] > _MOST_FLOPS:
        case["seq_q"] = case["seq_k"] = int(case["seq_k"] * 0.75)
        case["seq_min"] = min(case["seq_min"], case["seq_q"])
    del case["name"]
    return case


# ---------------------------------------------------------------- inputs


def _varlen_lengths(case):
    """Sequence lengths of a packed case: spread evenly over [seq_min, seq_q], the longest
    among them, in a scrambled order (the same for every seed: they are the case's size)."""
    n, lo, hi = case["batch"], case["seq_min"], case["seq_q"]
    spread = [hi - (hi - lo) * i // max(1, n - 1) for i in range(n)]
    order = sorted(range(n), key=lambda i: (i * 5 + 3) % 17 + i / 64.0)
    return [spread[i] for i in order]


def _inputs(case, seed):
    """The case's tensors, from the seed alone: N(0, 1) activations, weights near 1."""
    gen = torch.Generator(device="cuda").manual_seed(int(seed))
    dt = _DTYPES[case["dtype"]]

    def randn(*shape):
        return torch.randn(*shape, generator=gen, device="cuda", dtype=torch.float32).to(dt)

    t = {}
    if case["op"] == "norm":
        t["x"] = randn(case["rows"], case["width"])
        t["weight"] = (1 + 0.02 * randn(case["width"]).float()).to(dt)
        if case["kind"] == "layer":
            t["bias"] = (0.02 * randn(case["width"]).float()).to(dt)
        if case["train"]:
            t["grad"] = randn(case["rows"], case["width"])
        return t
    b, hq, hk, d = case["batch"], case["heads_q"], case["heads_kv"], case["dim"]
    if case["kind"] == "varlen":
        cu = [0]
        for n in _varlen_lengths(case):
            cu.append(cu[-1] + n)
        t["q"], t["k"], t["v"] = randn(cu[-1], hq, d), randn(cu[-1], hk, d), randn(cu[-1], hk, d)
        t["cu"] = torch.tensor(cu, dtype=torch.int32, device="cuda")
        t["grad"] = randn(cu[-1], hq, d) if case["train"] else None
        return t

    def heads(h, s):
        if case["layout"] == "rows":
            return randn(b, s, h * d).view(b, s, h, d).transpose(1, 2)
        return randn(b, h, s, d)

    t["q"], t["k"], t["v"] = heads(hq, case["seq_q"]), heads(hk, case["seq_k"]), heads(hk, case["seq_k"])
    t["grad"] = heads(hq, case["seq_q"]) if case["train"] else None
    t["mask"] = t["lengths"] = None
    if case["mask"] == "pad" or case["kind"] == "lengths":
        sk = case["seq_k"]
        low = max(1, sk // 50) if case["kind"] == "dense" else max(1, sk // 2)
        # Lengths spread over the range (so that every seed costs the same), in a random order.
        lengths = torch.linspace(low, sk, b, device="cuda").round().to(torch.int32)
        lengths = lengths[torch.randperm(b, generator=gen, device="cuda")]
        if case["kind"] == "lengths":
            t["lengths"] = lengths.contiguous()
        else:
            t["mask"] = (torch.arange(sk, device="cuda")[None, :] < lengths[:, None]).view(b, 1, 1, sk)
    elif case["mask"] == "additive":
        sq, sk = case["seq_q"], case["seq_k"]
        keep = torch.rand(1, 1, sq, sk, generator=gen, device="cuda") >= 0.1
        keep &= torch.ones(sq, sk, dtype=torch.bool, device="cuda").tril(max(0, sk - sq))
        keep[..., 0] = True
        t["mask"] = torch.zeros(1, 1, sq, sk, device="cuda", dtype=dt).masked_fill(~keep, float("-inf"))
    return t


def prepare(case, seed):
    t = _inputs(case, seed)
    if case["train"]:
        for name in ("q", "k", "v", "x", "weight", "bias"):
            if t.get(name) is not None:
                t[name] = t[name].requires_grad_()
    t["case"] = case
    return t


# ---------------------------------------------------------------- one call


def run(state):
    case = state["case"]
    if case["op"] == "norm":
        x, w = state["x"], state["weight"]
        if case["kind"] == "layer":
            y, params = F.layer_norm(x, [case["width"]], w, state["bias"], 1e-5), (x, w, state["bias"])
        else:
            y, params = F.rms_norm(x, [case["width"]], w, 1e-6), (x, w)
        return (y, *torch.autograd.grad(y, params, state["grad"])) if case["train"] else y
    q, k, v = state["q"], state["k"], state["v"]
    if case["kind"] == "varlen":
        out = kohakutt_amd.sdpa_varlen(q, k, v, state["cu"], max_q=case["seq_q"], max_k=case["seq_k"],
                                       is_causal=case["causal"])
    elif case["kind"] == "lengths":
        out = kohakutt_amd.sdpa(q, k, v, key_lengths=state["lengths"])
    else:
        out = F.scaled_dot_product_attention(q, k, v, attn_mask=state["mask"], is_causal=case["causal"],
                                             enable_gqa=case["heads_q"] != case["heads_kv"])
    return (out, *torch.autograd.grad(out, (q, k, v), state["grad"])) if case["train"] else out


# ---------------------------------------------------------------- the same in float64


def _exact_norm(case, t):
    x, w = t["x"].double(), t["weight"].double()
    layer = case["kind"] == "layer"
    mean = x.mean(-1, keepdim=True) if layer else 0.0
    rstd = ((x - mean).square().mean(-1, keepdim=True) + (1e-5 if layer else 1e-6)).rsqrt()
    xhat = (x - mean) * rstd
    y = xhat * w + (t["bias"].double() if layer else 0.0)
    if not case["train"]:
        return y
    dy = t["grad"].double()
    g = dy * w
    dx = rstd * (g - (g.mean(-1, keepdim=True) if layer else 0.0) - xhat * (g * xhat).mean(-1, keepdim=True))
    return (y, dx, (dy * xhat).sum(0), dy.sum(0)) if layer else (y, dx, (dy * xhat).sum(0))


def _exact_head(q, k, v, keep, bias, scale, do):
    """One head: out [Sq, D] and, with do, (dq, dk, dv), from 2-D float64 operands."""
    s = (q @ k.t().contiguous()) * scale
    if bias is not None:
        s += bias
    if keep is not None:
        s.masked_fill_(~keep, float("-inf"))
    p = torch.softmax(s, -1)
    del s
    out = p @ v
    if do is None:
        return out, None
    dv = p.t().contiguous() @ do
    dp = do @ v.t().contiguous()
    ds = p * (dp - (dp * p).sum(-1, keepdim=True))
    return out, (ds @ k * scale, ds.t().contiguous() @ q * scale, dv)


def exact(case, seed):
    t = _inputs(case, seed)
    if case["op"] == "norm":
        return _exact_norm(case, t)
    # A part is a batch entry of [B, H, S, D] or a packed sequence's tokens of [T, H, D]: either
    # way x[part, head] is one head's [S, D].
    varlen = case["kind"] == "varlen"
    if varlen:
        cu = t["cu"].tolist()
        parts = [slice(a, b) for a, b in zip(cu[:-1], cu[1:])]
    else:
        parts = range(case["batch"])
    scale = 1.0 / math.sqrt(case["dim"])
    group = case["heads_q"] // case["heads_kv"]
    out = torch.zeros(t["q"].shape, dtype=torch.float64, device="cuda")
    grads = [torch.zeros(t[n].shape, dtype=torch.float64, device="cuda") for n in ("q", "k", "v")] if case["train"] else None
    for part in parts:
        keep = bias = None
        sq, sk = t["q"][part, 0].size(0), t["k"][part, 0].size(0)
        if not varlen and t["lengths"] is not None:
            sk = int(t["lengths"][part])
        if not varlen and t["mask"] is not None:
            m = t["mask"][min(part, t["mask"].size(0) - 1), 0]
            keep, bias = (m, None) if m.dtype == torch.bool else (None, m.double())
        if case["causal"]:
            keep = torch.ones(sq, sk, dtype=torch.bool, device="cuda").tril()
        for h in range(case["heads_q"]):
            q = t["q"][part, h].double()
            k, v = t["k"][part, h // group][:sk].double(), t["v"][part, h // group][:sk].double()
            do = t["grad"][part, h].double() if case["train"] else None
            o, g = _exact_head(q, k, v, keep, bias, scale, do)
            out[part, h] = o
            if g is not None:
                grads[0][part, h] = g[0]
                grads[1][part, h // group][:sk] += g[1]
                grads[2][part, h // group][:sk] += g[2]
    return (out, *grads) if case["train"] else out


# ---------------------------------------------------------------- work and tolerance


def work(case):
    size = {"bf16": 2, "f16": 2, "f32": 4}[case["dtype"]]
    if case["op"] == "norm":
        n, w = case["rows"] * case["width"], case["width"]
        params = 2 if case["kind"] == "layer" else 1
        # Training also reads dy, writes dx and the parameter gradients.
        return {"bytes": float(((4 if case["train"] else 2) * n + (2 if case["train"] else 1) * params * w) * size),
                "flops": float((16 if case["train"] else 6) * n)}
    hq, hk, d = case["heads_q"], case["heads_kv"], case["dim"]
    mask_bytes = 0
    if case["kind"] == "varlen":
        lens = _varlen_lengths(case)
        nq = nk = sum(lens)
        pairs = sum(n * (n + 1) // 2 if case["causal"] else n * n for n in lens)
    else:
        b, sq, sk = case["batch"], case["seq_q"], case["seq_k"]
        nq, nk = b * sq, b * sk
        pairs = b * (sq * (sq + 1) // 2 if case["causal"] else sq * sk)
        if case["mask"] == "pad" or case["kind"] == "lengths":
            low = max(1, sk // 50) if case["kind"] == "dense" else max(1, sk // 2)
            nk = sum(round(low + (sk - low) * i / max(1, b - 1)) for i in range(b))
            pairs = nk * sq
            mask_bytes = b * sk if case["mask"] == "pad" else 4 * b
        elif case["mask"] == "additive":
            pairs = b * sum(min(sk, i + 1 + max(0, sk - sq)) for i in range(sq))
            mask_bytes = sq * sk * size
    q_bytes, kv_bytes = nq * hq * d * size, 2 * nk * hk * d * size
    if case["train"]:  # and dO read; dQ, dK and dV written
        q_bytes, kv_bytes = 2 * q_bytes, 2 * kv_bytes
    return {"bytes": float(2 * q_bytes + kv_bytes + mask_bytes), "flops": (3.5 if case["train"] else 1.0) * 4.0 * d * hq * pairs}


def tolerance(case):
    # Attention rounds P (and dS) to 16 bits for the second product and the result once
    # more; a norm rounds its result once (parameter gradients are 32-bit sums first).
    # About four times what the outputs are off float64.
    if case["op"] == "norm":
        return {"bf16": {"rel": 7e-3, "max": 3e-2}, "f16": {"rel": 1e-3, "max": 4e-3}, "f32": {"rel": 2e-6, "max": 5e-5}}[
            case["dtype"]
        ]
    rel = 1e-2 if case["dtype"] == "bf16" else 1.3e-3
    return {"rel": rel, "max": 12 * rel}
