"""Prefill forwards against float64 around the plan's line for the 32x32x16 tile kernel
(attn_tile_kernel): row and key counts one off its 32-row groups, 64- and 128-row workgroups
and 32- to 128-key tiles, GQA, causal, masks (rows that keep no key among them), key lengths,
packed ragged batches, a value head dim of its own, and scales of any sign.  CASES and the
packed batch lie on both sides of the line; ROUTED and the longer packed batch name the form
that takes them (the plan is asked) and cover each padded head dim, both workgroup sizes, both
types, each mask type and packed masks."""

from __future__ import annotations

import math

import pytest
import torch
import torch.nn.functional as F

from kohakutt_amd import capi

pytestmark = pytest.mark.gpu


def _attend(q, k, v, bias, scale):
    """float64 attention and its lse; a row whose every key is masked is over its raw scores
    and its lse carries the -5e5 offset (bias: -inf where masked)."""
    s = q.double() @ k.double().transpose(-1, -2).contiguous() * scale
    if bias is not None:
        b = bias.double()
        dead = (b == -math.inf).all(-1, keepdim=True)
        s = s + torch.where(dead, torch.zeros_like(b), b)
    p = torch.softmax(s, -1)
    lse = torch.logsumexp(s, -1)
    if bias is not None:
        lse = lse - 5e5 * dead.squeeze(-1)
    return p @ v.double(), p @ v.double().abs(), lse


HALF_ULP = {torch.bfloat16: 2.0**-8, torch.float16: 2.0**-11}


def _close(got, want, weight, dtype):
    # P rounds to the operand type (half an ulp of each weight), its row sum is of the rounded
    # weights (the same again at most), and the result rounds once: three half ulps of sum(P |v|).
    err = (got.double() - want).abs()
    bound = 3 * HALF_ULP[dtype] * weight + 1e-6
    assert torch.isfinite(got).all() and (err <= bound).all(), (err / bound).max().item()


CASES = [
    # b, hq, hk, sq, sk, d, causal, mask, dtype
    (16, 16, 16, 129, 131, 128, False, None, torch.bfloat16),
    (16, 28, 4, 65, 65, 128, True, None, torch.bfloat16),
    (4, 24, 24, 127, 257, 96, False, None, torch.float16),
    (2, 12, 2, 700, 700, 128, True, None, torch.float16),
    (8, 16, 16, 513, 300, 64, False, None, torch.bfloat16),
    (8, 12, 12, 300, 297, 40, False, None, torch.float16),
    (8, 16, 16, 1030, 1030, 64, True, None, torch.bfloat16),
    (4, 12, 12, 330, 330, 32, True, None, torch.bfloat16),
    (3, 8, 8, 350, 333, 256, False, None, torch.bfloat16),
    (2, 12, 6, 600, 600, 160, True, None, torch.bfloat16),
    (4, 16, 16, 255, 259, 64, False, "add", torch.bfloat16),
    (8, 16, 16, 300, 300, 64, False, "add", torch.float16),
    (6, 8, 8, 400, 401, 128, False, "add", torch.bfloat16),
    (6, 8, 4, 300, 129, 128, False, "f32", torch.bfloat16),
    (3, 8, 8, 450, 449, 128, False, "bool", torch.bfloat16),
    (6, 12, 12, 256, 256, 64, False, "pad", torch.bfloat16),
    (12, 12, 12, 385, 384, 80, False, "pad", torch.float16),
    (4, 8, 2, 200, 320, 256, False, "pad", torch.bfloat16),
]


def _kernel(q, k, v, mask=None, causal=False, cu=None, longest=0):
    """The kernel the plan gives a call: dense [B, H, S, D], or packed [T, H, D] with host
    offsets (mask then flat and block-packed)."""
    a = capi.AttnArgs()
    a.q, a.k, a.v, a.out = q.data_ptr(), k.data_ptr(), v.data_ptr(), q.data_ptr()
    a.dtype = {torch.bfloat16: capi.KMI_BF16, torch.float16: capi.KMI_F16}[q.dtype]
    a.causal = int(causal)
    a.head_dim, a.head_dim_v, a.scale = q.size(-1), v.size(-1), 1.0
    axes = (0, 1, 2)
    if cu is None:
        a.batch, a.heads_q, a.seq_q = q.shape[:3]
        a.heads_kv, a.seq_k = k.shape[1:3]
    else:
        a.batch, a.heads_q, a.heads_kv, a.seq_q, a.seq_k = len(cu) - 1, q.size(1), k.size(1), longest, longest
        a.cu_seqlens_q = a.cu_seqlens_k = q.data_ptr()
        a.total_q = a.total_k = q.size(0)
        axes = (0, 1, 0)
    for field, t in (("q_stride", q), ("k_stride", k), ("v_stride", v)):
        getattr(a, field)[:] = [t.stride(i) for i in axes]
    a.o_stride[:] = [8 * math.ceil(s / 8) for s in a.q_stride]
    if mask is not None:
        a.mask = mask.data_ptr()
        a.mask_dtype = {torch.bool: capi.KMI_BOOL, torch.bfloat16: capi.KMI_BF16, torch.float16: capi.KMI_F16,
                        torch.float32: capi.KMI_F32}[mask.dtype]  # fmt: skip
        if cu is None:
            a.mask_mode = capi.KMI_MASK_STRIDED
            m = mask.expand(q.size(0), q.size(1), q.size(2), k.size(2))
            a.mask_stride[:] = list(m.stride())
        else:
            a.mask_mode, a.mask_numel = capi.KMI_MASK_PACKED, mask.numel()
    return capi.attn_fwd_kernel(a)


BF, HF = torch.bfloat16, torch.float16
ROUTED = [
    # as CASES, and the kernel
    (8, 16, 16, 300, 297, 32, False, None, BF, "tile64"),
    (10, 16, 16, 300, 300, 32, True, None, HF, "tile128"),
    (8, 16, 16, 300, 290, 64, False, None, HF, "tile64"),
    (10, 16, 16, 300, 261, 64, False, None, BF, "tile128"),
    (4, 24, 24, 129, 257, 96, False, None, HF, "tile64"),
    (4, 24, 24, 300, 257, 96, False, None, BF, "tile128"),
    (6, 24, 24, 300, 300, 96, True, None, BF, "tile64"),
    (7, 24, 24, 300, 300, 96, True, None, HF, "tile128"),
    (4, 24, 12, 300, 200, 128, False, None, HF, "tile64"),
    (8, 24, 12, 300, 300, 128, True, None, HF, "tile128"),
    (4, 16, 16, 300, 300, 32, False, "bool", HF, "tile64"),
    (8, 16, 16, 400, 300, 32, False, "add", BF, "tile128"),
    (8, 16, 16, 400, 333, 40, False, "f32", HF, "tile128"),
    (8, 16, 16, 400, 333, 64, False, "add", BF, "tile128"),
    (8, 16, 16, 400, 333, 64, False, "bool", BF, "tile128"),
    (8, 12, 12, 400, 384, 64, False, "pad", HF, "tile128"),
    (6, 8, 8, 400, 401, 96, False, "add", HF, "tile64"),
    (8, 12, 12, 400, 384, 96, False, "pad", BF, "tile128"),
    (8, 12, 12, 400, 384, 128, False, "pad", BF, "tile128"),
    (6, 8, 8, 200, 320, 192, False, "bool", BF, "tile64"),
    (6, 8, 8, 300, 320, 256, False, "pad", BF, "tile64"),
    (6, 8, 8, 300, 319, 256, False, "add", HF, "tile64"),
    # wavefronts whose rows all lie past the end, in both forms
    (64, 12, 12, 65, 300, 64, False, None, BF, "tile128"),
    (128, 28, 4, 4, 300, 64, False, None, BF, "tile64"),
    (128, 28, 4, 4, 300, 128, False, None, HF, "tile64"),
    (128, 28, 4, 4, 300, 128, True, None, BF, "tile128"),
    (32, 16, 16, 20, 512, 64, False, "pad", BF, "tile64"),
    (64, 12, 12, 70, 80, 128, False, "pad", BF, "tile128"),
    (32, 16, 16, 31, 300, 64, False, "add", BF, "tile64"),
    (32, 16, 16, 31, 300, 256, False, "f32", BF, "tile64"),
]  # fmt: skip

# Masked calls whose last key tile is partial: fewer than four keys, and every remainder of four.
PARTIAL = [(6, 16, 16, 128, sk, d, False, kind, BF, "tile64")
           for sk in (3, 4, 5, 31, 66, 127, 129, 190) for d in (64, 128) for kind in ("bool", "add", "f32", "pad")]  # fmt: skip
PARTIAL += [(28, 16, 16, 70, sk, 64, False, kind, HF, "tile128") for sk in (5, 66, 191) for kind in ("bool", "add", "f32", "pad")]


@pytest.mark.parametrize("case", CASES + ROUTED + PARTIAL, ids=lambda c: "x".join(map(str, c)))
def test_dense_calls_meet_float64(native, dev, case):
    b, hq, hk, sq, sk, d, causal, mask, dtype = case[:9]
    print(f"tile {case}", flush=True)
    g = torch.Generator(device=dev).manual_seed(sum(case[:6]))
    randn = lambda *s: torch.randn(*s, generator=g, device=dev).to(dtype)  # noqa: E731
    q, k, v = randn(b, hq, sq, d), randn(b, hk, sk, d), randn(b, hk, sk, d)
    m = bias = None
    if mask in ("add", "f32"):
        m = randn(1, 1, sq, sk) if mask == "add" else randn(b, 1, sq, sk).float()
        m = m.masked_fill(torch.rand(m.shape, generator=g, device=dev) < 0.3, -math.inf)
        m[:, :, sq // 3] = -math.inf  # a row that keeps no key
        m[:, :, : sq // 2, sk // 2 :] = -math.inf  # whole tiles masked for some rows
        bias = m
    elif mask == "bool":
        m = torch.rand(b, hq, sq, sk, generator=g, device=dev) < 0.5
        m[:, 1, 7] = False
    elif mask == "pad":
        lens = torch.randint(1, sk + 1, (b,), generator=g, device=dev)
        lens[0] = sk
        m = (torch.arange(sk, device=dev)[None] < lens[:, None]).view(b, 1, 1, sk)
        m[1] = False  # no key at all: raw scores
    if m is not None and m.dtype == torch.bool:
        bias = torch.zeros(m.shape, device=dev).masked_fill(~m, -math.inf)
    if len(case) > 9:
        assert _kernel(q, k, v, m, causal) == case[9]
    if causal:
        bias = torch.zeros(sq, sk, device=dev).masked_fill(~torch.ones(sq, sk, dtype=torch.bool, device=dev).tril(), -math.inf)
    native.reset_counters()
    out, lse = torch.ops.aten._scaled_dot_product_fused_attention_overrideable(q, k, v, m, 0.0, causal)[:2]
    torch.cuda.synchronize()
    assert native.counters()["attention"] == 1
    kr, vr = k.repeat_interleave(hq // hk, 1), v.repeat_interleave(hq // hk, 1)
    for i in range(b):
        bi = None if bias is None else (bias if bias.dim() == 2 else bias[min(i, bias.size(0) - 1)])
        want, weight, want_lse = _attend(q[i], kr[i], vr[i], bi, 1 / math.sqrt(d))
        _close(out[i], want, weight, dtype)
        # The row sum is of the rounded weights: half an ulp; fp32 for the rest.
        off = ((lse[i].double() - want_lse).abs() - 2e-6 * want_lse.abs()).max().item()
        assert off <= HALF_ULP[dtype] + 1e-4, off


@pytest.mark.parametrize("scale", [-0.3, 0.0])
@pytest.mark.parametrize("mask", [False, True])
def test_scale_of_any_sign(native, dev, scale, mask):
    print(f"scale {scale} mask {mask}", flush=True)
    g = torch.Generator(device=dev).manual_seed(11)
    q, k, v = (torch.randn(8, 16, 260, 128, generator=g, device=dev).bfloat16() for _ in range(3))
    m = torch.randn(1, 1, 260, 260, generator=g, device=dev).bfloat16() if mask else None
    out = F.scaled_dot_product_attention(q, k, v, attn_mask=m, scale=scale)
    for i in (0, 7):
        want, weight, _ = _attend(q[i], k[i], v[i], None if m is None else m[0], scale)
        _close(out[i], want, weight, torch.bfloat16)


@pytest.mark.parametrize("d,dv", [(64, 64), (128, 128), (128, 64), (96, 256)])
@pytest.mark.parametrize("causal", [False, True])
def test_packed_ragged_batches_meet_float64(native, dev, d, dv, causal):
    print(f"packed {d} {dv} {causal}", flush=True)
    lens = [700, 1, 129, 64, 333, 520, 65, 31, 250, 400, 128, 610]
    cu = [0]
    for n in lens:
        cu.append(cu[-1] + n)
    g = torch.Generator(device=dev).manual_seed(d + dv)
    randn = lambda *s: torch.randn(*s, generator=g, device=dev).bfloat16()  # noqa: E731
    q, k, v = randn(cu[-1], 24, d), randn(cu[-1], 12, d), randn(cu[-1], 12, dv)
    out = native.sdpa_varlen(q, k, v, torch.tensor(cu, dtype=torch.int32, device=dev), max_q=max(lens), max_k=max(lens),
                             is_causal=causal)
    for a, b in zip(cu[:-1], cu[1:]):
        qs, ks, vs = (t[a:b].transpose(0, 1) for t in (q, k.repeat_interleave(2, 1), v.repeat_interleave(2, 1)))
        bias = None
        if causal:
            bias = torch.zeros(b - a, b - a, device=dev)
            bias = bias.masked_fill(~torch.ones(b - a, b - a, dtype=torch.bool, device=dev).tril(), -math.inf)
        want, weight, _ = _attend(qs, ks, vs, bias, 1 / math.sqrt(d))
        _close(out[a:b].transpose(0, 1), want, weight, torch.bfloat16)


@pytest.mark.parametrize("d,masked,kernel", [(64, False, "tile128"), (32, True, "tile128"), (64, True, "tile128"),
                                             (96, False, "tile128"), (128, True, "tile64")])  # fmt: skip
@pytest.mark.parametrize("causal", [False, True])
def test_longer_packed_batches_meet_float64(native, dev, d, masked, kernel, causal):
    """The batch of the test above and one more sequence, with a block-packed mask too (a row
    that keeps no key in each sequence of more than one)."""
    lens = [700, 1, 129, 64, 333, 520, 65, 31, 250, 400, 128, 610, 699]
    cu = [0]
    for n in lens:
        cu.append(cu[-1] + n)
    g = torch.Generator(device=dev).manual_seed(d + causal)
    randn = lambda *s: torch.randn(*s, generator=g, device=dev).bfloat16()  # noqa: E731
    q, k, v = randn(cu[-1], 24, d), randn(cu[-1], 12, d), randn(cu[-1], 12, d)
    blocks = []
    for n in lens:
        m = torch.randn(n, n, generator=g, device=dev).masked_fill(
            torch.rand(n, n, generator=g, device=dev) < 0.3, -math.inf)
        if n > 1:
            m[n // 2] = -math.inf
        blocks.append(m)
    packed = torch.cat([m.flatten() for m in blocks]).bfloat16() if masked else None
    assert _kernel(q, k, v, packed, causal, cu, max(lens)) == kernel
    out = native.sdpa_varlen(q, k, v, cu, is_causal=causal, packed_mask=packed)
    for a, b, m in zip(cu[:-1], cu[1:], blocks):
        n = b - a
        qs, ks, vs = (t[a:b].transpose(0, 1) for t in (q, k.repeat_interleave(2, 1), v.repeat_interleave(2, 1)))
        seen = torch.ones(n, n, dtype=torch.bool, device=dev)
        seen = seen.tril() if causal else seen
        bias = m.bfloat16().double() if masked else torch.zeros(n, n, device=dev, dtype=torch.float64)
        kept = ((bias > -math.inf) & seen).any(-1, keepdim=True)
        # (A row whose seen keys are all masked is over their raw scores.)
        bias = torch.where(kept, bias, torch.zeros_like(bias)).masked_fill(~seen, -math.inf)
        want, weight, _ = _attend(qs, ks, vs, bias, 1 / math.sqrt(d))
        _close(out[a:b].transpose(0, 1), want, weight, torch.bfloat16)


def test_key_lengths_meet_float64(native, dev):
    g = torch.Generator(device=dev).manual_seed(5)
    q, k, v = (torch.randn(8, 16, 300, 128, generator=g, device=dev).bfloat16() for _ in range(3))
    lens = torch.tensor([1, 31, 32, 64, 65, 200, 299, 300], dtype=torch.int32, device=dev)
    out = native.sdpa(q, k, v, key_lengths=lens)
    for i, n in enumerate(lens.tolist()):
        want, weight, _ = _attend(q[i], k[i, :, :n], v[i, :, :n], None, 1 / math.sqrt(128))
        _close(out[i], want, weight, torch.bfloat16)


@pytest.mark.parametrize("case", [
    # b, h, s, d, kind, dtype: the tile kernel (64 and 128 rows) and the smaller calls' kernel
    (2, 16, 400, 64, "add", torch.bfloat16),
    (8, 16, 400, 64, "add", torch.float16),
    (6, 8, 401, 128, "bool", torch.bfloat16),
    (8, 16, 300, 128, "pad", torch.bfloat16),
    (4, 8, 200, 256, "pad", torch.bfloat16),
    (1, 2, 100, 64, "add", torch.bfloat16),
    (1, 2, 100, 128, "pad", torch.bfloat16),
], ids=lambda c: "x".join(map(str, c)))  # fmt: skip
def test_masked_keys_may_hold_anything(native, dev, case):
    """A masked key has weight 0 whatever its K row holds: NaN, infinities, or values whose
    product overflows.  The result is that of the same call with zeros there, bit for bit."""
    b, h, s, d, kind, dtype = case
    print(f"masked rows {case}", flush=True)
    g = torch.Generator(device=dev).manual_seed(s + d)
    q, k, v = (torch.randn(b, h, s, d, generator=g, device=dev).to(dtype) for _ in range(3))
    hidden = torch.rand(s, generator=g, device=dev) < 0.4
    hidden[::32] = False  # each tile keeps a key
    if kind == "pad":
        m = (~hidden).view(1, 1, 1, s).expand(b, 1, 1, s)
    else:
        m = (torch.rand(1, 1, s, s, generator=g, device=dev) >= 0.2) & ~hidden
        m[..., 0] = True
        m[..., ::32] = True
        if kind == "add":
            m = torch.randn(1, 1, s, s, generator=g, device=dev).to(dtype).masked_fill(~m, -math.inf)
    clean = k.masked_fill(hidden[None, None, :, None], 0.0)
    spoilt = clean.clone()
    at = torch.nonzero(hidden).flatten()
    for i, value in enumerate((math.nan, math.inf, -math.inf, torch.finfo(dtype).max)):
        spoilt[:, :, at[i::4]] = value
    attend = torch.ops.aten._scaled_dot_product_fused_attention_overrideable
    out, lse = attend(q, spoilt, v, m, 0.0, False)[:2]
    want, want_lse = attend(q, clean, v, m, 0.0, False)[:2]
    assert torch.isfinite(want).all()
    assert torch.equal(out, want) and torch.equal(lse, want_lse)


@pytest.mark.parametrize("d", [64, 128])
def test_additive_mask_rounds_once(native, dev, d):
    """A logit of -1e5 over whole rows (kept: above -5e5) leaves the weights as they are but
    for the rounding of score + logit.  In base 2 that sum lies within 2^17 .. 2^18, so one
    rounding is off by 2^-6 / sqrt(12) in the mean, and a weight by ln 2 of it; f16 rounds the
    weights and the result by 2^-11 / sqrt(3) each."""
    b, h, s = 4, 8, 384
    g = torch.Generator(device=dev).manual_seed(d)
    q, k, v = (torch.randn(b, h, s, d, generator=g, device=dev).half() for _ in range(3))
    m = torch.full((1, 1, s, s), -1e5, device=dev)
    out = F.scaled_dot_product_attention(q, k, v, attn_mask=m)
    want = off = 0.0
    for i in range(b):
        ref, _, _ = _attend(q[i], k[i], v[i], None, 1 / math.sqrt(d))
        off += (out[i].double() - ref).square().sum().item()
        want += ref.square().sum().item()
    got = math.sqrt(off / want)
    once = math.hypot(2.0**-6 / math.sqrt(12) * math.log(2), 2.0**-11 / math.sqrt(3) * math.sqrt(2))
    print(f"d {d}: {got:.2e}, one rounding {once:.2e}", flush=True)
    assert got <= 1.15 * once  # (one rounding: 15% for what is left of a small sample)


@pytest.mark.parametrize("b,h,s,d,kind,kernel", [
    (8, 16, 1000, 128, "causal", "tile128"),
    (7, 12, 1000, 96, "causal", "tile128"),
    (8, 8, 1000, 128, "plain", "tile128"),
    (8, 8, 1000, 64, "add", "tile128"),
    (4, 8, 1000, 128, "add", "tile64"),
])  # fmt: skip
def test_as_close_to_float64_as_the_general_kernel(native, dev, b, h, s, d, kind, kernel):
    """The same rows through the tile kernel and, one batch entry at a time, through
    attn_fwd_kernel: the tile kernel's result is no further from float64 (half a percent for
    the roundings' chance)."""
    print(f"as close {b}x{h}x{s}x{d} {kind}", flush=True)
    g = torch.Generator(device=dev).manual_seed(s + d)
    q, k, v = (torch.randn(b, h, s, d, generator=g, device=dev).bfloat16() for _ in range(3))
    m = bias = None
    seen = torch.ones(s, s, dtype=torch.bool, device=dev)
    if kind == "add":
        keep = (torch.rand(1, 1, s, s, generator=g, device=dev) >= 0.1) & seen.tril()
        keep[..., 0] = True
        m = torch.zeros(1, 1, s, s, device=dev).masked_fill(~keep, -math.inf).bfloat16()
        bias = m[0, 0]
    elif kind == "causal":
        bias = torch.zeros(s, s, device=dev).masked_fill(~seen.tril(), -math.inf)
    attend = torch.ops.aten._scaled_dot_product_fused_attention_overrideable
    causal = kind == "causal"
    assert _kernel(q, k, v, m, causal) == kernel and _kernel(q[:1], k[:1], v[:1], m, causal) == "general"
    out = attend(q, k, v, m, 0.0, causal)[0]
    off = general = 0.0
    for i in range(b):
        want, _, _ = _attend(q[i], k[i], v[i], bias, 1 / math.sqrt(d))
        one = attend(q[i : i + 1], k[i : i + 1], v[i : i + 1], m, 0.0, causal)[0][0]
        off += (out[i].double() - want).square().sum().item()
        general += (one.double() - want).square().sum().item()
    print(f"  tile {off**0.5:.4f} general {general**0.5:.4f} ratio {(off / general) ** 0.5:.4f}", flush=True)
    assert off <= 1.005**2 * general
