"""GPU parity of the flash backward (``kmi_attn_bwd`` behind the overrideable SDPA
backward, the packed ops and key lengths): dq, dk, dv (causal top-left or not, GQA,
Sq != Sk, ragged lengths, bool and additive masks with fully-masked rows, packed
sequences with key masks and per-row masks, bf16 / fp16) against float64 autograd of the
same attention on the CPU, with the BASELINE bar: median relative error at most 1.5x
torch's CPU autograd at the same dtype."""

from __future__ import annotations

import ctypes

import pytest
import torch
import torch.nn.functional as F

import attn_cases as C
import numpy as np
from kohakutt_amd import capi
from oracle import attention as oatt

pytestmark = pytest.mark.gpu

CASES = [
    # b, hq, hk, sq, sk, d, causal
    (2, 4, 4, 128, 128, 64, False),
    (1, 14, 2, 300, 300, 64, True),
    (2, 8, 2, 100, 260, 128, False),
    (1, 4, 1, 200, 120, 64, True),
    (2, 6, 3, 77, 77, 128, True),
    (1, 2, 2, 1, 45, 64, False),
    # Enough workgroups that dK/dV and dQ run unsplit (direct writes, no partials):
    (16, 8, 8, 256, 256, 64, False),
    (8, 16, 4, 256, 256, 128, True),
]


def _grads(q, k, v, go, causal, dtype, dev=None):
    """(out, dq, dk, dv) of SDPA at ``dtype`` on ``dev`` (CPU when None)."""
    hq, hk = q.size(1), k.size(1)
    ts = [t.to(dtype) for t in (q, k, v)]
    if dev is not None:
        ts = [t.to(dev) for t in ts]
    ts = [t.detach().requires_grad_() for t in ts]
    qq, kk, vv = ts
    if dev is None:
        kk_, vv_ = kk.repeat_interleave(hq // hk, 1), vv.repeat_interleave(hq // hk, 1)
        out = F.scaled_dot_product_attention(qq, kk_, vv_, is_causal=causal)
    else:
        out = F.scaled_dot_product_attention(qq, kk, vv, is_causal=causal, enable_gqa=hq != hk)
    g = go.to(dtype)
    out.backward(g.to(dev) if dev is not None else g)
    return [t.detach().cpu() for t in (out, qq.grad, kk.grad, vv.grad)]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(map(str, c)))
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_flash_backward_meets_the_float64_ruler(native, dev, case, dtype):
    b, hq, hk, sq, sk, d, causal = case
    print(f"backward case {case} {dtype}", flush=True)
    g = C.gen(900 + sum(case))
    q, k, v = C.randn(g, b, hq, sq, d, dtype=torch.float32), C.randn(g, b, hk, sk, d, dtype=torch.float32), C.randn(
        g, b, hk, sk, d, dtype=torch.float32)
    go = C.randn(g, b, hq, sq, d, dtype=torch.float32)
    # Inputs rounded to the test dtype first: every path sees the same values.
    q, k, v, go = (t.to(dtype).to(torch.float32) for t in (q, k, v, go))
    native.reset_counters()
    gpu = _grads(q, k, v, go, causal, dtype, dev)
    torch.cuda.synchronize()
    c = native.counters()
    assert c["attention"] == 1 and c["attention_backward"] == 1, c
    ref = _grads(q, k, v, go, causal, torch.float64)
    # Baseline at the same dtype: torch's CPU autograd in that dtype.
    cpu = _grads(q, k, v, go, causal, dtype)
    for name, gg, cc, rr in zip(("out", "dq", "dk", "dv"), gpu, cpu, ref):
        ok, sg, sc = C.ruler_ok(gg, cc, rr, factor=1.5)
        print(f"  {name}: gpu rel_median {sg['rel_median']:.2e}  cpu {sc['rel_median']:.2e}", flush=True)
        assert ok, (name, sg, sc)
        scale = rr.abs().max().item()
        assert (gg.double() - rr).abs().max().item() <= 3e-2 * max(scale, 1.0), (name, scale)


# The 32x32 tiles' edges: one row / key past or short of a 32-row block, a 64-row tile and a
# 128-key workgroup; head dims padded within a 16-byte-chunk row (40, 96); splits of dK / dV
# (few key tiles, many query blocks) and of dQ (one query row, many keys).
TILE_EDGES = [
    (1, 2, 1, 33, 31, 40, True),
    (1, 3, 1, 65, 129, 96, False),
    (2, 4, 2, 64, 63, 128, True),
    (1, 1, 1, 127, 127, 64, True),
    (1, 7, 1, 97, 97, 32, True),
    (1, 8, 2, 1100, 70, 128, False),
    (1, 6, 2, 700, 700, 64, True),
    (1, 1, 1, 3, 2100, 64, False),
]


@pytest.mark.parametrize("case", TILE_EDGES, ids=lambda c: "x".join(map(str, c)))
def test_tile_edges_meet_the_float64_ruler(native, dev, case):
    test_flash_backward_meets_the_float64_ruler(native, dev, case, torch.bfloat16)


@pytest.mark.parametrize("scale", [0.0, -0.2])
@pytest.mark.parametrize("d", [64, 128])
def test_backward_scale_of_any_sign(native, dev, scale, d):
    """Score accumulators start from mask logits over the scale: a zero and a negative scale
    with an additive mask, and a negative one with a causal call, against float64."""
    print(f"scale {scale} d {d}", flush=True)
    g = C.gen(970 + d)
    q, k, v, go = (C.randn(g, 1, 2, 70, d) for _ in range(4))
    mask = torch.randn(1, 1, 70, 70, generator=g).masked_fill(torch.rand(1, 1, 70, 70, generator=g) < 0.2, -torch.inf)
    mask[..., 0] = 0.0
    for m, causal in ((mask.bfloat16(), False), (None, True))[: 1 if scale == 0.0 else 2]:
        ts = [t.to(dev).requires_grad_() for t in (q, k, v)]
        out = F.scaled_dot_product_attention(
            *ts, attn_mask=None if m is None else m.to(dev), is_causal=causal, scale=scale
        )
        out.backward(go.to(dev))
        got = [t.grad.cpu().double() for t in ts]
        rs = [t.double().requires_grad_() for t in (q, k, v)]
        bias = torch.zeros(70, 70, dtype=torch.float64) if m is None else m.double()
        if causal:
            bias = bias.masked_fill(~torch.ones(70, 70, dtype=torch.bool).tril(), -torch.inf)
        (torch.softmax(rs[0] @ rs[1].transpose(-1, -2) * scale + bias, -1) @ rs[2]).backward(go.double())
        want = [t.grad for t in rs]
        for name, a, b in zip(("dq", "dk", "dv"), got, want):
            # P and dS round to bf16 (2^-9 each), then the sums once more: 2^-7 of the largest value.
            assert (a - b).abs().max().item() <= 2.0**-7 * max(b.abs().max().item(), 1e-6), (name, scale, causal)


def test_gqa_key_gradients_sum_their_query_heads(native, dev):
    """dk / dv of a K/V head equal the sum over its query heads of the per-head gradients
    (the same call with K/V repeated per query head, reduced afterwards)."""
    g = C.gen(950)
    b, hq, hk, s, d = 1, 6, 2, 96, 64
    q, k, v, go = (C.randn(g, *shape) for shape in ((b, hq, s, d), (b, hk, s, d), (b, hk, s, d), (b, hq, s, d)))
    qd, kd, vd = (t.to(dev).requires_grad_() for t in (q, k, v))
    F.scaled_dot_product_attention(qd, kd, vd, is_causal=True, enable_gqa=True).backward(go.to(dev))
    kr = k.repeat_interleave(3, 1).to(dev).requires_grad_()
    vr = v.repeat_interleave(3, 1).to(dev).requires_grad_()
    q2 = q.to(dev).requires_grad_()
    F.scaled_dot_product_attention(q2, kr, vr, is_causal=True).backward(go.to(dev))
    torch.cuda.synchronize()
    dk_sum = kr.grad.float().view(b, hk, 3, s, d).sum(2)
    dv_sum = vr.grad.float().view(b, hk, 3, s, d).sum(2)
    assert (kd.grad.float() - dk_sum).abs().max().item() < 3e-2
    assert (vd.grad.float() - dv_sum).abs().max().item() < 3e-2
    assert torch.equal(qd.grad, q2.grad)


def _masked_grads(q, k, v, go, mask, dtype, dev=None):
    """(out, dq, dk, dv) of masked SDPA at ``dtype``; on the CPU a fully-masked row follows
    the reference (softmax over its raw scores): its mask entries are lifted to 0."""
    hq, hk = q.size(1), k.size(1)
    ts = [t.to(dtype) for t in (q, k, v)]
    m = mask
    if dev is not None:
        ts = [t.to(dev) for t in ts]
        m = mask.to(dev)
    else:
        keep = mask if mask.dtype == torch.bool else mask > -5e5
        dead = ~keep.any(-1, keepdim=True)
        if mask.dtype == torch.bool:
            m = mask | dead
        else:
            m = mask.masked_fill(dead.expand_as(mask), 0.0)
    if m.is_floating_point():
        m = m.to(dtype)
    ts = [t.detach().requires_grad_() for t in ts]
    qq, kk, vv = ts
    if dev is None:
        out = F.scaled_dot_product_attention(qq, kk.repeat_interleave(hq // hk, 1), vv.repeat_interleave(hq // hk, 1),
                                             attn_mask=m)
    else:
        out = F.scaled_dot_product_attention(qq, kk, vv, attn_mask=m, enable_gqa=hq != hk)
    out.backward(go.to(dtype).to(dev) if dev is not None else go.to(dtype))
    return [t.detach().cpu() for t in (out, qq.grad, kk.grad, vv.grad)]


@pytest.mark.parametrize("kind", ["bool", "additive", "bool_key_padding"])
def test_masked_backward_on_the_kernels(native, dev, kind):
    """Masked calls take the backward kernels with the forward's mask rules, fully-masked
    rows included (the reference's softmax over raw scores)."""
    g = C.gen(951 + len(kind))
    b, hq, hk, sq, sk, d = 2, 4, 2, 70, 90, 64
    q, k, v, go = (C.randn(g, *sh, dtype=torch.float32) for sh in ((b, hq, sq, d), (b, hk, sk, d), (b, hk, sk, d),
                                                                    (b, hq, sq, d)))
    q, k, v, go = (t.bfloat16().float() for t in (q, k, v, go))
    if kind == "bool":
        mask = torch.rand(b, hq, sq, sk, generator=g) > 0.3
        mask[0, 1, 7] = False  # a fully-masked row
    elif kind == "additive":
        mask = torch.randn(b, 1, sq, sk, generator=g).masked_fill(torch.rand(b, 1, sq, sk, generator=g) < 0.2,
                                                                   float("-inf"))
        mask[1, 0, 3] = float("-inf")
    else:
        lens = torch.tensor([90, 17])
        mask = (torch.arange(sk)[None, :] < lens[:, None]).reshape(b, 1, 1, sk)
    native.reset_counters()
    gpu = _masked_grads(q, k, v, go, mask, torch.bfloat16, dev)
    torch.cuda.synchronize()
    c = native.counters()
    assert c["attention"] == 1 and c["attention_backward"] == 1, c
    ref = _masked_grads(q, k, v, go, mask.double() if mask.is_floating_point() else mask, torch.float64)
    cpu = _masked_grads(q, k, v, go, mask, torch.bfloat16)
    for name, gg, cc, rr in zip(("out", "dq", "dk", "dv"), gpu, cpu, ref):
        ok, sg, sc = C.ruler_ok(gg, cc, rr, factor=1.5)
        print(f"  {kind} {name}: gpu rel_median {sg['rel_median']:.2e}  cpu {sc['rel_median']:.2e}", flush=True)
        assert ok, (kind, name, sg, sc)


def test_mask_with_its_own_gradient_takes_the_recompute(native, dev):
    """A float mask that requires grad gets its gradient from the fp32 recompute."""
    g = C.gen(955)
    q, k, v = (C.randn(g, 1, 2, 32, 64) for _ in range(3))
    mask = torch.randn(1, 1, 32, 32, generator=g).to(dev).requires_grad_()
    native.reset_counters()
    out = F.scaled_dot_product_attention(q.to(dev), k.to(dev), v.to(dev), attn_mask=mask.bfloat16())
    out.float().sum().backward()
    torch.cuda.synchronize()
    assert mask.grad is not None and mask.grad.abs().sum().item() > 0
    assert native.counters()["attention_backward"] == 0


def _varlen_ref_grads(q, k, v, go, cu_q, cu_k, causal, key_mask=None):
    """Per-sequence float64 autograd of torch CPU SDPA (bottom-right causal as an explicit
    mask; a bool key mask keeps True keys); packed [T, H, D] gradients."""
    grads = [torch.zeros(t.shape, dtype=torch.float64) for t in (q, k, v)]
    hq, hk = q.size(1), k.size(1)
    for i in range(len(cu_q) - 1):
        a, b, c, d = cu_q[i], cu_q[i + 1], cu_k[i], cu_k[i + 1]
        lq, lk = b - a, d - c
        qs, ks, vs = (t.double().transpose(0, 1)[None].requires_grad_() for t in (q[a:b], k[c:d], v[c:d]))
        keep = torch.ones(lq, lk, dtype=torch.bool)
        if causal:
            keep &= torch.arange(lk)[None, :] <= torch.arange(lq)[:, None] + (lk - lq)
        if key_mask is not None:
            keep &= key_mask[c:d][None, :]
        out = F.scaled_dot_product_attention(qs, ks.repeat_interleave(hq // hk, 1), vs.repeat_interleave(hq // hk, 1),
                                             attn_mask=keep)
        out.backward(go[a:b].double().transpose(0, 1)[None])
        for gsum, t, (lo, hi) in zip(grads, (qs, ks, vs), ((a, b), (c, d), (c, d))):
            gsum[lo:hi] = t.grad[0].transpose(0, 1)
    return grads


@pytest.mark.parametrize("kind", ["causal_self", "cross_noncausal", "causal_fewer_queries", "key_mask"])
def test_varlen_backward_matches_float64_autograd(native, dev, kind):
    """Gradients through ``kohakutt_amd.sdpa_varlen``: every sequence in one set of
    backward kernel launches (bottom-right causal, key masks)."""
    g = C.gen(960 + len(kind))
    hq, hk, d = 8, 2, 64
    if kind == "causal_self":
        lq = [70, 1, 130, 33]
        lk = lq
    elif kind == "cross_noncausal":
        lq, lk = [40, 77, 5], [90, 12, 64]
    else:
        lq, lk = [20, 50, 3], [64, 50, 40]
    cu_q = [0] + list(torch.tensor(lq).cumsum(0).tolist())
    cu_k = [0] + list(torch.tensor(lk).cumsum(0).tolist())
    causal = kind in ("causal_self", "causal_fewer_queries")
    q, go = C.randn(g, cu_q[-1], hq, d), C.randn(g, cu_q[-1], hq, d)
    k, v = C.randn(g, cu_k[-1], hk, d), C.randn(g, cu_k[-1], hk, d)
    key_mask = None
    if kind == "key_mask":
        key_mask = torch.rand(cu_k[-1], generator=g) > 0.3
        for c in cu_k[:-1]:
            key_mask[c] = True  # every row keeps a key
    qd, kd, vd = (t.to(dev).requires_grad_() for t in (q, k, v))
    native.reset_counters()
    out = native.sdpa_varlen(qd, kd, vd, cu_q, cu_k, is_causal=causal,
                             attn_mask=None if key_mask is None else key_mask.to(dev))
    out.backward(go.to(dev))
    torch.cuda.synchronize()
    assert native.counters()["attention_backward"] == 1, native.counters()
    ref = _varlen_ref_grads(q, k, v, go, cu_q, cu_k, causal, key_mask)
    for name, got, want in zip(("dq", "dk", "dv"), (qd.grad, kd.grad, vd.grad), ref):
        err = (got.cpu().double() - want).abs().max().item()
        assert err <= 3e-2 * max(want.abs().max().item(), 1.0), (kind, name, err)


def test_varlen_fp32_inputs_give_fp32_gradients(native, dev):
    """fp32 q / k / v that require gradients: the forward casts to bf16 and returns fp32,
    the backward runs the bf16 kernels on bf16 copies and returns fp32 gradients, within
    bf16 accuracy of float64 autograd."""
    g = C.gen(977)
    hq, hk, d = 4, 2, 64
    lq = [50, 17, 90]
    cu = [0] + list(torch.tensor(lq).cumsum(0).tolist())
    q, go = torch.randn(cu[-1], hq, d, generator=g), torch.randn(cu[-1], hq, d, generator=g)
    k, v = torch.randn(cu[-1], hk, d, generator=g), torch.randn(cu[-1], hk, d, generator=g)
    qd, kd, vd = (t.to(dev).requires_grad_() for t in (q, k, v))
    native.reset_counters()
    out = native.sdpa_varlen(qd, kd, vd, cu, cu, is_causal=True)
    assert out.dtype == torch.float32
    out.backward(go.to(dev))
    torch.cuda.synchronize()
    assert native.counters()["attention_backward"] == 1, native.counters()
    # The kernels see bf16 operands: compare with float64 autograd of those.
    ref = _varlen_ref_grads(*(t.bfloat16() for t in (q, k, v, go)), cu, cu, True)
    for name, got, want in zip(("dq", "dk", "dv"), (qd.grad, kd.grad, vd.grad), ref):
        assert got.dtype == torch.float32, name
        err = (got.cpu().double() - want).abs().max().item()
        assert err <= 3e-2 * max(want.abs().max().item(), 1.0), (name, err)


def test_reference_varlen_ops_forward_and_backward(native, dev):
    """The reference's packed ops as its glue calls them (``torch_backend/varlen.py``):
    ``_varlen_plan`` on the host, ``_sdpa_varlen(..., stats=True, key_mask)`` and
    ``_sdpa_varlen_backward`` from the output, in the reference's key-mask form (bf16,
    divided by the scale).  Gradients also flow through autograd on ``_sdpa_varlen``."""
    g = C.gen(970)
    cu_q, cu_k = [0, 30, 31, 120], [0, 40, 41, 150]
    hq, hk, d = 4, 2, 64
    scale = d ** -0.5
    q, go = C.randn(g, cu_q[-1], hq, d), C.randn(g, cu_q[-1], hq, d)
    k, v = C.randn(g, cu_k[-1], hk, d), C.randn(g, cu_k[-1], hk, d)
    keep = torch.rand(cu_k[-1], generator=g) > 0.25
    for c in cu_k[:-1]:
        keep[c] = True
    # varlen.key_mask: bool -> (mask - 1) * (5e5 / scale) in bf16
    km = ((keep.to(torch.bfloat16) - 1.0) * (5e5 / scale)).to(torch.bfloat16)
    records, masks = torch.ops.ktt._varlen_plan(cu_q, cu_k, True, scale, False)
    records, masks = records.to(dev), masks.to(dev)
    qd, kd, vd = (t.to(dev).requires_grad_() for t in (q, k, v))
    native.reset_counters()
    out, lse = torch.ops.ktt._sdpa_varlen(qd, kd, vd, records, masks, cu_q, cu_k, True, scale, True, km.to(dev),
                                          False)
    assert lse.shape == (hq, cu_q[-1])
    out.backward(go.to(dev))
    torch.cuda.synchronize()
    c = native.counters()
    assert c["attention"] == 1 and c["attention_backward"] == 1, c
    ref_out, _ = oatt.sdpa_varlen(C.f64(q), C.f64(k), C.f64(v), cu_q, cu_k, is_causal=True,
                                  key_mask=keep.numpy())
    assert np.abs(out.detach().cpu().double().numpy() - ref_out).max() < 2e-2
    ref = _varlen_ref_grads(q, k, v, go, cu_q, cu_k, True, keep)
    for name, got, want in zip(("dq", "dk", "dv"), (qd.grad, kd.grad, vd.grad), ref):
        err = (got.cpu().double() - want).abs().max().item()
        assert err <= 3e-2 * max(want.abs().max().item(), 1.0), (name, err)
    # The backward op called directly gives the same gradients.
    dq, dk, dv = torch.ops.ktt._sdpa_varlen_backward(go.to(dev), out.detach(), qd.detach(), kd.detach(), vd.detach(),
                                                     records, masks, records, masks, cu_q, cu_k, True, scale,
                                                     km.to(dev))
    assert torch.equal(dq, qd.grad) and torch.equal(dk, kd.grad) and torch.equal(dv, vd.grad)


def test_varlen_packed_mask_backward(native, dev):
    """Per-row block-packed masks (config 4's masked run form) through autograd, one
    fully-masked row included."""
    g = C.gen(971)
    lens = [40, 75]
    cu = [0, 40, 115]
    hq, hk, d = 4, 2, 128
    q, go = C.randn(g, cu[-1], hq, d), C.randn(g, cu[-1], hq, d)
    k, v = C.randn(g, cu[-1], hk, d), C.randn(g, cu[-1], hk, d)
    blocks = []
    for i, n in enumerate(lens):
        keep = torch.ones(n, n, dtype=torch.bool).tril() & (torch.rand(n, n, generator=g) > 0.1)
        if i == 0:
            keep[5] = False
        blocks.append(torch.zeros(n, n).masked_fill(~keep, float("-inf")).reshape(-1))
    pm = torch.cat(blocks)
    qd, kd, vd = (t.to(dev).requires_grad_() for t in (q, k, v))
    native.reset_counters()
    out = native.sdpa_varlen(qd, kd, vd, cu, is_causal=True, packed_mask=pm.to(dev))
    out.backward(go.to(dev))
    torch.cuda.synchronize()
    assert native.counters()["attention_backward"] == 1
    # float64 reference per sequence with the reference's fully-masked-row rule.
    grads = [torch.zeros(t.shape, dtype=torch.float64) for t in (q, k, v)]
    off = 0
    for a, b in zip(cu[:-1], cu[1:]):
        n = b - a
        m = pm[off:off + n * n].reshape(n, n).double().clamp_min(-5e5)
        off += n * n
        # causal visibility stays; a row whose visible keys are all masked attends over
        # their raw scores (the forward's rule)
        vis = torch.ones(n, n, dtype=torch.bool).tril()
        dead = ((m <= -5e5) | ~vis).all(-1, keepdim=True)
        m = m.masked_fill(dead & vis, 0.0).masked_fill(~vis, float("-inf"))
        qs, ks, vs = (t.double().transpose(0, 1)[None].requires_grad_() for t in (q[a:b], k[a:b], v[a:b]))
        o = F.scaled_dot_product_attention(qs, ks.repeat_interleave(2, 1), vs.repeat_interleave(2, 1), attn_mask=m)
        o.backward(go[a:b].double().transpose(0, 1)[None])
        for gsum, t in zip(grads, (qs, ks, vs)):
            gsum[a:b] = t.grad[0].transpose(0, 1)
    for name, got, want in zip(("dq", "dk", "dv"), (qd.grad, kd.grad, vd.grad), grads):
        err = (got.cpu().double() - want).abs().max().item()
        assert err <= 5e-2 * max(want.abs().max().item(), 1.0), (name, err)


def test_torch_varlen_attn_forward_and_backward(native, dev):
    """torch.nn.attention.varlen.varlen_attn on GPU tensors: both of torch's ops run the
    kernels (``torch_attn::_varlen_attn`` and ``_varlen_attn_backward``)."""
    from torch.nn.attention.varlen import varlen_attn

    g = C.gen(972)
    cu = [0, 50, 51, 130]
    q, go = C.randn(g, cu[-1], 4, 64), C.randn(g, cu[-1], 4, 64)
    k, v = C.randn(g, cu[-1], 4, 64), C.randn(g, cu[-1], 4, 64)
    qd, kd, vd = (t.to(dev).requires_grad_() for t in (q, k, v))
    cu_t = torch.tensor(cu, dtype=torch.int32, device=dev)
    native.reset_counters()
    out = varlen_attn(qd, kd, vd, cu_t, cu_t, 79, 79, is_causal=True)
    out.backward(go.to(dev))
    torch.cuda.synchronize()
    c = native.counters()
    assert c["attention"] == 1 and c["attention_backward"] == 1, c
    ref = _varlen_ref_grads(q, k, v, go, cu, cu, True)
    for name, got, want in zip(("dq", "dk", "dv"), (qd.grad, kd.grad, vd.grad), ref):
        err = (got.cpu().double() - want).abs().max().item()
        assert err <= 3e-2 * max(want.abs().max().item(), 1.0), (name, err)


def _grads_of(q, k, v, go, mask):
    ts = [t.detach().requires_grad_() for t in (q, k, v)]
    F.scaled_dot_product_attention(*ts, attn_mask=mask).backward(go)
    return [t.grad for t in ts]


@pytest.mark.parametrize("kind", ["add", "bool", "pad"])
@pytest.mark.parametrize("b,h,s,d", [(1, 2, 70, 64), (1, 2, 70, 128), (4, 8, 257, 128), (4, 8, 257, 96), (2, 2, 66, 256)])
def test_masked_keys_may_hold_anything(native, dev, b, h, s, d, kind):
    """dK and dV do not depend on the K rows of masked keys (NaN, infinities, values whose
    product overflows) and are exactly 0 there.  (dQ sums dS K over every key, so a NaN row
    reaches it.)"""
    print(f"masked rows {b}x{h}x{s}x{d} {kind}", flush=True)
    g = C.gen(980 + d)
    q, k, v, go = (C.randn(g, b, h, s, d).to(dev) for _ in range(4))
    hidden = torch.rand(s, generator=g) < 0.4
    hidden[::32] = False  # each tile keeps a key
    if kind == "pad":
        m = (~hidden).view(1, 1, 1, s).expand(b, 1, 1, s)
    else:
        m = (torch.rand(1, 1, s, s, generator=g) >= 0.2) & ~hidden
        m[..., ::32] = True
        if kind == "add":
            m = torch.randn(1, 1, s, s, generator=g).bfloat16().masked_fill(~m, -torch.inf)
    hidden, m = hidden.to(dev), m.to(dev)
    clean = k.masked_fill(hidden[None, None, :, None], 0.0)
    spoilt = clean.clone()
    at = torch.nonzero(hidden).flatten()
    for i, value in enumerate((torch.nan, torch.inf, -torch.inf, torch.finfo(k.dtype).max)):
        spoilt[:, :, at[i::4]] = value
    _, dk, dv = _grads_of(q, spoilt, v, go, m)
    _, want_dk, want_dv = _grads_of(q, clean, v, go, m)
    assert torch.isfinite(want_dk).all() and torch.isfinite(want_dv).all()
    assert torch.equal(dk, want_dk) and torch.equal(dv, want_dv)
    assert not dk[:, :, at].any() and not dv[:, :, at].any()


@pytest.mark.parametrize("b,h,s", [(2, 2, 128), (4, 8, 257)])
def test_additive_mask_rounds_once(native, dev, b, h, s):
    """A logit of -1e5 over whole rows leaves the probabilities as they are but for roundings
    at its size.  In base 2 (2^17 .. 2^18, a rounding is off by 2^-6 / sqrt(12) in the mean):
    one of score + logit, one of the forward's lse before and one after it is scaled back to
    base 2, and one of its natural value (2^-7 log2(e) / sqrt(12)).  dV is off by ln 2 times
    their root sum of squares."""
    print(f"rounds once {b}x{h}x{s}", flush=True)
    g = C.gen(990 + s)
    q, k, v, go = (C.randn(g, b, h, s, 128).half() for _ in range(4))
    mask = torch.full((1, 1, s, s), -1e5)
    _, _, dv = _grads_of(q.to(dev), k.to(dev), v.to(dev), go.to(dev), mask.to(dev))
    p = torch.softmax(q.double() @ k.double().transpose(-1, -2) / 128**0.5, -1)
    want = p.transpose(-1, -2) @ go.double()
    off = ((dv.cpu().double() - want).norm() / want.norm()).item()
    once = 2.0**-6 / 12**0.5 * (3 + (np.log2(np.e) / 2) ** 2) ** 0.5 * np.log(2)
    print(f"  {off:.2e}, derived {once:.2e}", flush=True)
    assert off <= 1.2 * once


@pytest.mark.parametrize("kind", ["bool", "additive", "float32", "pad"])
@pytest.mark.parametrize("b,hq,hk,sq,sk,d,dtype", [
    (4, 8, 8, 257, 259, 128, torch.bfloat16),
    (4, 8, 8, 257, 259, 96, torch.float16),
    (6, 12, 6, 161, 225, 128, torch.float16),
])  # fmt: skip
def test_masked_backward_of_128_key_workgroups(native, dev, b, hq, hk, sq, sk, d, dtype, kind):
    """Masked calls large enough that a dK / dV workgroup takes 128 keys (32-row tiles, V in
    LDS), with key and row counts off both, and a row that keeps no key."""
    # 64-key and 64- or 128-row workgroups in all: more than the 256 that keep 64 keys each.
    dq_wgs = b * hq * -(-sq // 128)
    assert b * hk * -(-sk // 64) + (dq_wgs if dq_wgs >= 256 else b * hq * -(-sq // 64)) > 256
    print(f"128-key workgroups {b}x{hq}/{hk}x{sq}/{sk}x{d} {kind}", flush=True)
    g = C.gen(d + sq + len(kind))
    q, go = C.randn(g, b, hq, sq, d).to(dtype), C.randn(g, b, hq, sq, d).to(dtype)
    k, v = C.randn(g, b, hk, sk, d).to(dtype), C.randn(g, b, hk, sk, d).to(dtype)
    if kind == "bool":
        mask = torch.rand(b, hq, sq, sk, generator=g) > 0.3
        mask[1, 1, 7] = False
    elif kind == "pad":
        lens = torch.randint(1, sk + 1, (b,), generator=g)
        mask = (torch.arange(sk)[None, :] < lens[:, None]).reshape(b, 1, 1, sk)
    else:
        mask = torch.randn(b if kind == "float32" else 1, 1, sq, sk, generator=g)
        mask = mask.masked_fill(torch.rand(mask.shape, generator=g) < 0.2, -torch.inf)
        mask[0, 0, 3] = -torch.inf
        if kind == "additive":
            mask = mask.to(dtype)
    ts = [t.to(dev).requires_grad_() for t in (q, k, v)]
    native.reset_counters()
    out = F.scaled_dot_product_attention(*ts, attn_mask=mask.to(dev), enable_gqa=hq != hk)
    out.backward(go.to(dev))
    assert native.counters()["attention_backward"] == 1
    keep = mask if kind in ("bool", "pad") else mask > -torch.inf
    dead = ~keep.any(-1, keepdim=True)  # these rows are over their raw scores
    bias = torch.zeros(mask.shape, dtype=torch.float64) if kind in ("bool", "pad") else mask.double().masked_fill(~keep, 0.0)
    bias = bias.masked_fill(~keep & ~dead, -torch.inf)
    rs = [t.double().requires_grad_() for t in (q, k, v)]
    kr, vr = (t.repeat_interleave(hq // hk, 1) for t in rs[1:])
    p = torch.softmax(rs[0] @ kr.transpose(-1, -2) / d**0.5 + bias, -1)
    (p @ vr).backward(go.double())
    half_ulp = 2.0**-9 if dtype == torch.bfloat16 else 2.0**-12
    for name, a, r in zip(("dq", "dk", "dv"), ts, rs):
        # P, dS, out and the gradient itself round to the type, O in the row dot too: five half
        # ulps of what the gradient's size is made of, in the mean over a tensor.
        off = ((a.grad.cpu().double() - r.grad).norm() / r.grad.norm()).item()
        print(f"  {name} {off:.2e}", flush=True)
        assert torch.isfinite(a.grad).all() and off <= 5 * half_ulp, (name, off)


@pytest.mark.parametrize("b,hq,hk,s,d", [(1, 14, 2, 2048, 64), (1, 24, 24, 1000, 128), (1, 2, 1, 70, 256)])
def test_backward_in_a_workspace_of_the_plans_size(native, dev, b, hq, hk, s, d):
    """kmi_attn_bwd in the least workspace it takes gives autograd's gradients and writes
    nothing past it."""
    print(f"workspace {b}x{hq}/{hk}x{s}x{d}", flush=True)
    g = C.gen(77 + d)
    q, k, v, go = (C.randn(g, b, h, s, d).to(dev) for h in (hq, hk, hk, hq))
    ts = [t.detach().requires_grad_() for t in (q, k, v)]
    F.scaled_dot_product_attention(*ts, is_causal=True, enable_gqa=True).backward(go)
    out, lse = torch.ops.aten._scaled_dot_product_fused_attention_overrideable(q, k, v, None, 0.0, True)[:2]
    grads = [torch.full_like(t, torch.nan) for t in (q, k, v)]
    a = capi.AttnBwdArgs()
    for field, t in zip(("q", "k", "v", "out", "grad_out", "lse", "grad_q", "grad_k", "grad_v"),
                        (q, k, v, out, go, lse, *grads)):  # fmt: skip
        setattr(a, field, t.data_ptr())
    for field, t in zip(("q", "k", "v", "o", "do", "dq", "dk", "dv", "lse"), (q, k, v, out, go, *grads, lse)):
        getattr(a, field + "_stride")[:] = t.stride()[:3]
    a.dtype, a.causal, a.scale = capi.KMI_BF16, 1, d**-0.5
    a.batch, a.heads_q, a.heads_kv, a.seq_q, a.seq_k, a.head_dim = b, hq, hk, s, s, d
    n = ctypes.c_size_t()
    capi.check(capi.lib().kmi_attn_bwd_plan_bytes(ctypes.byref(a), ctypes.byref(n)))
    work = torch.full((n.value + 4096,), 0xAB, dtype=torch.uint8, device=dev)
    capi.check(capi.lib().kmi_attn_bwd(ctypes.byref(a), work.data_ptr(), n.value, torch.cuda.current_stream().cuda_stream))
    torch.cuda.synchronize()
    assert (work[n.value :] == 0xAB).all()
    for got, t in zip(grads, ts):
        assert torch.equal(got, t.grad)


def _close_to_float64(got, want, dtype, what):
    """P, dS, out and the gradient itself round to the type, O in the row dot too: five half ulps
    of what the gradient's size is made of, in the mean over a tensor."""
    half_ulp = 2.0**-9 if dtype == torch.bfloat16 else 2.0**-12
    off = ((got.cpu().double() - want).norm() / want.norm()).item()
    print(f"  {what} {off:.2e}", flush=True)
    assert torch.isfinite(got).all() and off <= 5 * half_ulp, (what, off)


@pytest.mark.parametrize("layout", ["rows", "keys first", "every second key", "per batch", "per head"])
@pytest.mark.parametrize("kind", ["bool", "additive", "float32"])
@pytest.mark.parametrize("b,h,sq,sk,d", [(2, 3, 22, 22, 72), (2, 2, 33, 65, 64), (3, 2, 70, 90, 128), (2, 2, 40, 31, 32)])
def test_masked_blocks_at_the_edges(native, dev, b, h, sq, sk, d, kind, layout):
    """Masks in every stride order over row and key counts off the 32x32 blocks."""
    print(f"mask edges {b}x{h}x{sq}/{sk}x{d} {kind} {layout}", flush=True)
    g = C.gen(sq + d + len(layout))
    dtype = torch.bfloat16
    q, go = (C.randn(g, b, h, sq, d) for _ in range(2))
    k, v = (C.randn(g, b, h, sk, d) for _ in range(2))
    lead = {"per batch": (b, 1), "per head": (1, h)}.get(layout, (1, 1))
    mask = torch.randn(*lead, sq, sk, generator=g)
    if kind == "additive":
        mask = mask.to(dtype)
    hidden = torch.rand(*lead, sq, sk, generator=g) < 0.3
    hidden[..., 0] = False
    mask = ~hidden if kind == "bool" else mask.masked_fill(hidden, -torch.inf)
    if layout == "keys first":
        placed = mask.transpose(-1, -2).contiguous().to(dev).transpose(-1, -2)
    elif layout == "every second key":
        placed = torch.zeros(*lead, sq, 2 * sk, dtype=mask.dtype, device=dev)[..., ::2]
        placed.copy_(mask)
    elif layout == "per batch":
        placed = mask[:, :, :1].to(dev).expand(-1, -1, sq, -1)  # one row of keys for every row
        mask = mask[:, :, :1].expand(-1, -1, sq, -1)
    else:
        placed = mask.to(dev)
    ts = [t.to(dev).requires_grad_() for t in (q, k, v)]
    native.reset_counters()
    F.scaled_dot_product_attention(*ts, attn_mask=placed).backward(go.to(dev))
    assert native.counters()["attention_backward"] == 1
    rs = [t.double().requires_grad_() for t in (q, k, v)]
    bias = torch.zeros(mask.shape, dtype=torch.float64).masked_fill(~mask, -torch.inf) if kind == "bool" else mask.double()
    (torch.softmax(rs[0] @ rs[1].transpose(-1, -2) / d**0.5 + bias, -1) @ rs[2]).backward(go.double())
    for name, a, r in zip(("dq", "dk", "dv"), ts, rs):
        _close_to_float64(a.grad, r.grad, dtype, name)


@pytest.mark.parametrize("mask", ["none", "causal", "bool"])
@pytest.mark.parametrize("b,hq,hk,sq,sk", [(1, 2, 2, 1, 1), (2, 6, 3, 17, 50), (1, 14, 2, 32, 64), (2, 4, 1, 33, 64), (2, 4, 4, 32, 65),
                                              (4, 32, 8, 9, 2050)])
@pytest.mark.parametrize("d,dtype", [(24, torch.bfloat16), (64, torch.float16), (72, torch.bfloat16), (128, torch.float16)])
def test_few_rows_and_keys(native, dev, b, hq, hk, sq, sk, d, dtype, mask):
    """Both sides of the line between attn_bwd_grads and the tile kernel."""
    print(f"few rows {b}x{hq}/{hk}x{sq}/{sk}x{d} {mask}", flush=True)
    g = C.gen(sq + sk + d)
    q, go = (C.randn(g, b, hq, sq, d).to(dtype) for _ in range(2))
    k, v = (C.randn(g, b, hk, sk, d).to(dtype) for _ in range(2))
    seen = torch.ones(sq, sk, dtype=torch.bool)
    if mask == "causal":
        seen = seen.tril()
    elif mask == "bool":
        seen = torch.rand(sq, sk, generator=g) > 0.3
        seen[:, 0] = True
    ts = [t.to(dev).requires_grad_() for t in (q, k, v)]
    native.reset_counters()
    F.scaled_dot_product_attention(*ts, attn_mask=seen.to(dev) if mask == "bool" else None, is_causal=mask == "causal",
                                   enable_gqa=hq != hk).backward(go.to(dev))
    assert native.counters()["attention_backward"] == 1
    rs = [t.double().requires_grad_() for t in (q, k, v)]
    kr, vr = (t.repeat_interleave(hq // hk, 1) for t in rs[1:])
    bias = torch.zeros(sq, sk, dtype=torch.float64).masked_fill(~seen, -torch.inf)
    (torch.softmax(rs[0] @ kr.transpose(-1, -2) / d**0.5 + bias, -1) @ vr).backward(go.double())
    for name, a, r in zip(("dq", "dk", "dv"), ts, rs):
        if sk > 1 or name == "dv":  # (one key: dq and dk are zero but for roundings)
            _close_to_float64(a.grad, r.grad, dtype, name)
