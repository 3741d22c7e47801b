"""The attention kernels on both sides of the rules that pick their forms, at lengths that leave the
last tile and block of every head partly past T, against fp64 attention: many heads, where the
128-row kernels run, and fewer, where the others do.  Each case states the forms it means to run."""
import math

import pytest
import torch

from gpu_util import sched
from test_gpu_f32_forms import attention64

pytestmark = pytest.mark.gpu


def inputs(B, H, T, d, dtype=torch.float32):
    g = torch.Generator(device="cuda:0").manual_seed(B * H + T + d)
    return [torch.randn((B, H, T, d), generator=g, device="cuda:0").to(dtype) for _ in range(4)]


def nan(*shape):
    return torch.full(shape, float("nan"), device="cuda:0")


def pack(q, k, v, do):
    """(B, T, 3HC) QKV and the merged dO."""
    B, H, T, d = q.shape
    qkv = torch.stack([x.transpose(1, 2) for x in (q, k, v)], 2).reshape(B, T, 3 * H * d)
    return qkv.contiguous(), do.transpose(1, 2).reshape(B, T, H * d).contiguous()


def unpack(dqkv, B, H, T, d):
    return dqkv.reshape(B, T, 3, H, d).permute(2, 0, 3, 1, 4)


def worst(got, want):
    return float((got.double() - want).abs().max())


S, W = "shared", "per-wave"


@pytest.mark.parametrize("d,T,B,H,forms", [
    (64, 901, 4, 16, (S, S, S)), (64, 1000, 10, 16, (S, W, S)), (64, 777, 3, 9, (W, W, W)),
    (64, 2047, 4, 8, (S, S, S)), (64, 2080, 4, 8, (W, W, W)), (64, 100, 20, 10, (S, W, S)),
    (128, 901, 8, 8, (S, S, S)), (128, 257, 8, 15, (S, W, S)), (128, 700, 3, 14, (W, W, W)),
    (128, 100, 20, 10, (S, S, S))])
def test_fp32(lib, d, T, B, H, forms):
    """Head-major and from the packed layout into the merged one, in the two-stage order and the
    dS-first one, whose dK and dV are the same bits."""
    assert tuple(sched("form", st, d, T, B * H) for st in ("fwd", "dq", "dkdv")) == forms
    q, k, v, do = inputs(B, H, T, d)
    scale = 1.0 / math.sqrt(d)
    want = attention64(q, k, v, do, scale)
    o, m, l = lib.attention_forward(q, k, v, scale)
    grads = lib.attention_backward(q, k, v, o, do, m, l, scale)[:3]
    for name, got, exp in zip(("o", "dq", "dk", "dv"), (o, *grads), want):
        assert worst(got, exp) <= 1e-5, name
    qkv, dom = pack(q, k, v, do)
    om, two, one = nan(B, T, H * d), torch.full_like(qkv, math.nan), torch.full_like(qkv, math.nan)
    m2, l2, ws, ws2 = (nan(B, H, T) for _ in range(4))
    ds = nan(lib.f32_ds_workspace_bytes(B, H, T, d) // 4)
    a = (B, H, T, d, scale)
    lib.fused_causal_attention_forward(qkv, om, *a, m2, l2)
    lib.fused_causal_attention_backward(qkv, om, dom, m2, l2, two, ws, *a)
    lib.fused_causal_attention_backward_ds(qkv, om, dom, m2, l2, one, ws2, ds, *a)
    torch.cuda.synchronize()
    assert torch.equal(om.reshape(B, T, H, d).transpose(1, 2), o)
    assert torch.equal(ws, ws2)
    for i, (x, y) in enumerate(zip(unpack(two, B, H, T, d), unpack(one, B, H, T, d))):
        assert torch.equal(x, grads[i])
        if i > 0:
            assert torch.equal(x, y)
        else:
            assert worst(y, want[1]) <= 1e-5


# heads below all of the three stages' limits and above
BF16 = [(32, 777, 40, 56), (32, 1531, 28, 48), (64, 257, 29, 43), (64, 777, 20, 28),
        (64, 1531, 17, 24), (128, 300, 20, 40), (128, 777, 14, 21), (128, 1531, 10, 17)]


@pytest.mark.parametrize("d,T,H,form", [(d, T, h, f) for d, T, few, many in BF16
                                        for h, f in ((few, "split"), (many, "block"))])
def test_bf16(lib, d, T, H, form):
    assert {sched("form", st, 1, d, T, H) for st in ("fwd", "dq", "dkdv")} == {form}
    q, k, v, do = inputs(1, H, T, d, torch.bfloat16)
    scale = 1.0 / math.sqrt(d)
    o, m, l = lib.attention_forward(q, k, v, scale)
    dq, dk, dv, _ = lib.attention_backward(q, k, v, o, do, m, l, scale)
    torch.cuda.synchronize()
    for name, got, exp in zip(("o", "dq", "dk", "dv"), (o, dq, dk, dv),
                              attention64(q, k, v, do, scale)):
        assert float((got.double() - exp).norm() / exp.norm()) <= 2e-2, name


# heads below the limits of the forward and the backward and above both
THREE = [(32, 100, 47, 50), (32, 300, 46, 55), (32, 777, 32, 36), (32, 1211, 24, 27),
         (64, 100, 60, 66), (64, 300, 37, 46), (64, 777, 18, 27), (64, 1211, 14, 23)]


@pytest.mark.parametrize("d,T,H,form", [(d, T, h, f) for d, T, few, many in THREE
                                        for h, f in ((few, "split"), (many, "block"))])
def test_three_planes(lib, d, T, H, form):
    """From the packed layout into the merged one, with the forward's planes, in the two-stage order
    and with dS."""
    stages = ("dkdv",) if T <= 256 else ("fwd", "dkdv")  # short forwards share nothing
    assert {sched("form", st, 3, d, T, H) for st in stages} == {form}
    q, k, v, do = inputs(1, H, T, d)
    scale = 1.0 / math.sqrt(d)
    want = attention64(q, k, v, do, scale)
    qkv, dom = pack(q, k, v, do)
    a = (1, H, T, d, scale)
    o, m, l, ws, ws2 = nan(1, T, H * d), *(nan(1, H, T) for _ in range(4))
    planes = torch.empty(lib.f32x3_planes_bytes(1, H, T, d), dtype=torch.uint8, device="cuda:0")
    lib.fused_causal_attention_forward_f32x3(qkv, o, *a, planes, m, l)
    assert worst(o.reshape(1, T, H, d).transpose(1, 2), want[0]) <= 1e-5
    one, two = torch.full_like(qkv, math.nan), torch.full_like(qkv, math.nan)
    n = lib.f32x3_ds_workspace_bytes(1, H, T, d)
    ds = nan(n // 4) if n else None
    lib.fused_causal_attention_backward_ds_f32x3(qkv, o, dom, m, l, one, ws, ds, *a, planes, True)
    two_ws = torch.empty(lib.f32x3_workspace_bytes(1, H, T, d), dtype=torch.uint8, device="cuda:0")
    lib.fused_causal_attention_forward_f32x3(qkv, o, *a, two_ws, m, l)
    lib.fused_causal_attention_backward_dq_f32x3(qkv, o, dom, m, l, two, ws2, *a, two_ws, True)
    lib.causal_attention_backward_dkdv_f32x3(qkv, m, l, ws2, two, *a, two_ws)
    torch.cuda.synchronize()
    for i, (x, y) in enumerate(zip(unpack(one, 1, H, T, d), unpack(two, 1, H, T, d))):
        assert worst(x, want[1 + i]) <= 1e-5 and worst(y, want[1 + i]) <= 1e-5, "qkv"[i]
        if i > 0:
            assert torch.equal(x, y), "qkv"[i]


# (d, T, heads, form of dQ): heads few enough for the forward whose statistics are of unrounded c*Q
@pytest.mark.parametrize("d,T,H,form", [(32, 511, 8, "split"), (64, 511, 8, "split"),
                                        (64, 1531, 23, "block"), (128, 777, 6, "split"),
                                        (128, 777, 20, "block")])
def test_bf16_dq_of_few_heads(lib, d, T, H, form):
    """dQ forms P from the scores that the forward's statistics are of, so that peaky rows (scores
    of variance 16) cost it no accuracy: P, dS and dQ are rounded to bf16 and D is taken from the
    rounded O, 2^-9 = 2e-3 of their terms at most each."""
    assert sched("form", "fwd", 1, d, T, H) == "split" and sched("form", "dq", 1, d, T, H) == form
    q, k, v, do = inputs(1, H, T, d)
    q, k, v, do = ((2 * q).bfloat16(), (2 * k).bfloat16(), v.bfloat16(), do.bfloat16())
    scale = 1.0 / math.sqrt(d)
    o, m, l = lib.attention_forward(q, k, v, scale)
    dq = lib.attention_backward(q, k, v, o, do, m, l, scale)[0]
    torch.cuda.synchronize()
    want = attention64(q, k, v, do, scale)[1]
    assert float((dq.double() - want).norm() / want.norm()) <= 5e-3
