"""Keys whose scores overflow to -infinity have weight 0 and no gradient, also where they are all
that one wave of a workgroup sees of a row: a whole 32-key tile, or the one visible key of a
diagonal tile."""
import math

import pytest
import torch

from gpu_util import default_scale

pytestmark = pytest.mark.gpu

BIG = 2.0 ** 66  # q.k = -2^132 for the masked keys


def reference(q, k, v, do, scale):
    q, k, v, do = (x.double().cpu() for x in (q, k, v, do))
    T = q.shape[1]
    s = torch.matmul(q, k.transpose(1, 2).contiguous()) * scale
    p = torch.softmax(s.masked_fill(torch.ones(T, T, dtype=torch.bool).triu(1), -math.inf), -1)
    o = torch.matmul(p, v)
    dp = torch.matmul(do, v.transpose(1, 2).contiguous())
    ds = p * (dp - (do * o).sum(-1, keepdim=True)) * scale
    tr = lambda x: x.transpose(1, 2).contiguous()
    return o, torch.matmul(ds, k), torch.matmul(tr(ds), q), torch.matmul(tr(p), do)


def run(lib, dtype, q, k, v, do, scale):
    N, T, d = q.shape
    q, k, v, do = (x.view(1, N, T, d) for x in (q, k, v, do))
    if dtype != "f32x3":
        o, m, l = lib.attention_forward(q, k, v, scale)
        dq, dk, dv, _ = lib.attention_backward(q, k, v, o, do, m, l, scale)
    else:
        f = dict(device="cuda:0", dtype=torch.float32)
        o, dq, dk, dv = (torch.empty_like(q) for _ in range(4))
        m, l, ws = (torch.empty((1, N, T), **f) for _ in range(3))
        planes = torch.empty(lib.f32x3_workspace_bytes(1, N, T, d), dtype=torch.uint8,
                             device="cuda:0")
        lib.tiled_causal_attention_forward_f32x3(q, k, v, o, 1, N, T, d, scale, planes, m, l)
        lib.tiled_causal_attention_backward_f32x3(q, k, v, o, do, m, l, dq, dk, dv, ws, 1, N, T,
                                                  d, scale, planes, True)
    torch.cuda.synchronize()
    return [x[0].double().cpu() for x in (o, dq, dk, dv, m, l)]


KINDS = [("f32", 32), ("f32", 64), ("f32", 128), ("f32x3", 32), ("f32x3", 64), ("bf16", 32),
         ("bf16", 64), ("bf16", 128)]
# few heads, which share out a workgroup's waves, and many; masked keys among the first 32 too (but
# for bf16 with many heads, whose kernels take a row's reference from its first 32 keys)
CASES = [(dtype, d, heads, first) for dtype, d in KINDS for heads in (2, 120)
         for first in (False, True) if not (first and dtype == "bf16" and heads > 2)]


@pytest.mark.parametrize("dtype,d,heads,first", CASES)
def test_masked_keys(lib, dtype, d, heads, first):
    T, scale = 300, default_scale(d)
    g = torch.Generator(device="cuda:0").manual_seed(d + heads)
    q, k, v, do = (torch.randn((heads, T, d), generator=g, device="cuda:0") for _ in range(4))
    masked = list(range(32, 64)) + [64, 129, 160, 287] + list(range(192, 224))
    if first:
        masked += list(range(32))
    q[:, :, 0] = BIG
    k[:, :, 0] = 0.0
    k[:, masked, 0] = -BIG
    if dtype == "bf16":
        q, k, v, do = (x.bfloat16() for x in (q, k, v, do))
    if first:  # rows without a key have no result
        do[:, :65] = 0.0
    want = reference(q, k, v, do, scale)
    o, dq, dk, dv, m, l = run(lib, dtype, q, k, v, do, scale)
    r0 = 65 if first else 0
    assert bool(torch.isfinite(m[:, r0:]).all()) and bool((l[:, r0:] > 0).all())
    tol = {"f32": 4e-6, "f32x3": 8e-6, "bf16": 2.5e-2}[dtype]  # rounding of the dtype, in 2-norms
    rel = lambda a, b: float((a - b).norm() / b.norm())
    assert rel(o[:, r0:], want[0][:, r0:]) < tol
    if first:
        return
    # column 0 of dK carries the factor of q's
    dk[:, :, 0] /= BIG
    want[2][:, :, 0] /= BIG
    for got, exp in zip((dq, dk, dv), want[1:]):
        assert bool(torch.isfinite(got).all())
        assert rel(got[:, :, 1:], exp[:, :, 1:]) < tol
    assert bool((dk[:, masked] == 0).all()) and bool((dv[:, masked] == 0).all())
