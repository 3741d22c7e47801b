"""The attention kernels whose waves share out the streamed rows of a 32-row block (few heads), in
bf16 and for fp32 as three bf16 planes, against fp64 attention: fewer tiles than waves, one tile
more or less than the waves' turns and ragged last tiles (bf16 up to 256 keys: the 128-row kernels).
More heads, on either side of the rule that chooses the form: test_gpu_form_limits.py."""
import math

import pytest
import torch

from test_gpu_f32_forms import attention64

pytestmark = pytest.mark.gpu

LENGTHS = [1, 31, 33, 64, 97, 129, 160, 257, 289, 511, 1199, 1201]


def rel(a, b):
    return float((a.double() - b).norm() / b.norm())


@pytest.mark.parametrize("d", [32, 64, 128])
@pytest.mark.parametrize("T", LENGTHS)
def test_bf16(lib, T, d):
    B, H = 1, 3
    g = torch.Generator(device="cuda:0").manual_seed(T + d)
    q, k, v, do = (torch.randn((B, H, T, d), generator=g, device="cuda:0").bfloat16()
                   for _ in range(4))
    scale = 1.0 / math.sqrt(d)
    o, m, l = lib.attention_forward(q, k, v, scale)
    dq, dk, dv, _ = lib.attention_backward(q, k, v, o, do, m, l, scale)
    torch.cuda.synchronize()
    want = attention64(q, k, v, do, scale)
    s = torch.matmul(q.double(), k.double().transpose(2, 3).contiguous()) * scale
    mask = torch.ones((T, T), dtype=torch.bool, device=q.device).triu_(1)
    lse = torch.logsumexp(s.masked_fill(mask, -math.inf), -1)
    # m + ln l against fp64: the scores' scale and bf16 rounding of c*q in the folded forward
    assert float((m.double() + l.double().log() - lse).abs().max()) <= 2e-2
    for name, got, exp in zip(("o", "dq", "dk", "dv"), (o, dq, dk, dv), want):
        # bf16's gate; T = 1 has dq = dk = 0 exactly
        if float(exp.norm()) < 1e-9:
            assert float(got.double().abs().max()) <= 1e-2, name
        else:
            assert rel(got, exp) <= 2e-2, name


@pytest.mark.parametrize("d", [32, 64])
@pytest.mark.parametrize("T", LENGTHS)
def test_three_planes(lib, T, d):
    B, H = 1, 3
    g = torch.Generator(device="cuda:0").manual_seed(T + d)
    q, k, v, do = (torch.randn((B, H, T, d), generator=g, device="cuda:0") for _ in range(4))
    scale = 1.0 / math.sqrt(d)
    nan = lambda *s: torch.full(s, float("nan"), device="cuda:0")
    planes = torch.empty(lib.f32x3_workspace_bytes(B, H, T, d), dtype=torch.uint8, device="cuda:0")
    o, m, l, ws = nan(B, H, T, d), nan(B, H, T), nan(B, H, T), nan(B, H, T)
    dq, dk, dv = (nan(B, H, T, d) for _ in range(3))
    lib.tiled_causal_attention_forward_f32x3(q, k, v, o, B, H, T, d, scale, planes, m, l)
    # the forward's planes of q, k and v are the backward's
    lib.tiled_causal_attention_backward_f32x3(q, k, v, o, do, m, l, dq, dk, dv, ws, B, H, T, d,
                                              scale, planes, True)
    torch.cuda.synchronize()
    for name, got, exp in zip(("o", "dq", "dk", "dv"), (o, dq, dk, dv),
                              attention64(q, k, v, do, scale)):
        assert float((got.double() - exp).abs().max()) <= 1e-5, name
