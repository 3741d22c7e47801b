"""The fp32 attention kernels on either side of the rule that chooses between their shared-tile
and per-wave forms (workgroups per CU, evenness of the last round, head dimension, stage), each
with ragged lengths, against fp64 attention on the same inputs."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu


def attention64(q, k, v, do, scale):
    """O, dQ, dK, dV of causal attention in fp64, head by head."""
    T = q.shape[2]
    mask = torch.ones((T, T), dtype=torch.bool, device=q.device).triu_(1)
    outs = []
    for b in range(q.shape[0]):
        Q, K, V, G = (x[b].double() for x in (q, k, v, do))
        s = torch.matmul(Q, K.transpose(1, 2).contiguous()) * scale
        p = torch.softmax(s.masked_fill(mask, -math.inf), -1)
        dp = torch.matmul(G, V.transpose(1, 2).contiguous())
        ds = p * (dp - (dp * p).sum(-1, keepdim=True)) * scale
        outs.append((torch.matmul(p, V), torch.matmul(ds, K),
                     torch.matmul(ds.transpose(1, 2).contiguous(), Q),
                     torch.matmul(p.transpose(1, 2).contiguous(), G)))
    return [torch.stack(x) for x in zip(*outs)]


@pytest.mark.parametrize("B,H,T,d", [
    (1, 27, 777, 64),    # under one workgroup a CU: per-wave
    (4, 16, 1024, 64),   # 512 = two a CU, even: shared
    (4, 16, 1000, 64),   # the same, ragged
    (4, 24, 769, 64),    # 672 with a nearly empty last block: per-wave
    (9, 16, 900, 64),    # over four a CU: dK/dV shared, forward and dQ per-wave
    (3, 15, 1000, 128),  # 360: dK/dV shared, forward and dQ per-wave
    (8, 8, 901, 128),    # 512: all shared
    (3, 14, 700, 128),   # 252: all per-wave
])
def test_forms_vs_fp64(lib, B, H, T, d):
    g = torch.Generator(device="cuda:0").manual_seed(B * H + T + d)
    q, k, v, do = (torch.randn((B, H, T, d), generator=g, device="cuda:0") for _ in range(4))
    scale = 1.0 / math.sqrt(d)
    o, m, l = lib.attention_forward(q, k, v, scale)
    dq, dk, dv, _ = lib.attention_backward(q, k, v, o, do, m, l, scale)
    torch.cuda.synchronize()
    for name, got, want in zip(("o", "dq", "dk", "dv"), (o, dq, dk, dv),
                               attention64(q, k, v, do, scale)):
        err = float((got.double() - want).abs().max())
        assert err <= 1e-5, f"{name}: {err:.3e}"
