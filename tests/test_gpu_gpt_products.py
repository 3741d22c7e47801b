"""The training-step harness's products with what they do to their sums (gpt_gemm.hpp), each alone
against fp64: bias, residual, GELU and its derivative on the outputs, and the bias gradient from the
operand tiles, on every tile shape with ragged M, N and K, with one slice of K and several.

The functions are internal to libtcamd_gpt.so, called by their linker names."""
import ctypes
import math

import pytest
import torch

from gpu_util import sched

pytestmark = pytest.mark.gpu

# (M, N, K, tile and slices): edges short of and past a tile
SIZES = [(4095, 4093, 1000, "256x256 1"), (767, 3071, 8190, "256x256 7"),
         (767, 767, 8190, "256x128 14"), (4093, 4099, 300, "128x128 1"),
         (771, 765, 4100, "128x128 12"), (4100, 770, 770, "128x64 1"), (1030, 1025, 500, "64x64 1"),
         (257, 513, 1000, "64x64 8"), (3, 5, 70, "64x64 1")]


@pytest.fixture(scope="module")
def raw():
    import __graft_entry__
    return __graft_entry__.load_gpt().raw()


def call(raw, name, signature, M, N, K, *tensors):
    scratch = raw["_ZN5tcamd3gpt15product_scratchEiii"]
    scratch.restype = ctypes.c_size_t
    n = scratch(M, N, K)
    buf = torch.full((max(n, 1),), float("nan"), device="cuda:0")
    f = raw[f"_ZN5tcamd3gpt{len(name)}{name}Eiii{signature}P12ihipStream_t"]
    f.restype = None
    ptr = lambda t: ctypes.c_void_p(t.data_ptr())
    f(M, N, K, *(ptr(t) for t in tensors), ptr(buf),
      ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    torch.cuda.synchronize()


def check(got, want, mag, K, slices):
    # as the product alone (test_gpu_gemm_planes.py), a rounding for each slice, and a few for what
    # follows, relative to the terms of the result
    lim = (6 * (K // 16 + 1) + slices + 12) * 2.0 ** -23 * mag
    bad = (got.double() - want).abs() > lim
    assert not bool(bad.any()), f"{int(bad.sum())} of {bad.numel()} outputs"


def gelu(x):
    return 0.5 * x * (1.0 + torch.tanh(math.sqrt(2.0 / math.pi) * (x + 0.044715 * x ** 3)))


@pytest.mark.parametrize("M,N,K,plan", SIZES)
def test_products(raw, M, N, K, plan):
    assert sched("tile", M, N, 1, K, 16, 1) == plan
    slices = int(plan.split()[1])
    g = torch.Generator(device="cuda:0").manual_seed(M + N + K)
    r = lambda *n: torch.randn(n, generator=g, device="cuda:0")
    nan = lambda *n: torch.full(n, float("nan"), device="cuda:0")
    A, W, bias, other = r(M, K), r(K, N) / math.sqrt(K), r(N), r(M, N)
    sums = torch.matmul(A.double(), W.double())
    mag = torch.matmul(A.double().abs(), W.double().abs())
    mn, f = nan(M, N), "PKfS2_"
    call(raw, "product_nn", f + "PfS3_", M, N, K, A, W, mn)
    check(mn, sums, mag, K, slices)
    mn = nan(M, N)
    call(raw, "product_nn_bias", f + "S2_PfS3_", M, N, K, A, W, bias, mn)
    pre = sums + bias.double()
    check(mn, pre, mag + bias.double().abs(), K, slices)
    mn = nan(M, N)
    call(raw, "product_nn_bias_residual", f + "S2_S2_PfS3_", M, N, K, A, W, bias, other, mn)
    check(mn, pre + other.double(), mag + bias.double().abs() + other.double().abs(), K, slices)
    mn, act = nan(M, N), nan(M, N)
    call(raw, "product_nn_bias_gelu", f + "S2_PfS3_S3_", M, N, K, A, W, bias, mn, act)
    check(mn, pre, mag + bias.double().abs(), K, slices)
    # |gelu'| <= 1.13
    check(act, gelu(pre), 1.2 * (mag + bias.double().abs()), K, slices)
    Wt = W.t().contiguous()
    mn = nan(M, N)
    call(raw, "product_nt", f + "PfS3_", M, N, K, A, Wt, mn)
    check(mn, sums, mag, K, slices)
    mn = nan(M, N)
    call(raw, "product_nt_gelu_backward", f + "S2_PfS3_", M, N, K, A, Wt, other, mn)
    x = other.double().requires_grad_(True)
    slope, = torch.autograd.grad(gelu(x).sum(), x)
    check(mn, sums * slope, 1.2 * mag, K, slices)
    At = A.t().contiguous()
    mn = nan(M, N)
    call(raw, "product_tn", f + "PfS3_", M, N, K, At, W, mn)
    check(mn, sums, mag, K, slices)
    both = nan(M + 1, N)
    call(raw, "product_tn_bias", f + "PfS3_", M, N, K, At, W, both)
    check(both[:M], sums, mag, K, slices)
    # column sums: a tree of eight, a chain over the chunks and the slices
    cols = W.double()
    check(both[M], cols.sum(0), cols.abs().sum(0), K, slices)
