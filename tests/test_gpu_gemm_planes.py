"""The strided-batched GEMM on the bf16 matrix cores (three planes per fp32 operand): every
tile shape and its remainders against fp64, K that ends inside a chunk, and operands with
infinities, NaN and values that round to infinity in bf16."""
import numpy as np
import pytest
import torch

from gpu_util import sched

pytestmark = pytest.mark.gpu


def product64(A, B, ta, tb):
    A, B = A.double(), B.double()
    A = A.transpose(1, 2).contiguous() if ta else A
    B = B.transpose(1, 2).contiguous() if tb else B
    return torch.matmul(A, B), torch.matmul(A.abs(), B.abs())


def run(lib, A, B, C, M, N, K, ta, tb, alpha=1.0, beta=0.0):
    lib.matmul_batched_strided(A, B, C, M, N, K, M * K, K * N, M * N, A.shape[0], ta, tb, alpha,
                               beta)
    torch.cuda.synchronize()


# (M, N, K, batch): 128 x 128 tiles (the first two sizes) and 64 x 64 ones, with ragged edges; K below, at and beyond the 16- and 32-deep chunks.  The
# other tiles: test_every_tile
@pytest.mark.parametrize("M,N,K,batch", [
    (2049, 2047, 33, 4), (1000, 1300, 47, 5), (900, 1100, 64, 4), (515, 701, 95, 4),
    (129, 65, 17, 3), (1, 1, 1, 1), (3, 130, 2, 2), (63, 64, 31, 7), (257, 2, 48, 2)])
@pytest.mark.parametrize("ta,tb", [(False, False), (False, True), (True, False), (True, True)])
def test_tiles_and_tails(lib, M, N, K, batch, ta, tb):
    g = torch.Generator(device="cuda:0").manual_seed(M + N + K)
    A = torch.randn((batch, K, M) if ta else (batch, M, K), generator=g, device="cuda:0")
    B = torch.randn((batch, N, K) if tb else (batch, K, N), generator=g, device="cuda:0")
    want, mag = product64(A, B, ta, tb)
    # one rounding per 16 products and plane product and the three products left out, each below
    # 2^-23 of the sum of magnitudes so far
    bound = (6 * (K // 16 + 1) + 2) * 2.0 ** -23 * mag
    for alpha, beta in ((1.0, 0.0), (0.5, -1.25)):
        C = torch.full((batch, M, N), float("nan"), device="cuda:0")
        if beta != 0.0:
            C = torch.randn((batch, M, N), generator=g, device="cuda:0")
        exp = alpha * want + (beta * C.double() if beta != 0.0 else 0.0)
        lim = abs(alpha) * bound + 2.0 ** -22 * exp.abs()
        if beta != 0.0:
            lim = lim + 2.0 ** -22 * (beta * C.double()).abs()
        run(lib, A, B, C, M, N, K, ta, tb, alpha, beta)
        assert bool(((C.double() - exp).abs() <= lim).all()), (alpha, beta)


@pytest.mark.parametrize("tile,M,N,K,batch", [
    ("256x256", 1023, 1021, 1000, 16), ("256x128", 1023, 509, 1501, 12),
    ("128x128", 1000, 1300, 47, 5), ("128x64", 1000, 500, 700, 8), ("64x64", 515, 701, 95, 4)])
@pytest.mark.parametrize("ta,tb", [(False, False), (False, True), (True, False), (True, True)])
def test_every_tile(lib, tile, M, N, K, batch, ta, tb):
    """Each tile shape with ragged rows, columns and K, at a size that the rule sends to it."""
    assert sched("tile", M, N, batch, K, 1, 1) == f"{tile} 1"
    g = torch.Generator(device="cuda:0").manual_seed(M + N + K)
    A = torch.randn((batch, K, M) if ta else (batch, M, K), generator=g, device="cuda:0")
    B = torch.randn((batch, N, K) if tb else (batch, K, N), generator=g, device="cuda:0")
    C = torch.full((batch, M, N), float("nan"), device="cuda:0")
    run(lib, A, B, C, M, N, K, ta, tb)
    want, mag = product64(A, B, ta, tb)
    # as test_tiles_and_tails
    assert bool(((C.double() - want).abs() <= (6 * (K // 16 + 1) + 3) * 2.0 ** -23 * mag).all())


@pytest.mark.parametrize("ta,tb", [(False, False), (False, True), (True, False)])
@pytest.mark.parametrize("beta", [0.0, 0.5])
def test_non_finite_operands(lib, ta, tb, beta):
    """Infinite, NaN and largest-magnitude elements: the same infinities and NaN as the fp32
    sum, the other outputs unaffected."""
    M, N, K = 150, 200, 70
    g = torch.Generator().manual_seed(5)
    A = torch.randn((M, K), generator=g)
    B = torch.randn((K, N), generator=g)
    C0 = torch.randn((M, N), generator=g)
    A[3, 5], A[7, 9], A[7, 11] = float("inf"), float("inf"), float("-inf")
    A[100, 69], A[20, 0] = float("nan"), -3.4028234663852886e38
    B[:, 31] = 0.0
    B[5, 40], B[6, 199] = 0.0, float("-inf")
    B[0, 50] = 1e-3
    want = (A[:, :, None] * B[None]).sum(1) + (beta * C0 if beta else 0.0)
    dev = lambda x, t: (x.t() if t else x).contiguous().cuda()[None]
    C = C0.cuda()[None].clone()
    run(lib, dev(A, ta), dev(B, tb), C, M, N, K, ta, tb, 1.0, beta)
    got = C[0].cpu()
    assert torch.equal(torch.isnan(got), torch.isnan(want))
    inf = torch.isinf(want)
    assert torch.equal(torch.isinf(got), inf) and torch.equal(got[inf], want[inf])
    fin = torch.isfinite(want)
    np.testing.assert_allclose(got[fin].numpy(), want[fin].numpy(), rtol=2e-5, atol=1e-4)


@pytest.mark.parametrize("ta,tb", [(False, False), (False, True), (True, False), (True, True)])
@pytest.mark.parametrize("M,N,K", [(150, 70, 515), (300, 260, 31), (64, 33, 16)])
def test_blocks_taken_again(lib, M, N, K, ta, tb):
    """Infinities in the last row, the last column and the last k (K with and without a remainder
    of 16), in batches that take every tile shape: the outputs beside them stay those of the fp32
    sum."""
    for batch in (1, 24):
        g = torch.Generator().manual_seed(M + batch)
        A = torch.randn((batch, M, K), generator=g)
        B = torch.randn((batch, K, N), generator=g)
        A[:, M - 1, K - 1] = float("inf")
        A[:, 3, 0] = float("-inf")
        B[:, K // 2, N - 1] = float("inf")
        # dense sums without the infinite terms; those rows and columns by their signs
        A0, B0 = A.clone(), B.clone()
        A0[torch.isinf(A0)] = 0.0
        B0[torch.isinf(B0)] = 0.0
        want, mag = product64(A0, B0, False, False)
        want[:, M - 1] = float("inf") * B[:, K - 1].sign().double()
        want[:, 3] = float("-inf") * B[:, 0].sign().double()
        col = want[:, :, N - 1]
        add = float("inf") * A[:, :, K // 2].sign().double()
        want[:, :, N - 1] = torch.where(torch.isinf(col), col + add, add)
        dev = lambda x, t: (x.transpose(1, 2) if t else x).contiguous().cuda()
        C = torch.empty((batch, M, N), device="cuda:0")
        run(lib, dev(A, ta), dev(B, tb), C, M, N, K, ta, tb)
        got = C.cpu().double()
        fin = torch.isfinite(want)
        assert torch.equal(torch.isnan(got), torch.isnan(want))
        assert torch.equal(got[torch.isinf(want)], want[torch.isinf(want)])
        # a rounding of 2^-23 of the magnitudes so far per k, whichever form a block takes
        lim = (K + 8) * 2.0 ** -23 * mag
        assert bool(((got - want).abs()[fin] <= lim[fin]).all())


def test_infinity_cost(lib):
    """An infinity in a row and in a column must not cost many times the product: their outputs are
    taken again by whole waves (2.9 times the product at 128 x 128 x 32768; a lane's serial sums of
    32768 terms took 77 times)."""
    M, N, K = 128, 128, 32768
    g = torch.Generator(device="cuda:0").manual_seed(1)
    A = torch.randn((1, M, K), generator=g, device="cuda:0")
    B = torch.randn((1, N, K), generator=g, device="cuda:0")
    C = torch.empty((1, M, N), device="cuda:0")

    def time_us():
        run(lib, A, B, C, M, N, K, False, True)
        e = [torch.cuda.Event(enable_timing=True) for _ in range(2)]
        best = float("inf")
        for _ in range(5):
            e[0].record()
            lib.matmul_batched_strided(A, B, C, M, N, K, M * K, K * N, M * N, 1, False, True, 1.0,
                                       0.0)
            e[1].record()
            torch.cuda.synchronize()
            best = min(best, e[0].elapsed_time(e[1]) * 1e3)
        return best

    plain = time_us()
    A[0, 7, 11] = B[0, 9, 12] = float("inf")
    again = time_us()
    print(f"{plain:.0f} us, with infinities {again:.0f} us")
    assert not bool(torch.isfinite(C[0, 7]).any()) and not bool(torch.isfinite(C[0, :, 9]).any())
    assert again < 8 * plain


@pytest.mark.parametrize("ta,tb", [(False, False), (False, True), (True, False), (True, True)])
@pytest.mark.parametrize("up,down", [(100, -125), (100, -115), (90, -100), (60, -60), (102, -102)])
def test_scaled_operands(lib, up, down, ta, tb):
    """Operands scaled by powers of two, which round nothing: the same bits as without, down to the
    smallest normal numbers and up to 2^103."""
    M, N, K = 70, 130, 100
    g = torch.Generator().manual_seed(2)
    draw = lambda *n: (1.0 + torch.rand(n, generator=g)) * (torch.randint(0, 2, n, generator=g) * 2 - 1)
    A, B = draw(1, M, K).cuda(), draw(1, K, N).cuda()
    dev = lambda x, t: (x.transpose(1, 2) if t else x).contiguous()
    C = [torch.empty((1, M, N), device="cuda:0") for _ in range(3)]
    run(lib, dev(A, ta), dev(B, tb), C[0], M, N, K, ta, tb)
    run(lib, dev(A * 2.0 ** up, ta), dev(B * 2.0 ** down, tb), C[1], M, N, K, ta, tb)
    run(lib, dev(A * 2.0 ** down, ta), dev(B * 2.0 ** up, tb), C[2], M, N, K, ta, tb)
    want = C[0] * 2.0 ** (up + down)
    assert torch.equal(C[1], want) and torch.equal(C[2], want)


@pytest.mark.parametrize("ta,tb", [(False, True), (True, False)])
@pytest.mark.parametrize("sa,sb", [
    (-149, 120), (-140, 126), (-135, 0), (-74, -73), (-126, -20),  # subnormal operands, results
    (104, -100), (126, -126), (120, 1), (45, 45), (63, 58)])       # beyond the planes' range
def test_operand_range(lib, sa, sb, ta, tb):
    """The ends of fp32's range, in operands and results."""
    M, N, K = 70, 66, 40
    g = torch.Generator().manual_seed(3)
    A = torch.ldexp(torch.rand((1, M, K), generator=g, dtype=torch.float64) + 0.5,
                    torch.tensor(sa)).float().double()
    B = torch.ldexp(torch.randn((1, K, N), generator=g, dtype=torch.float64) * 0.125,
                    torch.tensor(sb)).float().double()
    want, mag = product64(A, B, False, False)
    assert bool((mag < 2.0 ** 128).all())
    dev = lambda x, t: (x.transpose(1, 2) if t else x).contiguous().float().cuda()
    C = torch.empty((1, M, N), device="cuda:0")
    run(lib, dev(A, ta), dev(B, tb), C, M, N, K, ta, tb)
    # 2^-23 of the magnitudes so far for each of K roundings at most, and a subnormal result's last
    # bit for each
    lim = (K + 8) * (2.0 ** -23 * mag + 2.0 ** -149)
    assert bool(((C.cpu().double() - want).abs() <= lim).all())


@pytest.mark.parametrize("ta,tb", [(False, False), (False, True), (True, False), (True, True)])
@pytest.mark.parametrize("M,N,batch", [(1, 1, 1), (65, 130, 2), (300, 257, 30)])
def test_short_products(lib, M, N, batch, ta, tb):
    """One k: the rounded product itself; two and three: one rounding for each."""
    g = torch.Generator(device="cuda:0").manual_seed(4)
    for K in (1, 2, 3):
        A = torch.randn((batch, M, K), generator=g, device="cuda:0")
        B = torch.randn((batch, K, N), generator=g, device="cuda:0")
        dev = lambda x, t: (x.transpose(1, 2) if t else x).contiguous()
        for alpha, beta in ((1.0, 0.0), (1.0, 1.0)):
            C = torch.zeros((batch, M, N), device="cuda:0")
            run(lib, dev(A, ta), dev(B, tb), C, M, N, K, ta, tb, alpha, beta)
            want, mag = product64(A, B, False, False)
            if K == 1:
                assert torch.equal(C, A * B)
            assert bool(((C.double() - want).abs() <= K * 2.0 ** -24 * mag + 2.0 ** -149).all())


def test_more_tiles_than_one_launch_holds(lib):
    """9 437 184 products of 1 x 68 x 4: 2^24 and more 64 x 64 tiles."""
    n, N, K = 9 * 2 ** 20, 68, 4
    A = torch.arange(1.0, 5.0, device="cuda:0")
    B = torch.arange(float(K * N), device="cuda:0")
    C = torch.zeros(n * N, device="cuda:0")
    lib.matmul_batched_strided(A, B, C, 1, N, K, 0, 0, N, n, False, False, 1.0, 0.0)
    want = (A.cpu() @ B.cpu().view(K, N)).cuda()
    assert bool((C.view(n, N) == want).all())
