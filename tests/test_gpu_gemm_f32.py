"""fp32 GEMM (gemm_f32.hpp and the 128 x 128 tiles of gemm.hip): edges of the tiles, remainders of k, matrices inside wider ones, unaligned
pointers, batches.  Tolerance: the products are exact in the fp32 unit up to one rounding each, so the error of a sum of K terms is at
most K 2^-24 of the sum of magnitudes; measured against that bound element by element."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

EPS = 2.0 ** -24


def _case(dev, transa, M, N, K, batch=1, pad=0, shift=0, seed=0):
    """Y [batch, M, N] inside a larger buffer: rows of N + pad, everything `shift` floats past a 16-byte boundary"""
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    rows, cols = (K, N) if transa == 0 else (N, K)

    def matrix(r, c):
        ld = c + pad
        flat = torch.randn(shift + batch * r * ld + 8, device="cuda", generator=gen)
        return flat, flat[shift:shift + batch * r * ld].view(batch, r, ld)[:, :, :c], ld

    fx, X, ldx = matrix(M, K)
    fw, W, ldw = matrix(rows, cols)
    fy, Y, ldy = matrix(M, N)
    before = fy.clone()
    Wk = W if transa == 0 else W.transpose(1, 2)
    ref = torch.stack([X[b].double().cpu() @ Wk[b].double().cpu() for b in range(batch)])
    mag = torch.stack([X[b].double().abs().cpu() @ Wk[b].double().abs().cpu() for b in range(batch)])
    dev.call("lg_gemm_strided_batched_f32", transa, 0, N, M, K, W.data_ptr(), ldw, rows * ldw, X.data_ptr(), ldx, M * ldx, Y.data_ptr(), ldy, M * ldy, batch)
    dev.sync()
    assert bool(((Y.double().cpu() - ref).abs() <= K * EPS * mag).all())
    first = Y.clone()
    Y.copy_(before[shift:shift + batch * M * ldy].view(batch, M, ldy)[:, :, :N])
    assert torch.equal(fy, before)          # nothing outside the output was written
    return first, X, W


@pytest.mark.parametrize("transa", [0, 1])
@pytest.mark.parametrize("M,N,K", [(1, 1, 1), (3, 5, 7), (16, 16, 16), (17, 15, 15), (15, 33, 64), (31, 31, 65), (64, 64, 63), (65, 66, 130), (64, 256, 1024),
                                   (100, 257, 33), (127, 513, 200), (129, 130, 31), (200, 1000, 96), (333, 333, 64), (333, 1024, 512), (800, 1024, 128),
                                   (1024, 2050, 64), (2048, 2048, 48), (512, 8200, 40)])
def test_shapes(dev, transa, M, N, K):
    _case(dev, transa, M, N, K)


@pytest.mark.parametrize("transa", [0, 1])
@pytest.mark.parametrize("M,N,K,batch,pad,shift", [(33, 47, 50, 1, 3, 1), (70, 66, 100, 3, 1, 0), (200, 200, 64, 16, 0, 0), (200, 64, 200, 16, 0, 2), (333, 64, 333, 4, 0, 0),
                                                   (130, 260, 128, 2, 4, 0), (512, 512, 64, 40, 0, 0), (1000, 1030, 72, 4, 2, 3)])
def test_strides_and_batches(dev, transa, M, N, K, batch, pad, shift):
    _case(dev, transa, M, N, K, batch, pad, shift)


def test_infinities_stay_in_their_rows(dev):
    """Rows and k beyond the matrix are not multiplied in: an infinity in one token row leaves the others finite."""
    M, N, K = 50, 70, 37
    X, W, Y = torch.randn(M, K, device="cuda"), torch.randn(K, N, device="cuda"), torch.empty(M, N, device="cuda")
    X[49, 36] = float("inf")
    dev.call("lg_gemm_f32", 0, 0, N, M, K, W.data_ptr(), N, X.data_ptr(), K, Y.data_ptr(), N)
    dev.sync()
    assert bool(torch.isfinite(Y[:49]).all()) and not bool(torch.isfinite(Y[49]).any())


# shapes whose parts take smaller tiles than the whole, in both kernels; K with whole quarters, with a remainder and with fewer chunks than quarters
@pytest.mark.parametrize("transa", [0, 1])
@pytest.mark.parametrize("M,N,K", [(800, 4096, 1024), (1600, 1024, 1000), (1000, 4100, 333), (2048, 2048, 40), (1300, 2050, 17)])
def test_a_row_does_not_depend_on_its_call(dev, transa, M, N, K):
    """Rows and features of a decomposed call have the bits of the whole: every tile of both kernels sums in the same order."""
    gen = torch.Generator(device="cuda")
    gen.manual_seed(1)
    X = torch.randn(M, K, device="cuda", generator=gen)
    W = torch.randn(*((K, N) if transa == 0 else (N, K)), device="cuda", generator=gen)
    ldw = W.shape[1]

    def gemm(m0, m, n0, n):
        Y = torch.empty(m, n, device="cuda")
        dev.call("lg_gemm_f32", transa, 0, n, m, K, W.data_ptr() + 4 * n0 * (1 if transa == 0 else K), ldw, X.data_ptr() + 4 * m0 * K, K, Y.data_ptr(), n)
        dev.sync()
        return Y

    torch.cuda.synchronize()
    whole = gemm(0, M, 0, N)
    for m0, m in ((0, M // 2), (M // 2, M - M // 2), (M - 200, 200), (3, 64), (5, 1)):
        assert torch.equal(gemm(m0, m, 0, N), whole[m0:m0 + m])
    for n0, n in ((0, N // 4), (N // 4, N - N // 4), (N - 130, 130), (7, 16)):
        assert torch.equal(gemm(0, M, n0, n), whole[:, n0:n0 + n])


# K of the bf16 kernels (256 and more, whole chunks of 32; fewer chunks than slices, slices of unequal length), every tile, its edges, and
# operands that only the unaligned path takes
@pytest.mark.parametrize("transa", [0, 1])
@pytest.mark.parametrize("M,N,K,batch,pad,shift", [(1, 1, 256, 1, 0, 0), (17, 20, 256, 1, 0, 0), (15, 33, 288, 1, 0, 0), (33, 66, 544, 1, 2, 1), (64, 256, 1024, 1, 0, 0),
                                                   (65, 260, 320, 3, 0, 0), (200, 1001, 512, 1, 3, 0), (200, 1004, 512, 1, 0, 0), (800, 1024, 256, 1, 0, 0),
                                                   (1000, 2050, 320, 1, 0, 2), (1030, 4100, 288, 1, 0, 0), (333, 64, 352, 40, 0, 0)])
def test_split_products(dev, transa, M, N, K, batch, pad, shift):
    _case(dev, transa, M, N, K, batch, pad, shift)


@pytest.mark.parametrize("transa", [0, 1])
@pytest.mark.parametrize("M,N,K", [(40, 70, 512), (300, 1024, 256), (1100, 2048, 256)])
def test_split_of_what_bf16_does_not_hold(dev, transa, M, N, K):
    """Infinities, NaN, the largest numbers, sums that overflow and rows of tiny numbers come out as from fp32 products; what else shares a
    tile with them keeps its accuracy."""
    gen = torch.Generator(device="cuda")
    gen.manual_seed(2)
    X, W, Y = torch.randn(M, K, device="cuda", generator=gen), torch.randn(K, N, device="cuda", generator=gen), torch.empty(M, N, device="cuda")
    X[0, 5], X[1, 7], X[2, 9] = float("inf"), float("nan"), -float("inf")
    W[5] = torch.where(W[5].abs() < 0.25, torch.ones_like(W[5]), W[5])     # an infinity times a number, times one (exact in hi), never times 0
    X[3] = 0.0
    X[3, 11] = 3.4e38                                                      # hi rounds to infinity
    W[11] = W[11].clamp(-1.0, 1.0)
    X[4], X[5] = 2.0 ** 120 * X[4].abs() + 2.0 ** 120, X[5] * 2.0 ** -118  # overflows where a column sums up; below the smallest bf16 in lo
    W[:, 0] = W[:, 0].abs() + 2.0 ** 7
    W[:, 1] *= 2.0 ** -116
    Wd = W if transa == 0 else W.t().contiguous()
    dev.call("lg_gemm_f32", transa, 0, N, M, K, Wd.data_ptr(), N if transa == 0 else K, X.data_ptr(), K, Y.data_ptr(), N)
    dev.sync()
    ref, mag = X.double().cpu() @ W.double().cpu(), X.double().abs().cpu() @ W.double().abs().cpu()
    got = Y.double().cpu()
    assert torch.equal(got[0], ref[0]) and bool(torch.isnan(got[1]).all()) and torch.equal(got[2], ref[2])     # infinities with their signs
    assert float(ref[4, 0]) > 3.5e38 and float(got[4, 0]) == float("inf")
    inside = (ref.abs() < 3.4e38) & (mag < 3.4e38)
    tiny = K * 2.0 ** -149                                                  # products below the smallest fp32 number
    assert bool(((got - ref).abs() <= K * EPS * mag + tiny)[inside].all())


@pytest.mark.parametrize("transa", [0, 1])
@pytest.mark.parametrize("M,N,K", [(4096, 1024, 256), (1600, 4096, 320), (800, 1024, 1024)])
def test_a_row_of_a_split_product_does_not_depend_on_its_call(dev, transa, M, N, K):
    test_a_row_does_not_depend_on_its_call(dev, transa, M, N, K)


@pytest.mark.parametrize("M,N", [(64, 16384), (33, 512)])
def test_rows_far_apart(dev, M, N):
    """Rows further apart than 32-bit offsets within a tile reach: the same bits as rows next to each other."""
    K, ld = 256, (1 << 27) + 4
    gen = torch.Generator(device="cuda")
    gen.manual_seed(3)
    X, W = torch.randn(M, K, device="cuda", generator=gen), torch.randn(K, N, device="cuda", generator=gen)
    far = torch.empty((M - 1) * ld + K, device="cuda").as_strided((M, K), (ld, 1))
    far.copy_(X)
    near, got = torch.empty(M, N, device="cuda"), torch.empty(M, N, device="cuda")
    torch.cuda.synchronize()
    dev.call("lg_gemm_f32", 0, 0, N, M, K, W.data_ptr(), N, X.data_ptr(), K, near.data_ptr(), N)
    dev.call("lg_gemm_f32", 0, 0, N, M, K, W.data_ptr(), N, far.data_ptr(), ld, got.data_ptr(), N)
    dev.sync()
    assert torch.equal(near, got)


def _gemm(dev, transa, X, W, m0=0, m=None, n0=0, n=None):
    """Rows m0 .. and features n0 .. of X [M, K] times W ([K, N], or [N, K] if transa)"""
    K = X.shape[1]
    m, n = m or X.shape[0] - m0, n or W.shape[0 if transa else 1] - n0
    Y = torch.empty(m, n, device="cuda")
    torch.cuda.synchronize()
    dev.call("lg_gemm_f32", transa, 0, n, m, K, W.data_ptr() + 4 * n0 * (K if transa else 1), W.shape[1], X.data_ptr() + 4 * m0 * K, K, Y.data_ptr(), n)
    dev.sync()
    return Y


def _same(a, b):
    return bool(((a == b) | (a.isnan() & b.isnan())).all())


# small tiles, 64 x 64 and 128 x 128 ones, whose slices are 1, 2 and 4 chunks
@pytest.mark.parametrize("transa", [0, 1])
@pytest.mark.parametrize("M,N,K", [(40, 72, 256), (300, 1024, 512), (4096, 1024, 256), (1100, 4096, 1024)])
def test_bits_of_an_output_depend_on_its_row_and_column_alone(dev, transa, M, N, K):
    """Rows and features that the bf16 parts do not hold (infinities, NaN, large numbers, sums that overflow) leave their tile's other outputs
    alone, and a row with a slice of tiny numbers has the bits of a call of its own."""
    gen = torch.Generator(device="cuda")
    gen.manual_seed(4)
    X, W = torch.randn(M, K, device="cuda", generator=gen), torch.randn(*((N, K) if transa else (K, N)), device="cuda", generator=gen)
    X[1, :32] *= 2.0 ** -90         # one slice of tiny numbers, or a part of one, in an ordinary row
    X[2, 32:40] *= 2.0 ** -120
    plain = _gemm(dev, transa, X, W)
    for r in range(4):
        assert _same(_gemm(dev, transa, X, W, r, 1), plain[r:r + 1])
        assert _same(_gemm(dev, transa, X, W, r, 33), plain[r:r + 33])
    bad, col = X.clone(), W.clone()
    bad[5, 3], bad[7, 4], bad[8, 5], bad[9] = float("inf"), float("nan"), 3.0e38, bad[9] * 2.0 ** 120
    bad[M - 1] *= 2.0 ** -100
    (col[6] if transa else col[:, 6])[:] *= 2.0 ** 110
    got = _gemm(dev, transa, bad, col)
    rows, cols = torch.ones(M, dtype=torch.bool, device="cuda"), torch.ones(N, dtype=torch.bool, device="cuda")
    rows[[5, 7, 8, 9, M - 1]], cols[6] = False, False
    assert _same(got[rows][:, cols], plain[rows][:, cols])
    for r in (5, 8, 9, M - 1):
        assert _same(_gemm(dev, transa, bad, col, r, 1), got[r:r + 1])
    assert _same(_gemm(dev, transa, bad, col, 10, 30, 0, 17), got[10:40, :17])


# every tile of operands that go through registers: 16 x 16 up to 128 x 128, with and without rows and features beyond the matrix
@pytest.mark.parametrize("transa", [0, 1])
@pytest.mark.parametrize("M,N,K", [(8, 72, 256), (64, 1000, 288), (200, 1030, 256), (333, 1024, 1024), (801, 1030, 512), (800, 1024, 1024), (1100, 1026, 1024),
                                   (3000, 2048, 288)])
def test_unaligned_rows_have_the_bits_of_aligned_ones(dev, transa, M, N, K):
    _, X, W = _case(dev, transa, M, N, K, pad=1, shift=1)
    odd = torch.empty(M, N, device="cuda")
    dev.call("lg_gemm_f32", transa, 0, N, M, K, W.data_ptr(), W.stride(1), X.data_ptr(), X.stride(1), odd.data_ptr(), N)
    pad = -W.shape[2] % 4
    aligned = torch.zeros(W.shape[1], W.shape[2] + pad, device="cuda")
    aligned[:, :W.shape[2]] = W[0]
    Y, x = torch.empty(M, N + -N % 4, device="cuda"), X[0].contiguous()
    torch.cuda.synchronize()
    dev.call("lg_gemm_f32", transa, 0, N, M, K, aligned.data_ptr(), aligned.shape[1], x.data_ptr(), K, Y.data_ptr(), Y.shape[1])
    dev.sync()
    assert torch.equal(odd, Y[:, :N])


@pytest.mark.parametrize("transa", [0, 1])
@pytest.mark.parametrize("M,N", [(48, 80), (1100, 2048)])
def test_tiny_elements_beside_ordinary_ones(dev, transa, M, N):
    """One element of each row is 2^e times an ordinary one and all that a feature, which is zero elsewhere, sees.  The sum
    rounds its partial products, of which one or two are of the size of the whole: 2^-23 each at most."""
    K = 256
    gen = torch.Generator(device="cuda")
    gen.manual_seed(5)
    for e in (-100, -112, -118, -124, -140):
        for w in (1.0, 2.0 ** min(-e, 125)):
            X, W = torch.ones(M, K, device="cuda"), torch.zeros(K, N, device="cuda")
            X[:, 77] = (1 + torch.rand(M, device="cuda", generator=gen)) * 2.0 ** e
            W[77] = (1 + torch.rand(N, device="cuda", generator=gen)) * w
            ref = X.double() @ W.double()
            for x, y, r in ((X, W, ref), (W.t().contiguous(), X.t().contiguous(), ref.t())):      # as token rows, and as features
                got = _gemm(dev, transa, x, y.t().contiguous() if transa else y).double()
                assert bool(((got - r).abs() <= 4 * EPS * r.abs() + 2.0 ** -149).all()), (e, w)


@pytest.mark.parametrize("transa", [0, 1])
@pytest.mark.parametrize("M,N,K", [(256, 256, 256), (256, 512, 1024), (1024, 2048, 1024), (256, 256, 4096)])
def test_sparse_rows(dev, transa, M, N, K):
    """Rows of few nonzeros: no further from 64-bit sums (5 %: eight slices meet instead of four) than the same products summed in fp32 by quarters
    of K, as the fp32 unit's kernels do, and a single one correct to a rounding (and a 16th: the small products are 2^-8 of the whole and
    round seven times)."""
    gen = torch.Generator(device="cuda")
    gen.manual_seed(6)
    for nonzeros in (1, 2, 3, 8, 32):
        at = torch.rand(M, K, device="cuda", generator=gen).argsort(1)[:, :nonzeros].sort(1).values
        x, W = torch.randn(M, nonzeros, device="cuda", generator=gen), torch.randn(K, N, device="cuda", generator=gen)
        X = torch.zeros(M, K, device="cuda").scatter_(1, at, x)
        ref, quarters = X.double() @ W.double(), torch.zeros(4, M, N, device="cuda")
        for j in range(nonzeros):
            product = x[:, j:j + 1].double() * W[at[:, j]].double()
            for q in range(4):
                quarters[q] = torch.where((at[:, j] * 4 // K == q)[:, None], (quarters[q].double() + product).float(), quarters[q])
        fp32 = (quarters[0] + quarters[1] + quarters[2] + quarters[3]).double()
        got = _gemm(dev, transa, X, W.t().contiguous() if transa else W).double()
        assert float((got - ref).norm()) <= 1.05 * float((fp32 - ref).norm()), nonzeros
        if nonzeros == 1:
            assert bool(((got - ref).abs() <= (1 + 2.0 ** -4) * EPS * ref.abs()).all())
