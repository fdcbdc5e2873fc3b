"""fp16 GEMMs on the generic kernel with rows of any alignment: matrices inside wider ones, pointers an odd number of halves past a
16-byte boundary, sizes on both sides of a vector, a tile and a k-tile.  Tolerance, element by element: the products of halves are exact
in fp32, the sum of K of them is off by at most K 2^-23 of the sum of magnitudes in any order, and the result is rounded once to fp16
(2^-11 of it, 2^-25 below the normal range)."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("transa", [0, 1])
@pytest.mark.parametrize("M,N,K,batch,pad,shift", [(1, 1, 1, 3, 0, 1), (7, 9, 8, 2, 1, 3), (127, 129, 33, 1, 3, 0), (128, 128, 32, 2, 1, 1), (333, 333, 128, 6, 0, 0),
                                                   (333, 128, 333, 6, 0, 0), (65, 77, 41, 3, 2, 5), (130, 257, 100, 2, 4, 2), (53, 53, 96, 5, 0, 7), (200, 200, 64, 4, 0, 0)])
def test_any_alignment(dev, transa, M, N, K, batch, pad, shift):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(M + N)

    def matrix(r, c):
        ld = c + pad
        flat = torch.randn(shift + batch * r * ld + 8, device="cuda", generator=gen, dtype=torch.float16)
        return flat, flat[shift:shift + batch * r * ld].view(batch, r, ld)[:, :, :c], ld

    rows, cols = (K, N) if transa == 0 else (N, K)
    _, X, ldx = matrix(M, K)
    _, W, ldw = matrix(rows, cols)
    flat, Y, ldy = matrix(M, N)
    before = flat.clone()
    dev.call("lg_gemm_strided_batched_f16", transa, 0, N, M, K, W.data_ptr(), ldw, rows * ldw, X.data_ptr(), ldx, M * ldx, Y.data_ptr(), ldy, M * ldy, batch)
    dev.sync()
    x, w = X.double().cpu(), (W if transa == 0 else W.transpose(1, 2)).double().cpu()
    for b in range(batch):
        ref, mag = x[b] @ w[b], x[b].abs() @ w[b].abs()
        assert bool(((Y[b].double().cpu() - ref).abs() <= 2.0 ** -11 * ref.abs() + K * 2.0 ** -23 * mag + 2.0 ** -25).all())
    Y.copy_(before[shift:shift + batch * M * ldy].view(batch, M, ldy)[:, :, :N])
    assert torch.equal(flat, before)        # nothing outside the output was written
