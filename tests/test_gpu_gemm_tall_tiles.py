"""The 96-feature tiles of 160 to 256 token rows: edges of their rows (those of 160 and 224 rows do not hold a whole number of 16-byte chunks
for every thread), one k-tile, fewer and more than their rings hold, a last row of tiles with one token row.  The workgroups, read from a
captured launch, say that the tile is taken.  Tolerance, element by element: products of halves are exact in fp32, a sum of K of them is off by
at most K 2^-23 of the sum of magnitudes, and the result is rounded once to fp16."""
import pytest
import torch

from tests.test_gpu_gemm_dispatch import launches, stream  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("layout", [1, 2])
@pytest.mark.parametrize("M,N,K,rows", [(257, 12288, 64, 160), (319, 12288, 128, 160), (320, 9216, 512, 160), (384, 12288, 192, 192), (383, 12288, 1024, 192),
                                        (385, 12288, 256, 224), (448, 9216, 2048, 224), (500, 12288, 12288, 256), (512, 12288, 12288, 256)])
def test_tall_tiles(dev, stream, layout, M, N, K, rows):  # noqa: F811
    gen = torch.Generator(device="cuda")
    gen.manual_seed(M + K)
    X = torch.randn(M, K, device="cuda", generator=gen, dtype=torch.float16)
    W = torch.randn(N, K, device="cuda", generator=gen, dtype=torch.float16)
    stored = W
    if layout == 2:
        stored = torch.empty_like(W)
        dev.call("lg_weight_tile_f16", stored, W, N, K, 1, K)
    Y = torch.full((M + 1, N), 7.0, device="cuda", dtype=torch.float16)
    dev.sync()
    assert launches(dev, stream, "lg_gemm_f16", layout, 0, N, M, K, stored, K, X, K, Y, N) == [(M + rows - 1) // rows * (N // 96)]
    assert bool((Y[M] == 7.0).all())
    for n in range(0, N, 1536):
        w = W[n:n + 1536].double().T.contiguous()
        ref, mag = X.double() @ w, X.double().abs() @ w.abs()
        assert bool(((Y[:M, n:n + 1536].double() - ref).abs() <= 2.0 ** -11 * ref.abs() + K * 2.0 ** -23 * mag + 2.0 ** -25).all())
