"""Projections whose K goes in four slices when they come alone and in two pairs of slices when three come as one call: the same bits, whichever
way they come; the workgroups, read from captured launches, say that both ways are taken.  65 to 128 rows, the edges of
the 128-row tile among them, slices of several lengths."""
import ctypes as C

import pytest
import torch

from tests.test_gpu_gemm_dispatch import launches, stream  # noqa: F401

pytestmark = pytest.mark.gpu
D, ROWS = 128, 3


@pytest.mark.parametrize("layout", [1, 2])
@pytest.mark.parametrize("M,K", [(80, 12288), (97, 12288), (128, 12288), (100, 9216), (106, 12288 + 512)])
def test_alone_and_together(dev, stream, layout, M, K):  # noqa: F811
    N = 6144
    gen = torch.Generator(device="cuda")
    gen.manual_seed(M + K)
    X = torch.randn(M, K, device="cuda", generator=gen, dtype=torch.float16)
    W = [torch.randn(N, K, device="cuda", generator=gen, dtype=torch.float16) * 0.05 for _ in range(3)]
    bias = [torch.randn(N, device="cuda", generator=gen, dtype=torch.float16) for _ in range(3)]
    if layout == 2:
        stored = [torch.empty_like(w) for w in W]
        for s, w in zip(stored, W):
            dev.call("lg_weight_tile_f16", s, w, N, K, 1, K)
    else:
        stored = W
    alone, together = (torch.zeros(3, M, N // D, ROWS, D, device="cuda", dtype=torch.float16) for _ in range(2))
    dev.sync()
    for i in range(3):
        assert launches(dev, stream, "lg_gemm_fused_f16", layout, N, M, K, stored[i], K, X, K, alone[i], ROWS, dev.capi.EPI_BIAS_HEADS, bias[i], 1, D, N // D)[0] % 4 == 0
    p = lambda ts: (C.c_void_p * 3)(*[t.data_ptr() for t in ts])
    got = launches(dev, stream, "lg_gemm_fused_grouped_f16", layout, N, M, K, 3, p(stored), K, X, K, p(together), (C.c_int * 3)(ROWS, ROWS, ROWS),
                   dev.capi.EPI_BIAS_HEADS, p(bias), 1, D, N // D, replays=2)
    assert got == [2 * 3 * N // 192]
    assert torch.equal(alone, together)
    ref = X.float() @ W[1].float().T + bias[1].float()
    mag = X.float().abs() @ W[1].float().abs().T + bias[1].float().abs()
    y = together[1, :, :, 0].reshape(M, N).float()
    assert bool(((y - ref).abs() <= 2.0 ** -11 * ref.abs() + 2 * K * 2.0 ** -23 * mag + 2.0 ** -25).all())
    assert bool((together[:, :, :, 1:] == 0).all())
