"""LayerNorm rows on both sides of what a thread holds (one vector to eight), of 256 and of 512 threads, and beyond the vector kernel.  Against
64-bit sums.  A thread adds at most 64 numbers one after the other and ten steps follow, so the mean is off by at most 80 roundings (2^-24) of
the mean magnitude (times 1 / deviation, here below 2); variance, root and products by at most 2^-18 of the normalised value; fp16 outputs are rounded once."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,n", [(torch.float16, n) for n in (4088, 4096, 4104, 8192, 8200, 12288, 12296, 16384, 24584, 32768, 32776)] +
                         [(torch.float32, n) for n in (2048, 2052, 4100, 8196, 16384, 16388)])
@pytest.mark.parametrize("m", [1, 3])
def test_rows_of_any_length(dev, dtype, n, m):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(n)
    x = torch.randn(m, n, device="cuda", generator=gen, dtype=dtype) + 0.5
    g, b = (torch.randn(n, device="cuda", generator=gen, dtype=dtype) for _ in range(2))
    y = torch.empty_like(x)
    dev.call("lg_layer_norm_" + ("f16", "f32")[dtype == torch.float32], x, g, b, y, m, n)
    dev.sync()
    d = x.double() - x.double().mean(1, keepdim=True)
    ref = d / torch.sqrt((d * d).mean(1, keepdim=True) + 1e-6) * g.double() + b.double()
    bound = g.double().abs() * 80 * 2.0 ** -24 * x.double().abs().mean(1, keepdim=True) * 2 + 2.0 ** -18 * (ref - b.double()).abs() + 2.0 ** -23 * ref.abs()
    if dtype == torch.float16:
        bound += 2.0 ** -11 * ref.abs() + 2.0 ** -25
    assert bool(((y.double() - ref).abs() <= bound).all())
