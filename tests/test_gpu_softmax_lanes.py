"""Softmax where the lanes that hold a row change (8, 16, 32 and 64 vectors of 16 bytes) and workgroups end inside a head: rows on both
sides of each bound, masks that differ by batch and row.  Against 64-bit sums; the tolerance is that of tests/test_gpu_softmax_rows.py:
an exponent of magnitude up to 16 carries 2^-24 of itself three times, the quotient twice that (6e-6), and fp16 its rounding, 2^-11 and
2^-25 below the normal range."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,vector", [(torch.float32, 4), (torch.float16, 8)])
@pytest.mark.parametrize("vectors", [1, 8, 16, 32, 64])
@pytest.mark.parametrize("more", [-1, 0, 1])
def test_softmax_at_the_lane_bounds(dev, dtype, vector, vectors, more):
    seq, batch, heads, f16 = vectors * vector + more, 2, 3, dtype == torch.float16
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seq)
    n = batch * heads * seq * seq
    flat = torch.randn(n + 8, device="cuda", generator=gen, dtype=dtype) * 4
    qk = flat[:n].view(batch, heads, seq, seq)
    mask = (torch.rand(batch, 1, seq, seq, device="cuda", generator=gen) < 0.7).to(dtype)
    mask[..., 0] = 1
    behind = flat[n:].clone()
    t = qk.double() * 0.5 + (1 - mask.double()) * -10000
    e = torch.exp(t - t.amax(-1, keepdim=True))
    ref = e / (e.sum(-1, keepdim=True) + 1e-6)
    dev.call("lg_attn_softmax_f16" if f16 else "lg_attn_softmax_f32", qk.data_ptr(), mask.data_ptr(), batch, seq, heads, 0.5)
    dev.sync()
    bound = (6e-6 + (2.0 ** -11 if f16 else 0.0)) * ref + (2.0 ** -25 if f16 else 1e-30)
    assert bool(((qk.double() - ref).abs() <= bound).all())
    assert torch.equal(flat[n:], behind)
