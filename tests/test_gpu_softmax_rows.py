"""Softmax over rows of any length and alignment: shorter than a vector, on both sides of whole vectors and of 64, 128, 256 and 512 of
them, buffers an odd number of elements past a 16-byte boundary.  Against 64-bit sums.  Tolerance: an exponent t - max of magnitude up
to 16 carries 2^-24 of itself from each of scaling, subtraction and conversion to base 2, so exp is off by at most 3 x 16 x 2^-24 and the
quotient by twice that (6e-6); fp16 adds its rounding, 2^-11 and 2^-25 below the normal range."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
@pytest.mark.parametrize("seq,shift", [(1, 0), (3, 1), (7, 0), (8, 3), (9, 0), (53, 0), (200, 1), (255, 0), (257, 0), (333, 0), (511, 1), (513, 0), (777, 5), (1025, 0),
                                       (2047, 0), (2049, 0), (4095, 0), (4097, 0)])
def test_softmax_of_any_row(dev, dtype, seq, shift):
    batch, heads = (2, 3) if seq < 300 else (1, 2)
    rows = 5 if seq > 1000 else seq     # the entry takes square scores: only the first rows of long ones are compared
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seq)
    n, f16 = batch * heads * seq * seq, dtype == torch.float16
    flat = torch.randn(shift + n + 9, device="cuda", generator=gen, dtype=dtype) * 4
    mflat = (torch.rand(shift + batch * seq * seq, device="cuda", generator=gen) < 0.7).to(dtype)
    qk, mask = flat[shift:shift + n].view(batch, heads, seq, seq), mflat[shift:].view(batch, 1, seq, seq)
    mask[..., 0] = 1
    before = flat.clone()
    scalar = 0.5
    t = qk[:, :, :rows].double() * scalar + (1 - mask[:, :, :rows].double()) * -10000
    e = torch.exp(t - t.amax(-1, keepdim=True))
    ref = e / (e.sum(-1, keepdim=True) + 1e-6)
    dev.call("lg_attn_softmax_f16" if f16 else "lg_attn_softmax_f32", qk.data_ptr(), mask.data_ptr(), batch, seq, heads, scalar)
    dev.sync()
    bound = (6e-6 + (2.0 ** -11 if f16 else 0.0)) * ref + (2.0 ** -25 if f16 else 1e-30)
    assert bool(((qk[:, :, :rows].double() - ref).abs() <= bound).all())
    assert torch.equal(flat[:shift], before[:shift]) and torch.equal(flat[shift + n:], before[shift + n:])
