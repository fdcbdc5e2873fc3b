"""Decode attention whose keys are split over more blocks than the merge kernel takes partials of at once, and over a number that leaves some of
a group empty; one split holds the largest scores by far.  Against torch in 64 bits, element by element: the probabilities are fp32, the
output is rounded once to fp16."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("heads,d,length", [(3, 128, 300), (2, 128, 1100), (1, 64, 2100), (5, 128, 2100), (1, 96, 4300), (2, 128, 8200)])
def test_many_splits(dev, heads, d, length):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(length)
    rows = length + 3
    q = torch.randn(1, heads, d, device="cuda", generator=gen, dtype=torch.float16)
    k, v = (torch.randn(1, heads, rows, d, device="cuda", generator=gen, dtype=torch.float16) for _ in range(2))
    k[0, :, length // 3] = 3 * q[0]
    out = torch.empty(1, heads, d, device="cuda", dtype=torch.float16)
    ws = torch.full((2048 * (2 + d),), float("nan"), device="cuda")     # what no split has written must not be used
    scalar = 1 / math.sqrt(d)
    dev.call("lg_attn_decode_f16", q, k, v, out, ws, 1, heads, d, length, rows, scalar)
    dev.sync()
    s = (k[0, :, :length].double() @ q[0].double().unsqueeze(2)).squeeze(2) * float(torch.tensor(scalar, dtype=torch.float16))
    p = torch.softmax(s, 1)
    ref, mag = ((p.unsqueeze(1) @ x).squeeze(1) for x in (v[0, :, :length].double(), v[0, :, :length].double().abs()))
    assert bool(((out[0].double() - ref).abs() <= 2.0 ** -11 * ref.abs() + 2e-5 * mag + 2.0 ** -25).all())
