"""The two ways in which the LayerNorm kernels load gamma and beta (few rows, many rows) give a row the same bits, for rows that fill
their workgroup's vectors and rows that do not (tests/test_gpu_kernels.py compares few rows with the oracle)."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
@pytest.mark.parametrize("n", [8, 256, 1032, 4096, 12288, 16392])
def test_row_count_does_not_change_a_row(dev, dtype, n):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(n)
    suffix, many = ("f16", "f32")[dtype == torch.float32], 2 * torch.cuda.get_device_properties(0).multi_processor_count + 1
    x, add = (torch.randn(many, n, device="cuda", generator=gen, dtype=dtype) for _ in range(2))
    g, b, bias = (torch.randn(n, device="cuda", generator=gen, dtype=dtype) for _ in range(3))

    def all_modes(m):
        y, inplace, total, norm = torch.empty_like(x[:m]), x[:m].clone(), add[:m].clone(), torch.empty_like(x[:m])
        dev.call("lg_layer_norm_" + suffix, x, g, b, y, m, n)
        dev.call("lg_add_bias_input_layernorm_" + suffix, inplace, add, bias, g, b, m, n)
        dev.call("lg_add_bias_input_layernorm_2_" + suffix, x, g, b, bias, total, norm, m, n)
        dev.sync()
        return y, inplace, total, norm

    for few, whole in zip(all_modes(3), all_modes(many)):
        assert torch.equal(few, whole[:3])
