"""Dense float32 products of several rows: bit for bit what each row gives by itself."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bits,group", [(4, 32), (4, 64), (8, 64), (8, 128)])
@pytest.mark.parametrize("rows,n,k", [(2, 16, 128), (3, 50, 384), (8, 130, 640), (9, 200, 128), (17, 2048, 256), (61, 2306, 512), (6, 1030, 256)])
def test_rows_are_independent(rows, n, k, bits, group):
    """Remainders of rows and columns in a wave's tile, rows of fewer words than lanes; each tile of the rule: 2 x 1, 4 x 2 (8-bit at
    17 rows, 4-bit at 6), 4 x 4 and, with 4-bit codes at 61 rows, 8 x 4."""
    import mlx_rs_amd as m
    gen = torch.Generator(device="cuda").manual_seed(rows + n + bits)
    q, s, b = m.ops.quantize(torch.randn((n, k), generator=gen, device="cuda") * 0.02, group, bits, torch.float32)
    x = torch.randn((rows, k), generator=gen, device="cuda")
    x[rows - 1, 5] = float("inf")
    y = m.ops.quantized_linear(x, q, s, b, group_size=group, bits=bits)
    for i in range(rows):
        one = m.ops.quantized_linear(x[i:i + 1].contiguous(), q, s, b, group_size=group, bits=bits)
        assert torch.equal(y[i].view(torch.int32), one[0].view(torch.int32)), i
