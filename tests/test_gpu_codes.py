"""The tiled product on raw codes (quantized_linear in float16 and float32, and in bfloat16 with groups of 32 and 128)
at the edges of its tiles and of its sharing of K, against the float64 product of the dequantised matrix."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

# One rounding to the result's type, half a unit of 8 (bfloat16) or 11 (float16) significant bits, is at most 2^-8 or
# 2^-11 of each value, and so of the whole in the 2-norm (typically 0.4 of that).  float32: the sums run in
# float32 and the code and bias terms cancel to about an eighth, so 8 * 4 units of 2^-24.
BOUND = {"bfloat16": 2.0 ** -8, "float16": 2.0 ** -11, "float32": 32 * 2.0 ** -24}
SHAPES = [  # rows, N, K: one row; odd rows and columns; K of 3, 9 and 17 times 128 (uneven shares); each tile of the rule
    (1, 16, 128), (33, 37, 384), (65, 200, 1152), (31, 4100, 2176), (130, 1000, 256),
    (700, 1088, 640), (300, 4000, 384), (1100, 4112, 256),
]


def product(x, q, s, b, group, bits):
    per = 32 // bits
    shift = torch.arange(per, device=q.device) * bits
    codes = (((q.to(torch.int64) & 0xFFFFFFFF).unsqueeze(-1) >> shift) & ((1 << bits) - 1)).reshape(q.shape[0], -1).double()
    w = codes * s.double().repeat_interleave(group, 1) + b.double().repeat_interleave(group, 1)
    return x.double() @ w.t()


@pytest.mark.parametrize("dtype,group", [("float16", 32), ("float16", 64), ("float16", 128), ("bfloat16", 32), ("bfloat16", 128),
                                         ("float32", 32), ("float32", 64), ("float32", 128)])
@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("rows,n,k", SHAPES)
def test_products_on_raw_codes(rows, n, k, bits, dtype, group):
    import mlx_rs_amd as m
    dt = getattr(torch, dtype)
    gen = torch.Generator(device="cuda").manual_seed(rows + n + k)
    q, s, b = m.ops.quantize(torch.randn((n, k), generator=gen, device="cuda") * 0.02, group, bits, dt)
    x = torch.randn((rows, k), generator=gen, device="cuda").to(dt)
    lb = torch.randn(n, generator=gen, device="cuda").to(dt)
    ref = product(x, q, s, b, group, bits)
    y = m.ops.quantized_linear(x, q, s, b, group_size=group, bits=bits)
    assert y.dtype == dt and torch.isfinite(y).all()
    err = float((y.double() - ref).norm() / ref.norm())
    assert err <= BOUND[dtype], (err, BOUND[dtype])
    # the layer's bias: one more addition in the result's type, exactly
    yb = m.ops.quantized_linear(x, q, s, b, lb, group_size=group, bits=bits)
    assert torch.equal(yb, (y.float() + lb.float()).to(dt))
    # a batch's rows do not depend on how many there are beyond their own sums' order
    if rows > 1:
        one = m.ops.quantized_linear(x[:1].contiguous(), q, s, b, group_size=group, bits=bits)
        assert float((one.double() - ref[:1]).norm() / ref[:1].norm()) <= BOUND[dtype]


def test_large_float32_values_survive_the_split():
    """The three pieces are cut by truncation: the largest finite values do not overflow on the way."""
    import mlx_rs_amd as m
    x = torch.full((2, 128), np.finfo(np.float32).max / 1024, device="cuda")
    x[1] = 0
    w = torch.full((16, 128), 1.0, device="cuda")
    q, s, b = m.ops.quantize(w, 64, 4, torch.float32)
    y = m.ops.quantized_linear(x, q, s, b, group_size=64, bits=4)
    assert torch.allclose(y[0], (x[0].double().sum()).float().expand(16), rtol=1e-6) and (y[1] == 0).all()
