"""Dense float32 products of 64 rows and more on the float32 matrix instructions, against float64 and the plain sums of single rows."""
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def layer(rows, n, k, bits, group, seed=0):
    import mlx_rs_amd as m
    gen = torch.Generator(device="cuda").manual_seed(rows + n + bits + seed)
    q, s, b = m.ops.quantize(torch.randn((n, k), generator=gen, device="cuda") * 0.02, group, bits, torch.float32)
    x = torch.randn((rows, k), generator=gen, device="cuda")
    per = 32 // bits
    codes = (q.long().unsqueeze(-1) >> (bits * torch.arange(per, device="cuda")) & ((1 << bits) - 1)).reshape(n, k).double()
    w = codes * s.double().repeat_interleave(group, 1) + b.double().repeat_interleave(group, 1)
    return x, q, s, b, w, lambda v: m.ops.quantized_linear(v, q, s, b, group_size=group, bits=bits)


# rows and columns that fill no tile of each size of tile (32 x 32: one round of the chip of those; 64 x 32; 64 x 64), K of no multiple of eight runs of 32
@pytest.mark.parametrize("bits,group", [(4, 32), (4, 64), (8, 32), (8, 128)])
@pytest.mark.parametrize("rows,n,k", [(64, 2050, 1152), (65, 1040, 2304), (97, 2049, 1280), (600, 250, 1024), (1000, 145, 1152), (161, 901, 1152)])
def test_tiles_lose_no_more_than_plain_sums(rows, n, k, bits, group):
    """The bound is that of sums in float32, 2^-22 of the norm, as for the plain kernel; and no more than single rows lose, but for what the norm of the error of 64 n
    values varies by, a hundredth or so."""
    assert rows * n * k >= 150_000_000
    x, q, s, b, w, product = layer(rows, n, k, bits, group)
    y, ref = product(x), x.double() @ w.t()
    assert float((y.double() - ref).norm() / ref.norm()) <= 2.0 ** -22
    picked = list(range(0, rows, max(1, rows // 64)))[:64]
    alone = torch.cat([product(x[i:i + 1].contiguous()) for i in picked])
    err = [float((v.double() - ref[picked]).norm()) for v in (y[picked], alone)]
    assert err[0] <= 1.03 * err[1], err


def test_values_that_are_not_finite():
    x, q, s, b, w, product = layer(70, 2048, 1280, 4, 64)
    x[3, 7], x[69, 1279], x[5, 100] = float("inf"), float("-inf"), float("nan")
    s[9, 2] = float("inf")
    b[2047, 0] = float("-inf")
    y = product(x)
    alone = torch.cat([product(x[i:i + 1].contiguous()) for i in range(70)])
    assert torch.equal(y.isnan(), alone.isnan()) and torch.equal(y.isinf(), alone.isinf()) and torch.equal(y[y.isinf()], alone[y.isinf()])
    assert bool(y.isnan().any()) and bool(y.isinf().any())
