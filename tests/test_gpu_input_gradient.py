"""quantized_matmul with transpose = False (the gradient of a quantized linear layer with respect to its input) at the edges of
its tiles, against the float64 product of the dequantised matrix and against the plain kernel, which takes what is not aligned."""
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

# One rounding to the result's type: at most 2^-8 / 2^-11 of each value.  float32: a chain of at most K / 4 * 6 / 16 matrix
# instructions, each of which may cut a unit of 2^-24 off a running sum: 2^-24 * 0.1 K here, and four units for the rest.
BOUND = {"bfloat16": lambda k: 2.0 ** -8, "float16": lambda k: 2.0 ** -11, "float32": lambda k: (0.1 * k + 4) * 2.0 ** -24}
SHAPES = [  # rows, N, K: K below a step, not a whole number of steps, of an uneven share; N of 1, 3 and 65 times 32; each tile
    (1, 128, 8), (33, 128, 40), (5, 384, 1096), (65, 4224, 200), (300, 2176, 72), (1100, 2176, 136), (130, 2304, 328),
]


def operands(rows, n, k, bits, group, dtype, std=0.02):
    import mlx_rs_amd as m
    gen = torch.Generator(device="cuda").manual_seed(rows + n + k)
    q, s, b = m.ops.quantize(torch.randn((k, n), generator=gen, device="cuda") * std, group, bits, dtype)
    return torch.randn((rows, k), generator=gen, device="cuda").to(dtype), q, s, b


def dequantized(q, s, b, group, bits):
    shift = torch.arange(32 // bits, device=q.device) * bits
    codes = (((q.to(torch.int64) & 0xFFFFFFFF).unsqueeze(-1) >> shift) & ((1 << bits) - 1)).reshape(q.shape[0], -1).double()
    return codes * s.double().repeat_interleave(group, 1) + b.double().repeat_interleave(group, 1)


def off_by_one(x):
    """The same rows at an address that is not a multiple of 16 bytes: the plain kernel's."""
    buf = torch.empty(x.numel() + 1, dtype=x.dtype, device=x.device)
    buf[1:] = x.reshape(-1)
    return buf[1:].reshape(x.shape)


@pytest.mark.parametrize("dtype", ["bfloat16", "float16", "float32"])
@pytest.mark.parametrize("bits,group", [(4, 32), (4, 64), (4, 128), (8, 32), (8, 64), (8, 128)])
@pytest.mark.parametrize("rows,n,k", SHAPES)
def test_input_gradient(rows, n, k, bits, group, dtype):
    import mlx_rs_amd as m
    dt = getattr(torch, dtype)
    n = n + 32 if group == 32 else n  # (an output that fills no whole 64-column tile)
    x, q, s, b = operands(rows, n, k, bits, group, dt)
    y = m.ops.quantized_matmul(x, q, s, b, transpose=False, group_size=group, bits=bits)
    ref = x.double() @ dequantized(q, s, b, group, bits)
    err = float((y.double() - ref).norm() / ref.norm())
    assert y.dtype == dt and err <= BOUND[dtype](k), err
    plain = m.ops.quantized_matmul(off_by_one(x), q, s, b, transpose=False, group_size=group, bits=bits)
    perr = float((plain.double() - ref).norm() / ref.norm())
    assert err <= 1.01 * perr + 2.0 ** -24, (err, perr)  # (both have the same rounding of the result; sums in another order)


@pytest.mark.parametrize("dtype", ["bfloat16", "float16"])
@pytest.mark.parametrize("bits", [4, 8])
# the last rows of a tile whose launch gives an XCD 32 of them and the first of the next larger one's; K of no whole number of steps, and of one
@pytest.mark.parametrize("rows,n,k", [(64, 2688, 72), (65, 2688, 72), (128, 2688, 296), (129, 2688, 296), (256, 2688, 520), (320, 2688, 32), (321, 2688, 520)])
def test_tiles_around_a_round_of_an_xcd(rows, n, k, bits, dtype):
    test_input_gradient(rows, n, k, bits, 64, dtype)


@pytest.mark.parametrize("dtype", ["bfloat16", "float16", "float32"])
@pytest.mark.parametrize("bits", [4, 8])
def test_values_that_are_not_finite_or_leave_the_pieces(bits, dtype):
    """Infinities, NaNs and weights beyond the range of a piece: every element is what the plain kernel says, to the bit where
    the result is not finite or a piece has overflowed."""
    import mlx_rs_amd as m
    dt = getattr(torch, dtype)
    x, q, s, b = operands(40, 64, 200, bits, 32, dt)
    x[0, 3], x[33, 199], x[7, 0], x[39, 5] = float("inf"), float("-inf"), float("nan"), torch.finfo(dt).max
    run = lambda v, ss: m.ops.quantized_matmul(v, q, ss, b, transpose=False, group_size=32, bits=bits)  # noqa: E731
    y, plain = run(x, s), run(off_by_one(x), s)
    assert torch.equal(y.isnan(), plain.isnan()) and torch.equal(y.isinf(), plain.isinf())
    odd = ~plain.isfinite()
    assert odd.any() and torch.equal(y[odd].nan_to_num(), plain[odd].nan_to_num())
    big = (s.float() + (3.0e3 if dtype == "float16" else 2.0e37)).to(dt)  # (codes of 4 and 8 bits: well beyond 64)
    x = (x.nan_to_num(0, 0, 0).clamp(-1, 1) * 1e-3).to(dt)
    y, plain = run(x, big), run(off_by_one(x), big)
    assert torch.equal(y.isfinite(), plain.isfinite())
    ok = plain.isfinite()
    assert float((y[ok].double() - plain[ok].double()).norm()) <= 2.0 ** -7 * float(plain[ok].double().norm())


def shares_not_nearest(x, q, s, b, group, bits, ref):
    """Of the results, and of the plain kernel's: the share that is not the float64 product's nearest value.  It measures what the sums
    lose before the last rounding, an error d moving a result over a rounding boundary with probability |d| / spacing."""
    import mlx_rs_amd as m
    run = lambda v: m.ops.quantized_matmul(v, q, s, b, transpose=False, group_size=group, bits=bits)  # noqa: E731
    return tuple(float((v != ref.to(x.dtype)).double().mean()) for v in (run(x), run(off_by_one(x))))


@pytest.mark.parametrize("dtype", ["bfloat16", "float16"])
@pytest.mark.parametrize("bits,group", [(4, 32), (4, 64), (8, 64), (8, 128)])
@pytest.mark.parametrize("rows,n,k", [(20, 1024, 4096), (300, 2048, 2048), (1100, 2176, 1024)])
def test_sums_lose_no_more_than_plain_ones(rows, n, k, bits, group, dtype):
    """Matrices as quantize makes them, whose weights two pieces hold."""
    x, q, s, b = operands(rows, n, k, bits, group, getattr(torch, dtype))
    share, plain = shares_not_nearest(x, q, s, b, group, bits, x.double() @ dequantized(q, s, b, group, bits))
    assert share <= 1.25 * plain + 1e-4, (share, plain)


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("rows,n,k", [(20, 256, 1096), (300, 2176, 264), (1100, 2176, 328)])
def test_weights_of_more_bits_than_two_pieces(rows, n, k, bits):
    """Groups far from zero, 1 + q / 2^13, in some steps of K only, and rows that sum to zero, so that the rest of a weight is all that
    counts.  Two pieces of bfloat16 hold 17 bits of its 20 and more, which leaves a share of 0.11 to 0.14.  Sums that cancel as a whole show
    what a matrix instruction cuts off: about 2^-23 (half a unit of 2^-24 of its largest term, 4), 3 K / 16 times at random, 1.7e-6 for K =
    1096 against a spacing of 1.1e-4 at the results' root mean square 0.02 (4-bit), a share of 0.012.  Twice that is allowed."""
    x, q, s, b = operands(rows, n, k, bits, 64, torch.bfloat16)
    gen = torch.Generator(device="cuda").manual_seed(bits)
    q = torch.randint(-2 ** 31, 2 ** 31, q.shape, generator=gen, dtype=torch.int32, device="cuda")
    x[:, 1::2] = -x[:, ::2]
    far = (torch.arange(k, device="cuda") // 32 % 3 != 1).unsqueeze(1)
    s, b = torch.where(far, torch.full_like(s, 1.37 * 2.0 ** -13), torch.zeros_like(s)), torch.where(far, torch.ones_like(b), b.abs())
    pairs = dequantized(q, s, b, 64, bits)
    share, _ = shares_not_nearest(x, q, s, b, 64, bits, x[:, ::2].double() @ (pairs[::2] - pairs[1::2]))
    assert share <= 0.024, share
