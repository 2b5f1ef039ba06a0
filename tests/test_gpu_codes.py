"""The products on raw codes (quantized_linear in float16 and bfloat16; blocks with groups of 32 and 128) at the edges of their tiles
and of their sharing of K, and float32's plain sums, against the float64 product of the dequantised matrix."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

# One rounding to the result's type, half a unit of 8 (bfloat16) or 11 (float16) significant bits, is at most 2^-8 or
# 2^-11 of each value, and so of the whole in the 2-norm (typically 0.4 of that).  float32: a wave's 64 sums of up to K / 64 terms and
# their tree, each addition off by half a unit of 2^-24 at random: 1.0e-7 to 1.5e-7 up to K = 4096.  Sums that cancel against a
# bias term (codes that are not centred) are 3.3e-7 and more off.
BOUND = {"bfloat16": 2.0 ** -8, "float16": 2.0 ** -11, "float32": 2.0 ** -22}
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


@pytest.mark.parametrize("dtype", ["float16", "bfloat16"])
@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("rows,n,k", [(200, 4096, 4352), (200, 4096, 11008), (40, 2048, 8704)])
def test_shares_of_k_of_an_odd_number_of_groups(rows, n, k, bits, dtype):
    """Groups of 128 and K shared by two and by four groups of waves, each of 17, 43 and 17 groups: a share's scales start
    between two words and are more than one fetch holds.  Each row within the bound, which one wrong group in 34 is not."""
    import mlx_rs_amd as m
    dt = getattr(torch, dtype)
    gen = torch.Generator(device="cuda").manual_seed(rows + n + k)
    q, s, b = m.ops.quantize(torch.randn((n, k), generator=gen, device="cuda") * 0.02, 128, bits, dt)
    x = torch.randn((rows, k), generator=gen, device="cuda").to(dt)
    ref = product(x, q, s, b, 128, bits)
    y = m.ops.quantized_linear(x, q, s, b, group_size=128, bits=bits)
    err = (y.double() - ref).norm(dim=1) / ref.norm(dim=1)
    assert float(err.max()) <= BOUND[dtype], float(err.max())


def off_by_one(t):
    """The same values one element behind an aligned address."""
    buf = torch.empty(t.numel() + 1, dtype=t.dtype, device=t.device)
    buf[1:] = t.reshape(-1)
    return buf[1:].reshape(t.shape)


@pytest.mark.parametrize("dtype,group", [("float16", 64), ("float16", 128), ("bfloat16", 32), ("bfloat16", 128)])
@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("rows", [7, 40, 300])
def test_scales_between_two_words(rows, bits, dtype, group):
    """Scales or biases that start two bytes behind a word, which the kernels on raw codes read by words: the product goes to the
    plain kernel (as rows at such an address do)."""
    import mlx_rs_amd as m
    dt = getattr(torch, dtype)
    for n, k in ((48, 384), (37, 384)):
        gen = torch.Generator(device="cuda").manual_seed(rows + n)
        q, s, b = m.ops.quantize(torch.randn((n, k), generator=gen, device="cuda") * 0.02, group, bits, dt)
        x = torch.randn((rows, k), generator=gen, device="cuda").to(dt)
        run = lambda *a: m.ops.quantized_linear(*a, group_size=group, bits=bits)  # noqa: E731
        plain = run(off_by_one(x), q, s, b)
        assert torch.equal(run(x, q, off_by_one(s), b), plain)
        assert torch.equal(run(x, q, s, off_by_one(b)), plain)


@pytest.mark.parametrize("dtype", ["float16", "bfloat16"])
@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("rows", [2, 40, 300])
def test_an_odd_number_of_scales(rows, bits, dtype):
    """37 x 3 scales: their last word reaches behind the tensor, so the plain kernel takes them (as it does rows that start between
    two words)."""
    import mlx_rs_amd as m
    dt = getattr(torch, dtype)
    gen = torch.Generator(device="cuda").manual_seed(rows)
    q, s, b = m.ops.quantize(torch.randn((37, 384), generator=gen, device="cuda") * 0.02, 128, bits, dt)
    x = torch.randn((rows, 384), generator=gen, device="cuda").to(dt)
    run = lambda v: m.ops.quantized_linear(v, q, s, b, group_size=128, bits=bits)  # noqa: E731
    assert torch.equal(run(x), run(off_by_one(x)))


@pytest.mark.parametrize("dtype,group", [("bfloat16", 32), ("bfloat16", 64), ("bfloat16", 128), ("float16", 32), ("float16", 64), ("float16", 128)])
@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("rows,n", [(16, 16384), (300, 4096)])  # the kernel of a few rows, tiles
def test_sums_lose_no_more_than_plain_ones(rows, n, bits, dtype, group):
    """The share of results that are not the float64 product's nearest value measures what the sums lose before the last rounding:
    an error d moves a result over a rounding boundary with probability |d| / spacing.  Plain float32 sums over 4096 values are
    1.5e-7 of the results' root mean square off; 2^-22, 1.6 times that, is allowed, and its mean over a normal error is 0.8 of it.
    (Codes that are not centred: 3e-7 in float16, 1e-5 with bfloat16's 128 + q.)"""
    import mlx_rs_amd as m
    dt = getattr(torch, dtype)
    gen = torch.Generator(device="cuda").manual_seed(rows + group + bits)
    q, s, b = m.ops.quantize(torch.randn((n, 4096), generator=gen, device="cuda") * 0.02, group, bits, dt)
    x = torch.randn((rows, 4096), generator=gen, device="cuda").to(dt)
    ref = product(x, q, s, b, group, bits)
    y = m.ops.quantized_linear(x, q, s, b, group_size=group, bits=bits)
    spacing = torch.finfo(dt).eps * torch.exp2(torch.floor(torch.log2(ref.abs())))
    allowed = float((0.8 * 2.0 ** -22 * ref.square().mean().sqrt() / spacing).clamp(max=1).mean())
    share = float((y != ref.to(dt)).double().mean())
    assert share <= allowed, (share, allowed)


@pytest.mark.parametrize("transpose", [True, False])
def test_float32_values_near_the_largest(transpose):
    """Plain sums of them, and the input gradient's, which splits them into pieces: the first piece of the largest number is an
    infinity, and the result is computed again."""
    import mlx_rs_amd as m
    most = float(np.finfo(np.float32).max)
    x = torch.zeros((3, 128), device="cuda")
    x[0], x[2, 5] = most / 1024, most
    q, s, b = m.ops.quantize(torch.ones((64, 128) if transpose else (128, 64), device="cuda"), 64, 4, torch.float32)
    y = m.ops.quantized_matmul(x, q, s, b, transpose=transpose, group_size=64, bits=4)
    want = torch.tensor([[most / 8], [0.0], [most]], device="cuda").expand(3, 64)
    assert torch.allclose(y, want, rtol=1e-6)


def block_truth(blk, x, routing):
    """The block in float64 on the dequantised weights, with the routing the block itself reports."""
    c = blk.config
    out = torch.zeros(x.shape, dtype=torch.float64, device=x.device)
    for e in range(c.n_experts):
        hit = (routing["topk_idx"] == e).nonzero()
        if hit.numel() == 0:
            continue
        mats = (blk.gate_proj, blk.up_proj, blk.down_proj)
        prod = lambda v, p: product(v, p.weight[e], p.scales[e], p.biases[e], c.group_size, c.bits)  # noqa: E731
        g, u = prod(x[hit[:, 0]], mats[0]), prod(x[hit[:, 0]], mats[1])
        y = prod(g * torch.sigmoid(g) * u, mats[2])
        out.index_add_(0, hit[:, 0], y * routing["topk_w"][hit[:, 0], hit[:, 1]].double()[:, None])
    return out


@pytest.mark.parametrize("hidden,inter,experts,k", [(256, 384, 8, 2), (1152, 128, 5, 3), (256, 192, 4, 2)])
@pytest.mark.parametrize("bits,group", [(4, 32), (4, 128), (8, 32), (8, 128)])
@pytest.mark.parametrize("tokens,zipf", [(1, None), (17, None), (40, 1.5), (200, None), (700, 1.5)])
def test_blocks_with_groups_of_32_and_128(tokens, zipf, bits, group, hidden, inter, experts, k):
    """One row, one pass and several passes of the kernel of a few rows, tile lists with and without short segments, tiles
    of every list; the last shape is one the plain products keep with 4-bit codes.  Three roundings to bfloat16 (h, y and
    the result), each at most 2^-8 of its values and typically 0.42 of that, so 0.73 * 2^-8 together: 2^-8.  The plain
products round gate and up as well (0.94 * 2^-8, over as few as 256 values): 1.5 * 2^-8."""
    import mlx_rs_amd as m
    from mlx_rs_amd import synth
    if inter % group:
        pytest.skip("the intermediate size is a multiple of the group")
    cfg = m.MoeConfig(hidden, experts, k, inter, bits, group, 0)
    blk = synth.make_block(cfg, seed=tokens, device="cuda", zipf_s=zipf, gen_device="cuda")
    x = synth.make_tokens(cfg, tokens, seed=bits, device="cuda")
    out, routing = blk.forward(x, debug=True)
    ref = block_truth(blk, x, routing)
    err = float((out.double() - ref).norm() / ref.norm())
    bound = 1.5 * 2.0 ** -8 if bits == 4 and inter % 128 else 2.0 ** -8
    assert err <= bound, err
    # the same from the built-in scratch (no room for tile lists) where it fits
    if blk.workspace_bytes(tokens) < 8 << 20:
        again = blk.forward_static(x)
        assert float((again.double() - ref).norm() / ref.norm()) <= bound


@pytest.mark.parametrize("hidden,inter,experts,k", [(256, 384, 8, 2), (1152, 128, 9, 3), (128, 1152, 40, 8)])
@pytest.mark.parametrize("rows", [5, 15.9, 16, 30])
@pytest.mark.parametrize("bits,group", [(4, 32), (4, 128), (8, 32)])
def test_long_segments_on_both_sides_of_sixteen_rows_an_expert(bits, group, rows, hidden, inter, experts, k):
    """With 4-bit codes in groups of 32 the long segments' tiles hold their codes in registers below that average and in LDS from it on.
    Uneven routing: segments of one to all the tokens, in tiles of 1 to 64 rows; columns and K of 1, 3 and 9 times 128.  The bound is
    test_blocks_with_groups_of_32_and_128's.  The order of the tokens changes no bit of a row whose segment keeps its kernel."""
    import mlx_rs_amd as m
    from mlx_rs_amd import synth
    tokens = max(int(rows * experts / k), 17)
    cfg = m.MoeConfig(hidden, experts, k, inter, bits, group, 0)
    blk = synth.make_block(cfg, seed=int(rows), device="cuda", zipf_s=1.2, gen_device="cuda")
    x = synth.make_tokens(cfg, tokens, seed=bits, device="cuda")
    out, routing = blk.forward(x, debug=True)
    ref = block_truth(blk, x, routing)
    assert float((out.double() - ref).norm() / ref.norm()) <= 2.0 ** -8
    p = torch.randperm(tokens, generator=torch.Generator().manual_seed(3)).cuda()
    assert torch.equal(blk.forward(x[p].contiguous()), out[p])


def test_a_gate_that_is_not_finite_in_tiles_with_codes_in_registers():
    import mlx_rs_amd as m
    from mlx_rs_amd import synth
    cfg = m.MoeConfig(256, 8, 2, 384, 4, 32, 0)
    blk = synth.make_block(cfg, seed=2, device="cuda", zipf_s=1.0, gen_device="cuda")
    x = synth.make_tokens(cfg, 45, seed=1, device="cuda")
    blk.gate_proj.biases[:, 5, 2] = float("inf")
    blk.up_proj.biases[:, 7, 0] = float("-inf")
    blk.down_proj.scales[:, 9, 1] = float("inf")
    out, routing = blk.forward(x, debug=True)
    ref = block_truth(blk, x, routing)
    assert not ref.isfinite().all() and torch.equal(out.isnan(), ref.isnan()) and torch.equal(out.isinf(), ref.isinf())


@pytest.mark.parametrize("dtype", ["float16", "bfloat16"])
@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("group", [32, 64, 128])
@pytest.mark.parametrize("n", [208, 16384, 32784])
def test_waves_that_share_k_in_the_kernel_of_a_few_rows(n, group, bits, dtype):
    """Four, two and one (1024 and 2048 tiles of 16 weight rows), with columns past the last whole block; 17 chunks of 4-bit codes, so the shares
    are uneven."""
    import mlx_rs_amd as m
    dt, k = getattr(torch, dtype), 2176
    gen = torch.Generator(device="cuda").manual_seed(n + group + bits)
    q, s, b = m.ops.quantize(torch.randn((n, k), generator=gen, device="cuda") * 0.02, group, bits, dt)
    for rows in (2, 11):
        x = torch.randn((rows, k), generator=gen, device="cuda").to(dt)
        ref = product(x, q, s, b, group, bits)
        y = m.ops.quantized_linear(x, q, s, b, group_size=group, bits=bits)
        err = (y.double() - ref).norm(dim=1) / ref.norm(dim=1)
        assert float(err.max()) <= BOUND[dtype], (rows, err)


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("group", [32, 128])
@pytest.mark.parametrize("experts", [16, 32, 64])
def test_waves_that_share_k_in_a_block(experts, group, bits):
    """The same for the gate and up product: 512, 1024 and 2048 tiles of 16 weight rows."""
    test_blocks_with_groups_of_32_and_128(15, None, bits, group, 256, 512, experts, 5)


@pytest.mark.parametrize("tokens", [4, 6, 14])
def test_a_small_batch_with_long_rows(tokens):
    """No segment can be longer than one pass of the kernel of a few rows: no tile lists, and that kernel's LDS is that of the
    batch's own rows (with 16 of them 8576 values in groups of 32 would not fit)."""
    import mlx_rs_amd as m
    from mlx_rs_amd import synth
    cfg = m.MoeConfig(8576, 8, 8, 4096, 4, 32, 0)
    blk = synth.make_block(cfg, seed=tokens, device="cuda", gen_device="cuda")
    x = synth.make_tokens(cfg, tokens, seed=2, device="cuda")
    out, routing = blk.forward(x, debug=True)
    ref = block_truth(blk, x, routing)
    assert float((out.double() - ref).norm() / ref.norm()) <= 2.0 ** -8


@pytest.mark.parametrize("dtype,group", [("float16", 64), ("bfloat16", 32), ("float32", 128)])
@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("rows", [7, 70, 1100])
def test_values_that_are_not_finite(rows, bits, dtype, group):
    """Infinities and NaNs in the rows, the scales and the biases: every element is one where the product of the
    dequantised matrix is, with its sign, in the kernel of a few rows and in the tiles of both code orders."""
    import mlx_rs_amd as m
    dt = getattr(torch, dtype)
    gen = torch.Generator(device="cuda").manual_seed(rows + bits)
    q, s, b = m.ops.quantize(torch.randn((200, 384), generator=gen, device="cuda") * 0.02, group, bits, dt)
    x = torch.randn((rows, 384), generator=gen, device="cuda").to(dt)
    x[0, 3], x[rows - 1, 383], x[rows // 2, 130] = float("inf"), float("-inf"), float("nan")
    b[17, 1], s[199, 2] = float("inf"), float("inf")
    ref = product(x, q, s, b, group, bits)
    y = m.ops.quantized_linear(x, q, s, b, group_size=group, bits=bits)
    odd = ~ref.isfinite()
    assert odd.any() and torch.equal(y.isfinite(), ~odd)
    assert torch.equal(y[odd].double().nan_to_num(), ref[odd].nan_to_num())


def fastest(run, times=3):
    """ms of the fastest of a few calls."""
    run()
    ms = []
    for _ in range(times):
        a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        a.record()
        run()
        b.record()
        b.synchronize()
        ms.append(a.elapsed_time(b))
    return min(ms)


@pytest.mark.parametrize("way,dtype,bits", [("forward", "bfloat16", 4), ("forward", "float16", 8), ("backward", "bfloat16", 4), ("backward", "float32", 4)])
def test_rows_that_are_not_finite_cost_no_more_than_the_plain_kernel(way, dtype, bits):
    """An infinity in every row: all results are computed again, which took four to twenty times the plain kernel's time when it was
    done one by one, and takes 0.6 to 0.7 of it."""
    import mlx_rs_amd as m
    dt = getattr(torch, dtype)
    n, k = (4096, 4096) if way == "forward" else (2048, 4096)
    w = torch.randn((n, k) if way == "forward" else (k, n), device="cuda") * 0.02
    q, s, b = m.ops.quantize(w, 32, bits, dt)
    x = torch.randn((800, k), device="cuda").to(dt)
    x[:, 1] = float("inf")
    run = lambda v: m.ops.quantized_linear(v, q, s, b, transpose=way == "forward", group_size=32, bits=bits)  # noqa: E731
    other = off_by_one(x)
    assert fastest(lambda: run(x)) <= 1.5 * fastest(lambda: run(other))


@pytest.mark.parametrize("tokens,zipf", [(9, None), (300, 1.5)])
def test_a_block_whose_gate_is_not_finite(tokens, zipf):
    """Gate products that are infinite or no number (a scale that is) go through the activation as they are."""
    import mlx_rs_amd as m
    from mlx_rs_amd import synth
    cfg = m.MoeConfig(256, 4, 2, 128, 4, 32, 0)
    blk = synth.make_block(cfg, seed=tokens, device="cuda", zipf_s=zipf, gen_device="cuda")
    x = synth.make_tokens(cfg, tokens, seed=1, device="cuda")
    blk.gate_proj.biases[1, 5, 2] = float("inf")
    blk.up_proj.biases[2, 7, 0] = float("-inf")
    out, routing = blk.forward(x, debug=True)
    ref = block_truth(blk, x, routing)
    assert not ref.isfinite().all() and torch.equal(out.isnan(), ref.isnan()) and torch.equal(out.isinf(), ref.isinf())
