"""Blocks whose segments all go through short tiles on raw codes (groups of 64, 4-bit, 65 tokens and more up to 96 rows per expert), and
the tiles the dense products on raw codes choose from, against float64."""
import ctypes as C

import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

from test_dense_rule import COLUMNS, REGISTERS, REGISTERS_SHARED, REGISTERS_SMALL, SMALL, WIDE, rule  # noqa: E402,F401
from test_gpu_codes import BOUND, block_truth, product  # noqa: E402

# hidden, intermediate, experts, k: K of 1, 3, 5 and 9 stages of 128 (windows of eight, whole and started), columns that fill no block of
# 128 or 256, more experts than a wave has lanes; the last three have experts enough for 8 rows each
BLOCKS = [(128, 384, 8, 2), (1152, 128, 9, 3), (640, 1152, 16, 8), (256, 256, 70, 8), (128, 384, 64, 2), (384, 128, 96, 6)]


@pytest.mark.parametrize("hidden,inter,experts,k", BLOCKS)
@pytest.mark.parametrize("rows", [8, 33, 64, 90])
@pytest.mark.parametrize("zipf", [None, 1.4])
def test_blocks_in_short_tiles(zipf, rows, hidden, inter, experts, k):
    """On average `rows` rows an expert, or what makes 512 pairs and 65 tokens where that is more (the fewest that come this way): segments on
    both sides of 32 and 64 rows, and of several tiles.  Three roundings to
    bfloat16 (h, y and the result), each at most 2^-8 of its values and typically 0.42 of that: 0.73 * 2^-8 together.  The built-in
    scratch takes the same route; the order of the tokens changes no bit."""
    import mlx_rs_amd as m
    from mlx_rs_amd import synth
    tokens = max(rows * experts // k, 65, -(-512 // k))
    if tokens * k > 96 * experts:
        pytest.skip("more rows than this route takes")
    cfg = m.MoeConfig(hidden, experts, k, inter, 4, 64, 0)
    blk = synth.make_block(cfg, seed=rows, device="cuda", zipf_s=zipf, gen_device="cuda")
    x = synth.make_tokens(cfg, tokens, seed=k, device="cuda")
    out, routing = blk.forward(x, debug=True)
    ref = block_truth(blk, x, routing)
    err = (out.double() - ref).norm() / ref.norm()
    assert float(err) <= 2.0 ** -8, float(err)
    p = torch.randperm(tokens, generator=torch.Generator().manual_seed(3)).cuda()
    assert torch.equal(blk.forward(x[p].contiguous()), out[p])
    if blk.workspace_bytes(tokens) < 8 << 20:
        assert torch.equal(blk.forward_static(x), out)


# an average of 97 rows and more: K of one window of sixteen groups and of two, h of more groups than a window, fewer columns than a block's
@pytest.mark.parametrize("hidden,inter,experts,k", [(128, 384, 8, 2), (1152, 1280, 9, 3), (256, 128, 64, 2)])
@pytest.mark.parametrize("rows", [70, 97, 128, 300])
@pytest.mark.parametrize("zipf", [None, 1.4])
def test_blocks_in_longer_pieces(zipf, rows, hidden, inter, experts, k):
    """Pieces of 96 and 128 rows (70 rows an expert; beyond 96 with the segments of fewer than nine rows streamed beside them) and their last ones of every
    length, with the bound of test_blocks_in_short_tiles: the same roundings.  The scratch that is built in and the residual form take the same tiles."""
    import mlx_rs_amd as m
    from mlx_rs_amd import synth
    tokens = rows * experts // k
    cfg = m.MoeConfig(hidden, experts, k, inter, 4, 64, 0)
    assert m.capi.tile_rule(cfg.c_struct(), tokens) == ((2, 1) if rows <= 96 else (3, 9))
    blk = synth.make_block(cfg, seed=rows, device="cuda", zipf_s=zipf, gen_device="cuda")
    x = synth.make_tokens(cfg, tokens, seed=k, device="cuda")
    out, routing = blk.forward(x, debug=True)
    ref = block_truth(blk, x, routing)
    assert float((out.double() - ref).norm() / ref.norm()) <= 2.0 ** -8
    rms = ref.square().mean(1).sqrt()  # (a row in another's place would be as far off as itself)
    assert float(((out.double() - ref).norm(dim=1) / (rms * hidden ** 0.5)).max()) <= 2.0 ** -6
    p = torch.randperm(tokens, generator=torch.Generator().manual_seed(3)).cuda()
    assert torch.equal(blk.forward(x[p].contiguous()), out[p])
    if blk.workspace_bytes(tokens) < 8 << 20:
        assert torch.equal(blk.forward_static(x), out)
    one = torch.ones(hidden, dtype=torch.bfloat16, device="cuda")
    xn = m.ops.rms_norm(x, one, 1e-6)
    own, routing = blk.forward_residual(x, one, 1e-6, debug=True)
    ref = x.double() + block_truth(blk, xn, routing)
    assert float((own.double() - ref).norm() / ref.norm()) <= 2.0 ** -8


@pytest.mark.parametrize("group", [32, 128])
@pytest.mark.parametrize("bits", [4, 8])
# a decode batch (the router's one launch) and larger ones; rows of an odd number of groups of 128, of more than a window, columns that fill no block;
# the last two around the rows an expert between which 8-bit codes keep short segments apart
@pytest.mark.parametrize("hidden,inter,experts,k,tokens", [(128, 384, 8, 2, 17), (384, 128, 4, 2, 64), (2176, 640, 9, 3, 70), (384, 1152, 16, 8, 300),
                                                           (256, 256, 8, 2, 79), (256, 256, 8, 2, 80)])
def test_blocks_all_in_tiles(hidden, inter, experts, k, tokens, bits, group):
    """Groups of 32 and 128, segments of every length in tiles; the bound is test_blocks_in_short_tiles'."""
    import mlx_rs_amd as m
    from mlx_rs_amd import synth
    cfg = m.MoeConfig(hidden, experts, k, inter, bits, group, 0)
    blk = synth.make_block(cfg, seed=group, device="cuda", zipf_s=0.7, gen_device="cuda")
    x = synth.make_tokens(cfg, tokens, seed=bits, device="cuda")
    out, routing = blk.forward(x, debug=True)
    ref = block_truth(blk, x, routing)
    assert float((out.double() - ref).norm() / ref.norm()) <= 2.0 ** -8
    p = torch.randperm(tokens, generator=torch.Generator().manual_seed(3)).cuda()
    assert torch.equal(blk.forward(x[p].contiguous()), out[p])
    one = torch.ones(hidden, dtype=torch.bfloat16, device="cuda")
    own, routing = blk.forward_residual(x, one, 1e-6, debug=True)
    ref = x.double() + block_truth(blk, m.ops.rms_norm(x, one, 1e-6), routing)
    assert float((own.double() - ref).norm() / ref.norm()) <= 2.0 ** -8


def test_a_layer_around_short_tiles():
    """The normalised rows' memory takes the group sums of h once they have been read: the residual form against its parts."""
    import mlx_rs_amd as m
    from mlx_rs_amd import synth
    cfg = m.MoeConfig(256, 8, 2, 512, 4, 64, 0)
    blk = synth.make_block(cfg, seed=4, device="cuda", zipf_s=1.1, gen_device="cuda")
    x = synth.make_tokens(cfg, 300, seed=4, device="cuda")
    w = (1.0 + 0.1 * torch.randn(256, generator=torch.Generator().manual_seed(1))).to(torch.bfloat16).cuda()
    xn = m.ops.rms_norm(x, w, 1e-6)
    out, routing = blk.forward_residual(x, w, 1e-6, debug=True)
    ref = x.double() + block_truth(blk, xn, routing)
    assert float((out.double() - ref).norm() / ref.norm()) <= 2.0 ** -8


# (the second batch: pieces of 128 rows beside streamed segments)
@pytest.mark.parametrize("tokens", [270, 1000])
def test_short_tiles_with_a_gate_that_is_not_finite(tokens):
    import mlx_rs_amd as m
    from mlx_rs_amd import synth
    cfg = m.MoeConfig(256, 8, 2, 384, 4, 64, 0)
    blk = synth.make_block(cfg, seed=2, device="cuda", zipf_s=1.0, gen_device="cuda")
    x = synth.make_tokens(cfg, tokens, seed=1, device="cuda")
    assert m.capi.tile_rule(cfg.c_struct(), tokens) == ((2, 1) if tokens == 270 else (3, 9))
    blk.gate_proj.biases[1, 5, 2] = float("inf")
    blk.up_proj.biases[2, 7, 0] = float("-inf")
    blk.down_proj.scales[3, 9, 1] = float("inf")
    out, routing = blk.forward(x, debug=True)
    ref = block_truth(blk, x, routing)
    assert not ref.isfinite().all() and torch.equal(out.isnan(), ref.isnan()) and torch.equal(out.isinf(), ref.isinf())


# (pieces of 64, 96 and 128 rows, the last beside streamed segments; the list of groups of 32; more experts than waves have lanes, and not a multiple of those)
@pytest.mark.parametrize("experts,group,lengths,piece", [(70, 64, [0, 1, 31, 32, 33, 63, 64, 65], 64), (130, 64, [64, 96, 97, 32, 95, 0, 128, 33], 96),
                                                         (9, 64, [127, 128, 129, 9, 8, 255, 96, 97, 32], 128), (200, 32, [0, 64, 1, 63, 65, 32, 129, 33], 64)])
def test_segments_of_chosen_lengths(experts, group, lengths, piece):
    """Lengths on both sides of every one at which the list of pieces starts another, in the order of the experts: a piece that is left out, listed twice or
    listed for another expert leaves rows that are far off.  Every token has its expert's column large, and the router is the unit matrix.  The bound of a row
    is one and a half times test_blocks_in_short_tiles' of the whole."""
    import mlx_rs_amd as m
    from mlx_rs_amd import synth
    cfg = m.MoeConfig(256, experts, 1, 128, 4, group, 0)
    blk = synth.make_block(cfg, seed=4, device="cuda", gen_device="cuda")
    blk.gate_weight.copy_(torch.eye(256)[:experts])
    of = torch.cat([torch.full((lengths[e % len(lengths)],), e) for e in range(experts)]).cuda()
    tokens = of.numel()
    assert piece == (64 if group != 64 or tokens < 48 * experts else 96 if tokens < 80 * experts else 128)
    of = of[torch.randperm(tokens, generator=torch.Generator().manual_seed(1)).cuda()]
    x = synth.make_tokens(cfg, tokens, seed=4, device="cuda")
    x[torch.arange(tokens, device="cuda"), of] = 16.0
    out, routing = blk.forward(x, debug=True)
    assert torch.equal(routing["topk_idx"][:, 0].long(), of)
    ref = block_truth(blk, x, routing)
    err = (out.double() - ref).norm(dim=1) / ref.norm(dim=1)
    assert float(err.max()) <= 1.5 * 2.0 ** -8, float(err.max())


# 540, 1000 and 400 pairs on 8 experts: pieces of up to 96 rows, of 128 beside streamed segments, and the list of groups of 32 and 128
@pytest.mark.parametrize("group,tokens", [(64, 270), (64, 500), (32, 200), (128, 200)])
def test_tiles_with_gates_far_below_zero(group, tokens):
    """silu of gates around -88, where 1 + exp(-g) leaves the numbers whose reciprocal is normal, and far beyond, where it is infinite and the quotient zero.
    Column 0 of x is the gate and column 64 (one) times 2^100 the up product, exactly (scales of zero, biases in those columns' groups), so h is large enough to
    see; the down product is half the sum of a group of h, 128 equal values.  Three roundings to bfloat16 (h, y and the result), and the two routing weights
    sum to one up to 2^-8."""
    import mlx_rs_amd as m
    from mlx_rs_amd import synth
    cfg = m.MoeConfig(256, 8, 2, 256, 4, group, 0)
    blk = synth.make_block(cfg, seed=6, device="cuda", zipf_s=0.7, gen_device="cuda")
    gates = torch.tensor([-1e38, -1e30, -1000.0, -100.0, -89.0, -88.5, -88.0, -87.5, -87.0, -60.0, -3.0, -0.0, 0.25, 5.0, 88.0, 100.0]).bfloat16()
    x = torch.zeros((tokens, 256), dtype=torch.bfloat16, device="cuda")
    x[:, 0] = gates.repeat(tokens // 16 + 1)[:tokens].cuda()
    x[:, 128] = 1.0
    x[:, 129:] = torch.randn((tokens, 127), generator=torch.Generator().manual_seed(2)).bfloat16().cuda() * (torch.arange(129, 256, device="cuda") >= 128 + group)
    blk.gate_weight[:, 0] = 0.0  # (the routing is that of the rest)
    for bank, column, value in ((blk.gate_proj, 0, 1.0), (blk.up_proj, 128, 2.0 ** 100), (blk.down_proj, 0, 0.5 / group)):
        bank.scales.zero_()
        bank.biases.zero_()
        bank.biases[:, :, column // group] = value
    out, routing = blk.forward(x, debug=True)
    g = x[:, 0].float()
    ref = (g / (1.0 + torch.exp(-g))).double() * 2.0 ** 99 * routing["topk_w"].double().sum(1)
    assert bool(out.isfinite().all())
    assert bool(((out.double() - ref[:, None]).abs() <= 2.0 ** -7 * ref.abs()[:, None]).all())


# pieces of up to 96 rows, and of 128 beside streamed segments
@pytest.mark.parametrize("tokens", [270, 1000])
def test_sums_of_codes_that_overflow_in_pieces(tokens):
    """An activation of 3e38 against weights of up to fifteen 2^-125: the sum of its codes is infinite, the product of the dequantised weights is not.  One row of
    each 32 of an expert's pieces, the last of the segment among them; the others' results stay within the bound of all."""
    import mlx_rs_amd as m
    from mlx_rs_amd import synth
    cfg = m.MoeConfig(256, 8, 2, 384, 4, 64, 0)
    blk = synth.make_block(cfg, seed=2, device="cuda", zipf_s=0.5, gen_device="cuda")
    x = synth.make_tokens(cfg, tokens, seed=1, device="cuda")
    blk.gate_weight[:, 7] = 0.0
    for bank in (blk.gate_proj, blk.up_proj):
        bank.scales[:, :, 0] = 2.0 ** -125
        bank.biases[:, :, 0] = 0.0
    _, routing = blk.forward(x, debug=True)
    perm, offsets, hit = routing["perm"].long(), routing["offsets"].tolist(), []
    for e in range(8):
        hit += [r for r in range(offsets[e] + 31, offsets[e + 1], 32)] + ([offsets[e + 1] - 1] if offsets[e + 1] > offsets[e] else [])
    rows = (perm[torch.tensor(hit, device="cuda")] // 2).unique()
    x[rows, 7] = 3e38
    out, routing = blk.forward(x, debug=True)
    assert max(b - a for a, b in zip(offsets, offsets[1:])) > (96 if tokens == 270 else 128)
    ref = block_truth(blk, x, routing)
    assert bool(ref.isfinite().all()) and float(ref[rows].norm(dim=1).min()) > 10 * float(ref.norm(dim=1).median())
    err = (out.double() - ref).norm(dim=1) / ref.norm(dim=1)
    assert float(err.max()) <= 2.0 ** -6, float(err.max())


@pytest.mark.parametrize("dtype,group", [("float16", 32), ("float16", 64), ("float16", 128), ("bfloat16", 32), ("bfloat16", 64), ("bfloat16", 128)])
@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("rows,n,k", [(200, 4096, 1152), (260, 4090, 640), (1000, 4096, 1408), (1000, 4090, 2176)])
def test_dense_tiles(rows, n, k, bits, dtype, group):
    """Shares of K of an odd number of stages and columns that end inside a tile (each tile of the rule:
    test_every_dense_tile_loses_no_more_than_plain_sums)."""
    import mlx_rs_amd as m
    dt = getattr(torch, dtype)
    gen = torch.Generator(device="cuda").manual_seed(rows + n + k)
    q, s, b = m.ops.quantize(torch.randn((n, k), generator=gen, device="cuda") * 0.02, group, bits, dt)
    x = torch.randn((rows, k), generator=gen, device="cuda").to(dt)
    ref = product(x, q, s, b, group, bits)
    y = m.ops.quantized_linear(x, q, s, b, group_size=group, bits=bits)
    err = (y.double() - ref).norm(dim=1) / ref.norm(dim=1)
    assert float(err.max()) <= BOUND[dtype], float(err.max())


def share_off_nearest(got, ref, error):
    """The share of results that are not the float64 value's nearest, and what sums off by `error` (its root mean square) would give: an error d moves a
    result over a rounding boundary with probability |d| / spacing, and the mean of a normal |d| is 0.8 of its root mean square."""
    spacing = torch.finfo(got.dtype).eps * torch.exp2(torch.floor(torch.log2(ref.abs().clamp(min=1e-30))))
    return float((got != ref.to(got.dtype)).double().mean()), float((0.8 * error / spacing).clamp(max=1).mean())


# rows, and the tile that 4096 columns and 4096 values take with 4- and 8-bit codes; the last two leave 9 rows for the last 64-row tile, whose body is the
# one of 32 rows
DENSE = [(100, (SMALL, SMALL)), (200, (COLUMNS, SMALL)), (400, (REGISTERS_SHARED, REGISTERS_SHARED)), (777, (WIDE, REGISTERS)), (1609, (WIDE, WIDE))]


@pytest.mark.parametrize("dtype,group", [("float16", 32), ("float16", 64), ("float16", 128), ("bfloat16", 32), ("bfloat16", 64), ("bfloat16", 128)])
@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("rows,tiles", DENSE)
def test_every_dense_tile_loses_no_more_than_plain_sums(rows, tiles, bits, dtype, group, rule):
    """Each tile of the rule over shares of K that all have work, whole and remaining rows.  The bound on what the sums lose is
    test_sums_lose_no_more_than_plain_ones': 2^-22 of the results' root mean square."""
    import mlx_rs_amd as m
    want = tiles[bits == 8]
    if (dtype, bits, group, want) == ("bfloat16", 8, 32, SMALL) and rows == 100:
        want = REGISTERS_SMALL
    assert rule.tile(rows, 4096, 4096, bits, group, dtype == "bfloat16") == want
    if dtype == "bfloat16" and group == 64 and rows == 1609:
        pytest.skip("rounds the weights: the 256 x 256 tiles")
    dt = getattr(torch, dtype)
    gen = torch.Generator(device="cuda").manual_seed(rows + group + bits)
    q, s, b = m.ops.quantize(torch.randn((4096, 4096), generator=gen, device="cuda") * 0.02, group, bits, dt)
    x = torch.randn((rows, 4096), generator=gen, device="cuda").to(dt)
    ref = product(x, q, s, b, group, bits)
    y = m.ops.quantized_linear(x, q, s, b, group_size=group, bits=bits)
    err = (y.double() - ref).norm(dim=1) / ref.norm(dim=1)
    assert float(err.max()) <= BOUND[dtype], float(err.max())
    share, allowed = share_off_nearest(y, ref, 2.0 ** -22 * ref.square().mean().sqrt())
    assert share <= allowed, (share, allowed)


@pytest.mark.parametrize("dtype,group", [("float16", 32), ("float16", 64), ("float16", 128), ("bfloat16", 32), ("bfloat16", 64), ("bfloat16", 128)])
@pytest.mark.parametrize("rows,n,k,bits", [(585, 4090, 1024, 4), (550, 4096, 1152, 4), (640, 3200, 2176, 4), (585, 4090, 1024, 8), (550, 4096, 1152, 8),
                                            (640, 3200, 2176, 8), (770, 4090, 3072, 8), (1000, 4096, 3200, 8)])
def test_longer_tiles_lose_no_more_than_plain_sums(rows, n, k, bits, dtype, group, rule):
    """96 and 128 rows: a last tile of 9, 2 and 104 rows, columns that end inside one, shares of 4 and 4, 5 and 4, 9 and 8, 13 and 12 stages of 128 values.  The
    bounds are test_every_dense_tile_loses_no_more_than_plain_sums'."""
    import mlx_rs_amd as m
    assert rule.longer(rows, n, k, bits) == (96 if rows < 700 else 128)
    dt = getattr(torch, dtype)
    gen = torch.Generator(device="cuda").manual_seed(rows + group + bits)
    q, s, b = m.ops.quantize(torch.randn((n, k), generator=gen, device="cuda") * 0.02, group, bits, dt)
    x = torch.randn((rows, k), generator=gen, device="cuda").to(dt)
    x[rows - 1, 5] = float("inf")  # (one result in a row of its own that is computed again)
    ref = product(x, q, s, b, group, bits)
    y = m.ops.quantized_linear(x, q, s, b, group_size=group, bits=bits)
    assert torch.equal(y[-1].double().nan_to_num(), ref[-1].nan_to_num())
    y, ref = y[:-1], ref[:-1]
    err = (y.double() - ref).norm(dim=1) / ref.norm(dim=1)
    assert float(err.max()) <= BOUND[dtype], float(err.max())
    share, allowed = share_off_nearest(y, ref, 2.0 ** -22 * ref.square().mean().sqrt())
    assert share <= allowed, (share, allowed)


# (the tiles of 64 x 128 in registers where a tile of 96 or 128 rows does not fill a round: 8-bit codes, K below 3072)
@pytest.mark.parametrize("dtype,group", [("float16", 32), ("float16", 64), ("bfloat16", 64), ("bfloat16", 128)])
def test_tiles_in_registers_beside_longer_ones(dtype, group, rule):
    import mlx_rs_amd as m
    rows, n, k = 777, 4096, 2048
    assert rule.longer(rows, n, k, 8) == 0 and rule.tile(rows, n, k, 8, group, dtype == "bfloat16") == REGISTERS
    dt = getattr(torch, dtype)
    gen = torch.Generator(device="cuda").manual_seed(group)
    q, s, b = m.ops.quantize(torch.randn((n, k), generator=gen, device="cuda") * 0.02, group, 8, dt)
    x = torch.randn((rows, k), generator=gen, device="cuda").to(dt)
    ref = product(x, q, s, b, group, 8)
    y = m.ops.quantized_linear(x, q, s, b, group_size=group, bits=8)
    share, allowed = share_off_nearest(y, ref, 2.0 ** -22 * ref.square().mean().sqrt())
    assert share <= allowed, (share, allowed)


def one_hot(n, value):
    """A bank's matrix, 4-bit in groups of 64: `value` on the diagonal, or in column 0 (n < 0), exactly."""
    codes = torch.zeros((abs(n), abs(n)), dtype=torch.int64)
    codes[torch.arange(abs(n)), torch.arange(abs(n)) if n > 0 else torch.zeros(abs(n), dtype=torch.int64)] = 1
    q = (codes.reshape(abs(n), -1, 8) << (4 * torch.arange(8))).sum(-1).to(torch.int32)
    return q, torch.full((abs(n), abs(n) // 64), float(value)).bfloat16(), torch.zeros((abs(n), abs(n) // 64)).bfloat16()


@pytest.mark.parametrize("which", ["down", "gate and up"])
def test_what_the_sums_of_a_block_in_short_tiles_lose(which):
    """Codes as they are, 0 to 15 (the tiles of blocks leave out the centre), and the group sums that gate/up hand to the down product.  One expert a
    token, whose score is 1, so the result is the down product's.  Down alone: a gate of 64, whose SiLU is 64, and up the unit matrix make h = 64 x exactly.
    Gate and up alone: down is the unit matrix, the result is h.
    What the sums may lose: the codes' root mean square is 8.2 of 15 steps where the weights' is 3.2, so the code term and the bias term are 2.6 times their
    sum each, and lose 2.6 sqrt(2) = 3.6 times what plain sums do (2^-22, see above); the fast exponential and the division 2^-21 of h."""
    import mlx_rs_amd as m
    from mlx_rs_amd import synth
    n, experts, tokens = 2048, 8, 600
    cfg = m.MoeConfig(n, experts, 1, n, 4, 64, 0)
    assert m.capi.tile_rule(cfg.c_struct(), tokens)[0] == 2
    blk = synth.make_block(cfg, seed=5, device="cuda", zipf_s=0.5, gen_device="cuda")

    def put(bank, mat):
        for t, v in zip((bank.weight, bank.scales, bank.biases), mat):
            t.copy_(v.expand_as(t))
    x = synth.make_tokens(cfg, tokens, seed=5, device="cuda")
    if which == "down":
        x[:, 0] = 1.0
        put(blk.gate_proj, one_hot(-n, 64))
        put(blk.up_proj, one_hot(n, 1))
    else:
        put(blk.down_proj, one_hot(n, 1))
    out, routing = blk.forward(x, debug=True)
    assert bool((routing["topk_w"] == 1).all())
    expert = routing["topk_idx"][:, 0]
    ref, error = torch.empty((tokens, n), dtype=torch.float64, device="cuda"), torch.empty((tokens, n), dtype=torch.float64, device="cuda")
    lose = 3.6 * 2.0 ** -22
    for e in range(experts):
        hit = expert == e
        mat = lambda v, p: product(v, p.weight[e], p.scales[e], p.biases[e], 64, 4)  # noqa: E731
        if which == "down":
            ref[hit] = mat(64 * x[hit], blk.down_proj)
            error[hit] = lose * ref[hit].square().mean().sqrt()
        else:
            g, u = mat(x[hit], blk.gate_proj), mat(x[hit], blk.up_proj)
            sig = torch.sigmoid(g)
            dg, du = sig * (1 + g * (1 - sig)) * u * g.square().mean().sqrt(), g * sig * u.square().mean().sqrt()
            ref[hit] = g * sig * u
            error[hit] = lose * (dg.square() + du.square()).sqrt() + 2.0 ** -21 * ref[hit].abs()
    share, allowed = share_off_nearest(out, ref, error)
    assert share <= allowed, (share, allowed)


@pytest.mark.parametrize("dtype", ["float16", "bfloat16"])
@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("rows,n,k", [(40, 2000, 2432), (70, 1532, 1152), (40, 1040, 7680), (40, 1040, 7808), (40, 1040, 8064), (150, 3840, 3200), (33, 1030, 384)])
def test_scales_of_shares_that_begin_between_two_words(rows, n, k, bits, dtype):
    """Groups of 128 and K shared by four groups of waves in shares of 5, 3, 15 (a window and its first place), 16, 16, 7 and 1 groups; rows of an
    odd number of scales (19, 9, 61, 63, 25, 3).  One group with another's scale or bias is far outside each row's bound."""
    import mlx_rs_amd as m
    dt = getattr(torch, dtype)
    gen = torch.Generator(device="cuda").manual_seed(rows + n + k)
    q, s, b = m.ops.quantize(torch.randn((n, k), generator=gen, device="cuda") * 0.02, 128, bits, dt)
    x = torch.randn((rows, k), generator=gen, device="cuda").to(dt)
    ref = product(x, q, s, b, 128, bits)
    y = m.ops.quantized_linear(x, q, s, b, group_size=128, bits=bits)
    err = (y.double() - ref).norm(dim=1) / ref.norm(dim=1)
    assert float(err.max()) <= BOUND[dtype], float(err.max())


@pytest.mark.parametrize("pairs,experts", [(2047, 8), (2048, 128), (2049, 8), (2049, 512), (4095, 70)])
def test_dispatch_around_one_block(pairs, experts):
    """The last pair count of the one-block kernel and the first of the two-launch form."""
    import mlx_rs_amd as m
    e = torch.randint(0, experts, (pairs,), generator=torch.Generator().manual_seed(pairs), dtype=torch.int32)
    counts, offsets, perm, inv = (t.cpu().long() for t in m.ops.dispatch(e.cuda(), experts))
    want = torch.argsort(e.long(), stable=True)
    assert torch.equal(counts, torch.bincount(e.long(), minlength=experts)) and torch.equal(offsets[1:], counts.cumsum(0))
    assert torch.equal(perm, want) and torch.equal(inv[perm], torch.arange(pairs))


@pytest.mark.parametrize("pairs,experts", [(2049, 8), (4096, 512), (3000, 70)])
def test_dispatch_with_the_workspace_of_one_block(pairs, experts):
    """512 bytes are enough up to 4096 pairs, as before the two-launch form, for the products by index too; the results are those of a full workspace."""
    import mlx_rs_amd as m
    lib = m.load_library()
    e = torch.randint(0, experts, (pairs,), generator=torch.Generator().manual_seed(pairs), dtype=torch.int32).cuda()
    perm, ws = torch.empty_like(e), torch.empty(512, dtype=torch.uint8, device="cuda")
    st = torch.cuda.current_stream().cuda_stream

    def dispatch(size, n=pairs):
        return lib.mi_moe_dispatch(e.data_ptr(), n, experts, None, None, perm.data_ptr(), None, ws.data_ptr(), size, st)
    assert dispatch(512) == 0 and torch.equal(perm.cpu().long(), torch.argsort(e.cpu().long(), stable=True))
    assert dispatch(511) != 0 and b"workspace too small" in lib.mi_moe_last_error()
    assert lib.mi_moe_dispatch(e.data_ptr(), 4097, experts, None, None, perm.data_ptr(), None, ws.data_ptr(), 512, st) != 0  # (refused before anything is read)
    need = C.c_size_t()
    m.capi.check(lib.mi_moe_gather_qmm_workspace_size(experts, pairs, 1, C.byref(need)))
    full = C.c_size_t()
    m.capi.check(lib.mi_moe_dispatch_workspace_size(experts, pairs, C.byref(full)))
    q, s, b = m.ops.quantize(torch.randn((experts * 16, 128), device="cuda") * 0.02, 64, 4)
    x = torch.randn((pairs, 1, 128), device="cuda").bfloat16()
    want = m.ops.gather_qmm(x, q.reshape(experts, 16, -1), s.reshape(experts, 16, -1), b.reshape(experts, 16, -1), rhs_indices=e)
    least = need.value - (full.value - 512)
    y, ws = torch.empty_like(want), torch.empty(least, dtype=torch.uint8, device="cuda")

    def gather(size):
        return lib.mi_moe_gather_qmm(x.data_ptr(), q.data_ptr(), s.data_ptr(), b.data_ptr(), None, e.data_ptr(), pairs, pairs, 1, 16, 128, experts, 1, 64, 4, 0,
                                     y.data_ptr(), ws.data_ptr(), size, st)
    assert gather(least) == 0 and torch.equal(y, want)
    assert gather(least - 1) != 0 and b"workspace too small" in lib.mi_moe_last_error()


# all segments in pieces, pieces beside streamed segments; short segments beside tiles (8-bit codes), all in tiles
@pytest.mark.parametrize("hidden,inter,experts,k,tokens,bits,group", [(256, 1152, 8, 4, 150, 4, 64), (256, 512, 8, 4, 1100, 4, 64), (256, 512, 8, 2, 100, 8, 32),
                                                                      (256, 512, 8, 2, 600, 4, 32), (256, 512, 8, 2, 600, 8, 128)])
def test_blocks_in_a_workspace_without_the_group_sums(hidden, inter, experts, k, tokens, bits, group):
    """A workspace one byte short of the group sums is taken as well, by kernels that need none; the bound is test_blocks_in_short_tiles' and, for weights that
    are rounded to bfloat16 on the way, once more 0.42 of 2^-8 for each product."""
    import mlx_rs_amd as m
    from mlx_rs_amd import synth
    lib = m.load_library()
    cfg = m.MoeConfig(hidden, experts, k, inter, bits, group, 0)
    blk = synth.make_block(cfg, seed=3, device="cuda", zipf_s=0.7, gen_device="cuda")
    x = synth.make_tokens(cfg, tokens, seed=3, device="cuda")
    want, routing = blk.forward(x, debug=True)
    planes = C.c_size_t()
    m.capi.check(lib.mi_moe_router_logits_workspace_size(tokens, hidden, experts, C.byref(planes)))
    size = blk.workspace_bytes(tokens) - planes.value - 1
    ws, out = torch.empty(size, dtype=torch.uint8, device="cuda"), torch.empty_like(x)
    st = torch.cuda.current_stream().cuda_stream
    m.capi.check(lib.mi_moe_forward(blk._handle, x.data_ptr(), tokens, out.data_ptr(), ws.data_ptr(), size, None, st))
    ref = block_truth(blk, x, routing)
    assert float((out.double() - ref).norm() / ref.norm()) <= 1.5 * 2.0 ** -8
    assert not torch.equal(out, want)  # (other kernels: another order of the sums)
