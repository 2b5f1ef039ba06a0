"""Pieces of up to 64 rows: blocks with 4-bit codes in groups of 64 and up to sixty rows an expert on average, and with groups of 32 and 128, against float64."""
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

from test_gpu_codes import block_truth, product  # noqa: E402
from test_gpu_short_tiles import share_off_nearest  # noqa: E402

EDGES = [0, 1, 15, 16, 17, 31, 32, 33, 47, 48, 49, 63, 64, 65]  # lengths on both sides of every one at which another body or another piece begins


def chosen_block(hidden, inter, lengths, experts, bits, group):
    """A block whose expert e gets lengths[e % len(lengths)] tokens: the expert's column of a token is large, and the router is the unit matrix."""
    import mlx_rs_amd as m
    from mlx_rs_amd import synth
    cfg = m.MoeConfig(hidden, experts, 1, inter, bits, group, 0)
    blk = synth.make_block(cfg, seed=4, device="cuda", gen_device="cuda")
    blk.gate_weight.copy_(torch.eye(hidden)[:experts])
    of = torch.cat([torch.full((lengths[e % len(lengths)],), e) for e in range(experts)]).cuda()
    tokens = of.numel()
    of = of[torch.randperm(tokens, generator=torch.Generator().manual_seed(1)).cuda()]
    x = synth.make_tokens(cfg, tokens, seed=4, device="cuda")
    x[torch.arange(tokens, device="cuda"), of] = 16.0
    return blk, x, of


def chosen(hidden, inter, lengths, experts, bits=4, group=64):
    import mlx_rs_amd as m
    blk, x, of = chosen_block(hidden, inter, lengths, experts, bits, group)
    tokens = of.numel()
    assert max(512, 6 * experts) <= tokens < 60 * experts and (group != 64 or m.capi.tile_rule(blk.config.c_struct(), tokens) == (2, 1))
    return blk, x, of


# K of 1, 3, 8, 9 and 17 times 128 values: windows of 256, 512 and 1024, whole and started, rows of an odd number of groups of 128; output columns that fill no
# block of 256
@pytest.mark.parametrize("hidden,inter", [(128, 384), (384, 128), (1024, 1152), (1152, 1024), (2176, 256), (256, 2176)])
@pytest.mark.parametrize("bits,group", [(4, 64), (4, 32), (4, 128), (8, 32), (8, 128)])
def test_lengths_around_every_body_s(hidden, inter, bits, group):
    """Three roundings to bfloat16 (h, y and the result), each at most 2^-8 of its values and typically 0.42 of that: 0.73 * 2^-8 together; a row's bound is twice
    that.  A row's result does not depend on its place in a piece, or on the piece's length: without one expert's tokens the others' are the same bits."""
    blk, x, of = chosen(hidden, inter, EDGES, 42, bits, group)
    out, routing = blk.forward(x, debug=True)
    assert torch.equal(routing["topk_idx"][:, 0].long(), of)
    ref = block_truth(blk, x, routing)
    err = (out.double() - ref).norm(dim=1) / ref.norm(dim=1)
    assert float(err.max()) <= 1.5 * 2.0 ** -8, float(err.max())
    keep = torch.ones_like(of, dtype=torch.bool)
    keep[::3] = False
    assert int(keep.sum()) >= 512
    assert torch.equal(blk.forward(x[keep].contiguous()), out[keep])


@pytest.mark.parametrize("bits,group", [(4, 64), (4, 32), (4, 128), (8, 32), (8, 128)])
@pytest.mark.parametrize("tokens,zipf", [(150, 1.0), (100, None), (120, 0.5)])
def test_results_that_are_not_finite(tokens, zipf, bits, group):
    """Infinite scales and biases of each matrix, in pieces of every body; h's as well as the down product's own."""
    import mlx_rs_amd as m
    from mlx_rs_amd import synth
    cfg = m.MoeConfig(256, 16, 6, 384, bits, group, 0)
    blk = synth.make_block(cfg, seed=2, device="cuda", zipf_s=zipf, gen_device="cuda")
    x = synth.make_tokens(cfg, tokens, seed=1, device="cuda")
    assert group != 64 or (m.capi.tile_rule(cfg.c_struct(), tokens) == (2, 1)) is True
    blk.gate_proj.biases[1, 5, 1] = float("inf")
    blk.up_proj.biases[2, 7, 0] = float("-inf")
    blk.down_proj.scales[3, 9, 1] = float("inf")
    x[7, 3] = float("inf")
    x[11, 200] = float("nan")
    blk.gate_weight[:, 3] = blk.gate_weight[:, 200] = 0.0
    finite = torch.ones(tokens, dtype=torch.bool, device="cuda")
    finite[[7, 11]] = False  # (the routing of these is no number's)
    out, routing = blk.forward(x, debug=True)
    ref = block_truth(blk, x, routing)
    assert not ref[finite].isfinite().all()
    assert torch.equal(out[finite].isnan(), ref[finite].isnan()) and torch.equal(out[finite].isinf(), ref[finite].isinf())


@pytest.mark.parametrize("bits,group", [(4, 64), (4, 32), (4, 128), (8, 32), (8, 128)])
def test_sums_of_codes_that_overflow(bits, group):
    """An activation of 3e38 against weights of a code times 2^-125 (2^-129 with 8 bits): the sum of its codes is infinite, the product of the dequantised weights is not.  One row
    of each sixteen of every piece."""
    blk, x, of = chosen(384, 256, [40, 64, 20, 16, 30, 55], 24, bits, group)
    blk.gate_weight.copy_(torch.eye(384)[128:152])
    blk.gate_weight[:, 7] = 0.0
    x[torch.arange(len(of), device="cuda"), 128 + of] = 16.0
    for bank in (blk.gate_proj, blk.up_proj):
        bank.scales[:, :, 0] = 2.0 ** (-125 if bits == 4 else -129)
        bank.biases[:, :, 0] = 0.0
    _, routing = blk.forward(x, debug=True)
    perm, offsets = routing["perm"].long(), routing["offsets"].tolist()
    hit = [r for e in range(24) for r in range(offsets[e] + 5, offsets[e + 1], 16)]
    rows = perm[torch.tensor(hit, device="cuda")]
    x[rows, 7] = 3e38
    out, routing = blk.forward(x, debug=True)
    ref = block_truth(blk, x, routing)
    assert bool(ref.isfinite().all()) and float(ref[rows].norm(dim=1).min()) > 10 * float(ref.norm(dim=1).median())
    err = (out.double() - ref).norm(dim=1) / ref.norm(dim=1)
    assert float(err.max()) <= 2.0 ** -6, float(err.max())


@pytest.mark.parametrize("bits,group", [(4, 32), (4, 128), (8, 32), (8, 128)])
def test_what_the_sums_lose(bits, group):
    """Groups of 32 and 128, one expert a token, whose score is 1.  A gate of 64, whose SiLU is 64, and up the unit matrix, around the centre of the codes, make h = 64 x exactly, so the result is
    the down product's.  The bound is plain sums', 2^-22 of the results' root mean square: codes around their centre, or sums that start from the centre's share
    and end as those do."""
    import mlx_rs_amd as m
    from mlx_rs_amd import synth
    n, experts, tokens = 2048, 8, 300
    cfg = m.MoeConfig(n, experts, 1, n, bits, group, 0)
    blk = synth.make_block(cfg, seed=5, device="cuda", zipf_s=0.5, gen_device="cuda")
    for bank, column, value in ((blk.gate_proj, torch.zeros(n, dtype=torch.int64), 64.0), (blk.up_proj, torch.arange(n), 1.0)):
        mid, per = 1 << (bits - 1), 32 // bits
        codes = torch.full((n, n), mid, dtype=torch.int64)
        codes[torch.arange(n), column] += 1
        words = (codes.reshape(n, -1, per) << (bits * torch.arange(per))).sum(-1)
        bank.weight.copy_(words.to(torch.int32).expand_as(bank.weight))
        bank.scales.fill_(value)
        bank.biases.fill_(-mid * value)  # (a bias term of zero)
    x = synth.make_tokens(cfg, tokens, seed=5, device="cuda")
    x[:, 0] = 1.0
    out, routing = blk.forward(x, debug=True)
    assert bool((routing["topk_w"] == 1).all())
    ref = torch.empty((tokens, n), dtype=torch.float64, device="cuda")
    for e in range(experts):
        hit = routing["topk_idx"][:, 0] == e
        ref[hit] = product(64 * x[hit], blk.down_proj.weight[e], blk.down_proj.scales[e], blk.down_proj.biases[e], group, bits)
    share, allowed = share_off_nearest(out, ref, 2.0 ** -22 * ref.square().mean().sqrt())
    assert share <= allowed, (share, allowed)
