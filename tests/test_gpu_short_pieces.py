"""Pieces of up to 64 rows of blocks with 4-bit codes in groups of 64 and up to sixty rows an expert on average, against float64."""
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

from test_gpu_codes import block_truth  # noqa: E402

EDGES = [0, 1, 15, 16, 17, 31, 32, 33, 47, 48, 49, 63, 64, 65]  # lengths on both sides of every one at which another body or another piece begins


def chosen(hidden, inter, lengths, experts):
    """A block whose expert e gets lengths[e % len(lengths)] tokens: the expert's column of a token is large, and the router is the unit matrix."""
    import mlx_rs_amd as m
    from mlx_rs_amd import synth
    cfg = m.MoeConfig(hidden, experts, 1, inter, 4, 64, 0)
    blk = synth.make_block(cfg, seed=4, device="cuda", gen_device="cuda")
    blk.gate_weight.copy_(torch.eye(hidden)[:experts])
    of = torch.cat([torch.full((lengths[e % len(lengths)],), e) for e in range(experts)]).cuda()
    tokens = of.numel()
    assert max(512, 6 * experts) <= tokens < 60 * experts and m.capi.tile_rule(cfg.c_struct(), tokens) == (2, 1)
    of = of[torch.randperm(tokens, generator=torch.Generator().manual_seed(1)).cuda()]
    x = synth.make_tokens(cfg, tokens, seed=4, device="cuda")
    x[torch.arange(tokens, device="cuda"), of] = 16.0
    return blk, x, of


# K of 1, 3, 8 (a window), 9 and 17 (two windows and one) stages of 128 values, output columns that fill no block of 256
@pytest.mark.parametrize("hidden,inter", [(128, 384), (384, 128), (1024, 1152), (1152, 1024), (2176, 256), (256, 2176)])
def test_lengths_around_every_body_s(hidden, inter):
    """Three roundings to bfloat16 (h, y and the result), each at most 2^-8 of its values and typically 0.42 of that: 0.73 * 2^-8 together; a row's bound is twice
    that.  A row's result does not depend on its place in a piece, or on the piece's length: without one expert's tokens the others' are the same bits."""
    blk, x, of = chosen(hidden, inter, EDGES, 42)
    out, routing = blk.forward(x, debug=True)
    assert torch.equal(routing["topk_idx"][:, 0].long(), of)
    ref = block_truth(blk, x, routing)
    err = (out.double() - ref).norm(dim=1) / ref.norm(dim=1)
    assert float(err.max()) <= 1.5 * 2.0 ** -8, float(err.max())
    keep = torch.ones_like(of, dtype=torch.bool)
    keep[::3] = False
    assert int(keep.sum()) >= 512
    assert torch.equal(blk.forward(x[keep].contiguous()), out[keep])


@pytest.mark.parametrize("tokens,zipf", [(200, 1.0), (100, None), (150, 0.5)])
def test_results_that_are_not_finite(tokens, zipf):
    """Infinite scales and biases of each matrix, in pieces of every body; h's as well as the down product's own."""
    import mlx_rs_amd as m
    from mlx_rs_amd import synth
    cfg = m.MoeConfig(256, 16, 6, 384, 4, 64, 0)
    blk = synth.make_block(cfg, seed=2, device="cuda", zipf_s=zipf, gen_device="cuda")
    x = synth.make_tokens(cfg, tokens, seed=1, device="cuda")
    assert m.capi.tile_rule(cfg.c_struct(), tokens) == (2, 1) and tokens * 6 < 60 * 16 + 300
    blk.gate_proj.biases[1, 5, 2] = float("inf")
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


def test_sums_of_codes_that_overflow():
    """An activation of 3e38 against weights of up to fifteen 2^-125: the sum of its codes is infinite, the product of the dequantised weights is not.  One row
    of each sixteen of every piece."""
    blk, x, of = chosen(256, 384, [40, 64, 20, 16, 30, 55], 24)
    blk.gate_weight.copy_(torch.eye(256)[64:88])
    blk.gate_weight[:, 7] = 0.0
    x[torch.arange(len(of), device="cuda"), 64 + of] = 16.0
    for bank in (blk.gate_proj, blk.up_proj):
        bank.scales[:, :, 0] = 2.0 ** -125
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
