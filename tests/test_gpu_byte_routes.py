"""8-bit codes in groups of 64: results that are not finite on the pieces of a few rows, and that the pieces' kernels are what runs."""
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

from test_gpu_codes import block_truth  # noqa: E402
from test_gpu_short_pieces import chosen_block  # noqa: E402


# fourteen to 24 rows an expert: all segments on raw codes, either router; bodies of 16 to 64 rows
@pytest.mark.parametrize("tokens,k,zipf", [(60, 6, 1.0), (40, 6, None), (90, 4, 0.5), (75, 4, 1.3)])
def test_infinities_of_a_few_rows(tokens, k, zipf):
    """Infinite scales and biases of each matrix, and rows that are not finite."""
    import mlx_rs_amd as m
    from mlx_rs_amd import synth
    cfg = m.MoeConfig(256, 16, k, 384, 8, 64, 0)
    assert m.capi.tile_rule(cfg.c_struct(), tokens) == (2, 1)
    blk = synth.make_block(cfg, seed=2, device="cuda", zipf_s=zipf, gen_device="cuda")
    x = synth.make_tokens(cfg, tokens, seed=1, device="cuda")
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


def test_sums_of_bytes_that_overflow():
    """An activation of 3e38 against weights of a code times 2^-129: the sum of its codes is infinite, the product of the dequantised weights is not.  One row of each sixteen of every piece.  The
    scale keeps no more than four bits, h and the result round three times: 2^-6, as the pieces of other groups."""
    import mlx_rs_amd as m
    blk, x, of = chosen_block(384, 256, [40, 64, 20, 16, 0, 1, 17, 33, 0, 7, 49, 12], 24, 8, 64)
    assert m.capi.tile_rule(blk.config.c_struct(), len(of)) == (2, 1)
    blk.gate_weight.copy_(torch.eye(384)[128:152])
    blk.gate_weight[:, 7] = 0.0
    x[torch.arange(len(of), device="cuda"), 128 + of] = 16.0
    for bank in (blk.gate_proj, blk.up_proj):
        bank.scales[:, :, 0] = 2.0 ** -129
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


# K shared by two groups of waves in blocks of 128 columns, of 256, and not shared
@pytest.mark.parametrize("hidden,inter,experts,lengths", [(1024, 1152, 18, [0, 1, 16, 17, 33, 63, 65, 97, 129]), (2048, 256, 24, [45, 30, 60]), (256, 2176, 36, [5, 40, 70, 145])])
def test_the_kernel_of_long_pieces_is_what_runs(hidden, inter, experts, lengths):
    """A batch whose tile lists would be built, if its segments did not go in pieces: one launch of those a product, beside the streamed one, and none of a list of tiles."""
    import mlx_rs_amd as m
    blk, x, _ = chosen_block(hidden, inter, lengths, experts, 8, 64)
    assert m.capi.tile_rule(blk.config.c_struct(), x.shape[0])[0] == 1
    out, _, kernels = blk.forward_timed(x, kernels=True)
    assert [t > 0.0 for t in kernels] == 2 * [False, False, True, True]
    assert torch.equal(out, blk.forward(x))
