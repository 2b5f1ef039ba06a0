"""Pieces of up to 128 rows with 8-bit codes in groups of 64, against float64."""
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

from test_gpu_codes import block_truth  # noqa: E402
from test_gpu_short_pieces import chosen_block  # noqa: E402

EDGES = [0, 1, 16, 17, 31, 32, 33, 63, 64, 65, 95, 96, 97, 127, 128, 129, 145, 257]  # both sides of every length at which another kernel, body or piece begins


# K of 1, 2, 3, 8, 9 and 17 times 128 values: windows of 512 whole and started; 18 experts and few columns: K shared by two groups of waves where it is whole 256s, blocks of 128 columns;
# many columns: one group; output columns that fill no block of 256
@pytest.mark.parametrize("hidden,inter,experts", [(128, 384, 18), (384, 128, 18), (256, 512, 18), (1024, 1152, 18), (1152, 1024, 18), (2176, 256, 36), (256, 2176, 36), (768, 768, 90)])
def test_lengths_around_every_body_b(hidden, inter, experts):
    """Roundings to bfloat16 of the weights of three products, h, y and the result, each typically 0.42 * 2^-8 of its values: 1.03 * 2^-8 together; a row's bound is twice
    that.  Rows do not depend on their order in the batch."""
    check(hidden, inter, EDGES, experts)


def test_as_many_blocks_as_cus():
    """32 pieces at most by eight blocks of 256 columns: K shared by two groups of waves of 64 columns each."""
    check(2048, 256, [45, 30, 60], 24)


def check(hidden, inter, lengths, experts):
    blk, x, of = chosen_block(hidden, inter, lengths, experts, 8, 64)
    out, routing = blk.forward(x, debug=True)
    assert torch.equal(routing["topk_idx"][:, 0].long(), of)
    ref = block_truth(blk, x, routing)
    err = (out.double() - ref).norm(dim=1) / ref.norm(dim=1)
    assert float(err.max()) <= 2.06 * 2.0 ** -8, float(err.max())
    order = torch.randperm(len(of), generator=torch.Generator().manual_seed(3)).cuda()
    assert torch.equal(blk.forward(x[order].contiguous()), out[order])


@pytest.mark.parametrize("tokens,zipf", [(150, 1.0), (400, None)])
def test_infinities_of_long_pieces(tokens, zipf):
    """Infinite biases of each matrix and rows that are not finite."""
    import mlx_rs_amd as m
    from mlx_rs_amd import synth
    cfg = m.MoeConfig(256, 16, 6, 384, 8, 64, 0)
    blk = synth.make_block(cfg, seed=2, device="cuda", zipf_s=zipf, gen_device="cuda")
    x = synth.make_tokens(cfg, tokens, seed=1, device="cuda")
    blk.gate_proj.biases[1, 5, 1] = float("inf")
    blk.up_proj.biases[2, 7, 0] = float("-inf")
    blk.down_proj.biases[3, 9, 1] = float("inf")
    x[7, 3] = float("inf")
    x[11, 200] = float("nan")
    blk.gate_weight[:, 3] = blk.gate_weight[:, 200] = 0.0
    finite = torch.ones(tokens, dtype=torch.bool, device="cuda")
    finite[[7, 11]] = False  # (the routing of these is no number's)
    out, routing = blk.forward(x, debug=True)
    ref = block_truth(blk, x, routing)
    assert not ref[finite].isfinite().all()
    assert torch.equal(out[finite].isnan(), ref[finite].isnan()) and torch.equal(out[finite].isinf(), ref[finite].isinf())


FEW = [0, 1, 15, 16, 17, 31, 32, 33, 47, 48, 49, 63, 64, 65] + 10 * [0]  # twenty rows an expert on average


@pytest.mark.parametrize("hidden,inter", [(128, 384), (384, 128), (1024, 1152), (1152, 1024), (2176, 256), (256, 2176)])
def test_all_segments_of_a_few_rows_in_pieces(hidden, inter):
    """From fourteen to 24 rows an expert (six where the down product has a block for every CU): raw codes, so three roundings to bfloat16 (h, y and the result), each typically 0.42 * 2^-8 of its values: 0.73 * 2^-8 together; a
    row's bound is twice that."""
    import mlx_rs_amd as m
    blk, x, of = chosen_block(hidden, inter, FEW, 24, 8, 64)
    assert m.capi.tile_rule(blk.config.c_struct(), len(of)) == (2, 1)
    out, routing = blk.forward(x, debug=True)
    assert torch.equal(routing["topk_idx"][:, 0].long(), of)
    ref = block_truth(blk, x, routing)
    err = (out.double() - ref).norm(dim=1) / ref.norm(dim=1)
    assert float(err.max()) <= 1.5 * 2.0 ** -8, float(err.max())
    order = torch.randperm(len(of), generator=torch.Generator().manual_seed(3)).cuda()
    assert torch.equal(blk.forward(x[order].contiguous()), out[order])


@pytest.mark.parametrize("tokens", [57, 64, 65])
@pytest.mark.parametrize("residual", [False, True])
def test_few_rows_behind_either_router(tokens, residual):
    """Up to 64 tokens the router is one launch and the rows are prepared behind it; the same bits with a workspace that a larger batch has left."""
    import mlx_rs_amd as m
    from mlx_rs_amd import synth
    cfg = m.MoeConfig(512, 8, 2, 384, 8, 64, 0)
    assert m.capi.tile_rule(cfg.c_struct(), tokens) == (2, 1)
    blk = synth.make_block(cfg, seed=6, device="cuda", zipf_s=1.1, gen_device="cuda")
    x = synth.make_tokens(cfg, tokens, seed=6, device="cuda")
    if residual:
        w = torch.ones(512, dtype=torch.bfloat16, device="cuda")
        out = blk.forward_residual(x, w, 1e-6)
        blk.forward_residual(synth.make_tokens(cfg, 700, seed=7, device="cuda"), w, 1e-6)
        assert torch.equal(blk.forward_residual(x, w, 1e-6), out)
        n = m.ops.rms_norm(x, w, 1e-6)
        got, ref = out.double(), x.double() + blk.forward(n).double()
        assert float((got - ref).norm() / ref.norm()) <= 2.0 ** -8  # (one rounding for two)
    else:
        out, routing = blk.forward(x, debug=True)
        blk.forward(synth.make_tokens(cfg, 700, seed=7, device="cuda"))
        assert torch.equal(blk.forward(x), out)
        ref = block_truth(blk, x, routing)
        err = (out.double() - ref).norm(dim=1) / ref.norm(dim=1)
        assert float(err.max()) <= 1.5 * 2.0 ** -8, float(err.max())


# records of a pass; pieces of all segments; pieces beside streamed segments
ROUTES = [(256, 512, 32, 4, 40, 4, 1.3), (512, 384, 8, 2, 60, 8, 1.1), (256, 512, 8, 2, 70, 8, 1.1), (512, 512, 16, 4, 150, 8, 0.7)]


@pytest.mark.parametrize("hidden,inter,experts,k,tokens,bits,zipf", ROUTES)
def test_graph_replays_of_these_routes(hidden, inter, experts, k, tokens, bits, zipf):
    import mlx_rs_amd as m
    from mlx_rs_amd import synth
    blk = synth.make_block(m.MoeConfig(hidden, experts, k, inter, bits, 64, 0), seed=9, device="cuda", zipf_s=zipf, gen_device="cuda")
    x, other = synth.make_tokens(blk.config, tokens, seed=9, device="cuda"), synth.make_tokens(blk.config, 7, seed=10, device="cuda")
    blk.reserve(tokens)
    eager, out = blk.forward(x).clone(), torch.empty_like(x)
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        blk.forward(x, out=out)
    torch.cuda.current_stream().wait_stream(s)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        blk.forward(x, out=out)
    for rep in range(4):
        out.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(out.view(torch.int16), eager.view(torch.int16)), rep
        blk.forward(other)
        torch.cuda.synchronize()


@pytest.mark.parametrize("hidden,inter,experts,k,tokens,bits,zipf", ROUTES[:3])
def test_these_routes_in_a_workspace_without_their_share(hidden, inter, experts, k, tokens, bits, zipf):
    """A workspace one byte short of what the route adds is taken by the kernels that need none: streamed segments in one record each have the same bits; else the bound is that of six
    roundings to bfloat16, 1.03 * 2^-8 typically and twice that for a row."""
    import ctypes as C

    import mlx_rs_amd as m
    from mlx_rs_amd import synth
    lib = m.load_library()
    blk = synth.make_block(m.MoeConfig(hidden, experts, k, inter, bits, 64, 0), seed=9, device="cuda", zipf_s=zipf, gen_device="cuda")
    x = synth.make_tokens(blk.config, tokens, seed=9, device="cuda")
    want, routing = blk.forward(x, debug=True)
    planes = C.c_size_t()
    m.capi.check(lib.mi_moe_router_logits_workspace_size(tokens, hidden, experts, C.byref(planes)))
    size = blk.workspace_bytes(tokens) - (planes.value if tokens > 64 else 0) - 256 - 1
    ws, out = torch.empty(size, dtype=torch.uint8, device="cuda"), torch.empty_like(x)
    m.capi.check(lib.mi_moe_forward(blk._handle, x.data_ptr(), tokens, out.data_ptr(), ws.data_ptr(), size, None, torch.cuda.current_stream().cuda_stream))
    if bits == 4:
        assert torch.equal(out, want)
    ref = block_truth(blk, x, routing)
    assert float(((out.double() - ref).norm(dim=1) / ref.norm(dim=1)).max()) <= 2.06 * 2.0 ** -8
