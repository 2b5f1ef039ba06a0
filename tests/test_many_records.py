"""More segments of a pass than a launch has rows of blocks: longer records."""
import pytest

# hidden of an odd number of groups of 64, or an intermediate size that is no multiple of 128: layers without tiles, whose batches of any size stream
LAYERS = [(2048, 128, 8, 704, 8, 64), (192, 2, 2, 64, 8, 64), (192, 512, 32, 64, 8, 64)]


@pytest.mark.parametrize("hidden,experts,k,inter,bits,group", LAYERS)
@pytest.mark.parametrize("pairs", [1 << 10, 1 << 20, (1 << 20) + (1 << 13), 1 << 21, 1 << 26, 1 << 30])
def test_the_records_of_a_launch_fit_its_grid(hidden, experts, k, inter, bits, group, pairs):
    import mlx_rs_amd as m
    m.load_library()
    plan = m.capi.plan_forward(m.capi.Config(hidden, experts, k, inter, bits, group, 0), pairs // k)
    assert len(plan) == 2
    for name, info in plan:
        gx, gy = (int(v) for v in info["grid"].split("x"))
        assert 1 <= gx and 1 <= gy <= 65535, (name, info)


@pytest.mark.gpu
@pytest.mark.parametrize("bits,group", [(8, 64), (4, 32)])
def test_a_batch_of_longer_records(bits, group):
    """1.1 million rows, seventy thousand passes of sixteen.  Roundings to bfloat16 of h, y and the result, each typically 0.42 * 2^-8 of its values: 0.73 * 2^-8 together; the bound for 4000
    rows is twice that, which a single row of another one's values or of none would break by far."""
    import torch

    import mlx_rs_amd as m
    from mlx_rs_amd import synth
    from test_gpu_codes import block_truth
    cfg, tokens = m.MoeConfig(192, 2, 2, 64, bits, group, 0), 560_000
    blk = synth.make_block(cfg, seed=8, device="cuda", gen_device="cuda")
    x = synth.make_tokens(cfg, tokens, seed=8, device="cuda")
    out, routing = blk.forward(x, debug=True)
    for at in range(0, tokens, 4000):
        part = slice(at, at + 4000)
        ref = block_truth(blk, x[part], {n: routing[n][part] for n in ("topk_idx", "topk_w")})
        err = (out[part].double() - ref).norm(dim=1) / ref.norm()
        assert float(err.norm()) <= 1.5 * 2.0 ** -8, at
