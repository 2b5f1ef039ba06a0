"""A workspace sized for a layer's largest batch gives every smaller one what it takes in a workspace of its own."""
import ctypes as C

import pytest

# hidden, experts, k, intermediate: whole and ragged, few and many experts, one and all of them a token
SHAPES = [(2048, 128, 8, 768), (2048, 16, 8, 1408), (2048, 8, 4, 14336), (4096, 8, 2, 14336), (2304, 64, 2, 6400), (128, 512, 32, 128), (3200, 8, 8, 1792), (1280, 64, 1, 6272), (256, 4, 2, 384)]


@pytest.mark.parametrize("bits,group", [(b, g) for b in (2, 4, 8) for g in (32, 64, 128)])
@pytest.mark.parametrize("hidden,experts,k,inter", SHAPES)
def test_the_workspace_grows_with_the_batch(hidden, experts, k, inter, bits, group):
    import mlx_rs_amd as m
    lib = m.load_library()
    cfg, need, most = m.capi.Config(hidden, experts, k, inter, bits, group, 0), C.c_size_t(), 0
    # up to 200 rows an expert, beyond every line between routes; then to operands past 2 GiB
    dense = 200 * experts // k
    step = max(1, dense // 1500)
    near = {rows * experts // k + d for rows in (4, 6, 14, 20, 24, 32, 48, 60, 80, 96, 176) for d in (-1, 0, 1)}
    for tokens in sorted(set(range(1, dense, step)) | {t for t in near if t > 0} | set(range(dense, 60000, 601))):
        m.capi.check(lib.mi_moe_workspace_size(C.byref(cfg), tokens, C.byref(need)))
        assert need.value >= most, tokens
        most = need.value


@pytest.mark.gpu
@pytest.mark.parametrize("hidden,experts,k,inter,tokens,reserved", [(2048, 16, 8, 1408, 47, 48), (2048, 8, 4, 14336, 44, 48), (256, 8, 2, 512, 95, 96)])
def test_a_smaller_batch_in_a_reserved_workspace(hidden, experts, k, inter, tokens, reserved):
    """8-bit codes in groups of 64: twenty-four rows an expert are reserved, some fewer are run on other kernels, whose regions the larger batch does without."""
    import torch

    import mlx_rs_amd as m
    from mlx_rs_amd import synth
    blk = synth.make_block(m.MoeConfig(hidden, experts, k, inter, 8, 64, 0), seed=3, device="cuda", gen_device="cuda")
    assert m.capi.tile_rule(blk.config.c_struct(), tokens) == (2, 1) and m.capi.tile_rule(blk.config.c_struct(), reserved)[0] != 2
    x = synth.make_tokens(blk.config, tokens, seed=3, device="cuda")
    blk.reserve(tokens)
    own = blk.forward(x)
    blk.reserve(reserved)
    assert torch.equal(blk.forward(x).view(torch.int16), own.view(torch.int16))
