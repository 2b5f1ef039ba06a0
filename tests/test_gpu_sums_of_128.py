"""Blocks with groups of 128: what the sums of pieces lose."""
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def centred_sums(x, codes, s, b, bits, group=128):
    """x [rows, K], codes [N, K]: sums of centred codes as float32 holds them, two steps of 32 values for each 64, scaled and added up; then the bias term with the centre's share, rounded once for 1024
    values.  Every step is exact but for its one rounding."""
    mid = 1 << (bits - 1)
    total = torch.zeros((x.shape[0], codes.shape[0]), dtype=torch.float64, device=x.device)
    for k in range(0, x.shape[1], 64):
        part = (x[:, k:k + 32] @ (codes[:, k:k + 32] - mid).t()).float().double()
        part = (part + x[:, k + 32:k + 64] @ (codes[:, k + 32:k + 64] - mid).t()).float().double()
        total = (total + part * s[:, k // group]).float().double()
        if k % 1024 == 960:
            g = slice((k - 960) // group, (k + 64) // group)
            sums = x[:, k - 960:k + 64].reshape(x.shape[0], -1, group).sum(2)
            total = (total + sums @ (b[:, g] + mid * s[:, g]).t()).float().double()
    return total


@pytest.mark.parametrize("bits", [4, 8])
def test_groups_of_128_lose_what_sums_of_centred_codes_do(bits):
    """One expert a token, whose score is 1; a gate of 64, whose SiLU is 64, and up the unit matrix make h = 64 x exactly, so the result is the down product's.  The share of results that are not
    the nearest value, against that of the same sums made step by step: a quarter more is allowed, a tenth for the order of the products inside a matrix instruction and three times what counts
    of a thousand differ by.  (Codes without their centre make sums several times their result on the way: 1.5 times the share.)"""
    import mlx_rs_amd as m
    from mlx_rs_amd import synth
    n, experts, tokens, mid, per = 4096, 8, 2000, 1 << (bits - 1), 32 // bits
    blk = synth.make_block(m.MoeConfig(n, experts, 1, n, bits, 128, 0), seed=5, device="cuda", zipf_s=0.5, gen_device="cuda")
    for bank, column, value in ((blk.gate_proj, torch.zeros(n, dtype=torch.int64), 64.0), (blk.up_proj, torch.arange(n), 1.0)):
        codes = torch.full((n, n), mid, dtype=torch.int64)
        codes[torch.arange(n), column] += 1
        bank.weight.copy_((codes.reshape(n, -1, per) << (bits * torch.arange(per))).sum(-1).to(torch.int32).expand_as(bank.weight))
        bank.scales.fill_(value)
        bank.biases.fill_(-mid * value)  # (a bias term of zero)
    x = synth.make_tokens(blk.config, tokens, seed=5, device="cuda")
    x[:, 0] = 1.0
    out, routing = blk.forward(x, debug=True)
    assert bool((routing["topk_w"] == 1).all())
    shift, off, allowed = torch.arange(per, device="cuda") * bits, 0, 0
    for e in range(experts):
        hit, bank = routing["topk_idx"][:, 0] == e, blk.down_proj
        codes = ((bank.weight[e].long() & 0xFFFFFFFF).unsqueeze(-1) >> shift & ((1 << bits) - 1)).reshape(n, n).double()
        s, b, rows = bank.scales[e].double(), bank.biases[e].double(), 64 * x[hit].double()
        ref = (rows @ (codes * s.repeat_interleave(128, 1) + b.repeat_interleave(128, 1)).t()).to(torch.bfloat16)
        off += int((out[hit] != ref).sum())
        allowed += int((centred_sums(rows, codes, s, b, bits).to(torch.bfloat16) != ref).sum())
    assert off <= 1.25 * allowed, (off, allowed)
