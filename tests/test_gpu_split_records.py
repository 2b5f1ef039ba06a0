"""Batches whose segments all stream: a segment longer than a pass is several work records."""
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

from test_gpu_codes import block_truth  # noqa: E402
from test_gpu_short_pieces import chosen_block  # noqa: E402


@pytest.mark.parametrize("bits,group", [(4, 64), (8, 64), (4, 32), (8, 128)])
@pytest.mark.parametrize("lengths", [
    [9, 8, 17, 1, 16, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0],  # up to 64 tokens: the router's own dispatch
    [33, 0, 0, 0, 0, 31] + 18 * [0],
    [7, 8, 9, 15, 16, 17, 24, 25, 33, 1] + 62 * [0],  # a dispatch of its own, records past a wave of experts
])
def test_segments_of_several_records(lengths, bits, group):
    """Roundings to bfloat16 of h, y and the result, each typically 0.42 * 2^-8 of its values: 0.73 * 2^-8 together; a row's bound is twice that.  A row's result depends neither on its place
    nor on the other rows of its record."""
    blk, x, of = chosen_block(256, 384, lengths, len(lengths), bits, group)
    out, routing = blk.forward(x, debug=True)
    assert torch.equal(routing["topk_idx"][:, 0].long(), of)
    ref = block_truth(blk, x, routing)
    err = (out.double() - ref).norm(dim=1) / ref.norm(dim=1)
    assert float(err.max()) <= 1.5 * 2.0 ** -8, float(err.max())
    order = torch.randperm(len(of), generator=torch.Generator().manual_seed(3)).cuda()
    assert torch.equal(blk.forward(x[order].contiguous()), out[order])
