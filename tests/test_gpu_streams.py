"""Forwards that use the device's side streams while those belong to a capture."""
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


# groups of 32: tiles beside the short segments, with their codes in LDS and in registers; groups of 64: 64-row tiles on raw codes (no side stream),
# heavy batches with an average segment of the 128- and the 256-row class, a light batch, and one whose average segment is the 64-row class's
@pytest.mark.parametrize("group,tokens,experts,k", [(32, 200, 16, 4), (32, 50, 16, 4), (64, 200, 16, 4), (64, 400, 16, 4), (64, 1600, 16, 4), (64, 75, 16, 4), (64, 100, 4, 2)])
def test_a_forward_beside_another_streams_capture(group, tokens, experts, k):
    """Between the begin and the end of a capture the side streams stay in it.  A forward on another stream meanwhile runs at once, and
    the captured one is what an eager one gives."""
    import mlx_rs_amd as m
    from mlx_rs_amd import synth
    cfg = m.MoeConfig(512, experts, k, 256, 4, group, 0)
    one, other = (synth.make_block(cfg, seed=s, device="cuda", zipf_s=1.1, gen_device="cuda") for s in (1, 2))
    x = synth.make_tokens(cfg, tokens, seed=3, device="cuda")
    want_one, want_other = one.forward(x), other.forward(x)
    got_other = torch.empty_like(want_other)
    beside, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph, capture_error_mode="relaxed"):
        got_one = one.forward(x)
        with torch.cuda.stream(beside):
            other.forward(x, out=got_other)
        beside.synchronize()
        assert torch.cuda.is_current_stream_capturing()
    assert torch.equal(got_other, want_other)
    for _ in range(3):
        got_one.zero_()
        graph.replay()
        other.forward(x, out=got_other)
        torch.cuda.synchronize()
        assert torch.equal(got_one, want_one) and torch.equal(got_other, want_other)
