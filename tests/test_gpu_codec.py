"""quantize / dequantize at the edges of their launch: one group, a last block that is not full, every code width, group
size and element type; a group of one value, of a huge spread, and with NaN among its values.  Exact: every step is one
correctly rounded float32 operation, restated here in numpy (mlx-rs/src/ops/quantization.rs:31-47)."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def restated(w, group, bits):
    f = np.float32
    v = w.reshape(-1, group)
    lo, hi = np.fmin.reduce(v, axis=1), np.fmax.reduce(v, axis=1)
    top = f((1 << bits) - 1)
    mask = np.abs(lo) > np.abs(hi)
    scale = np.maximum((hi - lo) / top, f(1e-7))
    scale = np.where(mask, scale, -scale)
    edge = np.where(mask, lo, hi)
    q0 = np.rint(edge / scale)
    with np.errstate(divide="ignore", invalid="ignore"):
        scale, bias = np.where(q0 != 0, edge / q0, scale).astype(f), np.where(q0 != 0, edge, f(0)).astype(f)
        codes = np.fmin(np.fmax(np.rint((v - bias[:, None]) / scale[:, None]), f(0)), top).astype(np.uint32)
    return codes, scale, bias


@pytest.mark.parametrize("dtype", ["bfloat16", "float16", "float32"])
@pytest.mark.parametrize("group", [32, 64, 128])
@pytest.mark.parametrize("bits", [2, 4, 8])
@pytest.mark.parametrize("rows,cols", [(1, 128), (3, 128), (17, 384), (129, 2176)])
def test_codec_at_the_edges(rows, cols, bits, group, dtype):
    import mlx_rs_amd as m
    dt = getattr(torch, dtype)
    rng = np.random.default_rng(rows * 1000 + cols + bits + group)
    w = rng.normal(0, 0.02, (rows, cols)).astype(np.float32)
    w[0, :group] = 0.25
    if rows > 1:
        w[1, :group] *= np.exp(rng.uniform(-12, 12, group)).astype(np.float32)  # up to e^12 / 50 times a normal draw: below float16's 65504
        w[1, -1] = np.nan
    codes, scale, bias = restated(w, group, bits)
    q, s, b = m.ops.quantize(torch.from_numpy(w).cuda(), group, bits, dt)
    per = 32 // bits
    want = (codes.reshape(-1, per) << (np.arange(per, dtype=np.uint32) * bits)).sum(axis=1, dtype=np.uint32)
    assert np.array_equal(q.cpu().numpy().view(np.uint32).reshape(-1), want)
    for got, ref in ((s, scale), (b, bias)):
        assert torch.equal(got.cpu().reshape(-1), torch.from_numpy(ref).to(dt))
    # the values: one multiplication and one addition in float32, then the rounding to the type of the result
    s32, b32 = s.float().cpu().numpy().reshape(-1, 1), b.float().cpu().numpy().reshape(-1, 1)
    v = (codes.astype(np.float32) * s32 + b32).astype(np.float32).reshape(rows, cols)
    for out in {dt, torch.float32}:
        got = m.ops.dequantize(q, s, b, group, bits, out)
        assert torch.equal(got.cpu(), torch.from_numpy(v).to(out))


@pytest.mark.parametrize("dtype", ["bfloat16", "float16", "float32"])
@pytest.mark.parametrize("bits", [2, 4, 8])
def test_addresses_aligned_for_their_elements_only(bits, dtype):
    """Operands and results one element behind a 16-byte address: the same values, nothing around them touched."""
    import mlx_rs_amd as m
    from mlx_rs_amd import capi
    lib, dt = m.load_library(), getattr(torch, dtype)
    code = {"bfloat16": capi.DTYPE_BF16, "float16": capi.DTYPE_F16, "float32": capi.DTYPE_F32}[dtype]
    stream = torch.cuda.current_stream().cuda_stream

    def room(n, of):  # n elements with one before and one behind, all set
        return torch.full((n + 2,), 7, dtype=of, device="cuda")

    def inner(t, like):
        assert t[0] == 7 and t[-1] == 7
        return t[1:-1].reshape(like.shape)
    w = torch.randn((5, 192), device="cuda") * 0.02
    q, s, b = m.ops.quantize(w, 64, bits, dt)
    w1, q1, s1, b1 = room(w.numel(), torch.float32), room(q.numel(), torch.int32), room(s.numel(), dt), room(b.numel(), dt)
    w1[1:-1] = w.reshape(-1)
    at = lambda t: t.data_ptr() + t.element_size()  # noqa: E731
    assert lib.mi_moe_quantize_typed(at(w1), 5, 192, 64, bits, code, at(q1), at(s1), at(b1), stream) == 0
    assert torch.equal(inner(q1, q), q) and torch.equal(inner(s1, s), s) and torch.equal(inner(b1, b), b)
    for fn, of in ((lib.mi_moe_dequantize_native, dt), (lib.mi_moe_dequantize_typed, torch.float32)):
        want, got = m.ops.dequantize(q, s, b, 64, bits, of), room(w.numel(), of)
        assert fn(at(q1), at(s1), at(b1), 5, 192, 64, bits, code, at(got), stream) == 0
        assert torch.equal(inner(got, want), want)


def test_more_values_than_one_launch_has_threads_for():
    """2^35 + 4096 values of 2-bit codes (8.6 GB, 69 GB dequantised): more than 2^32 threads of eight values; and quantised again."""
    import mlx_rs_amd as m
    rows = (1 << 23) + 1
    if torch.cuda.mem_get_info()[0] < 250e9:
        pytest.skip("the card has no 250 GB left")
    q = torch.zeros((rows, 256), dtype=torch.int32, device="cuda")
    s, b = torch.ones((rows, 32), device="cuda").bfloat16(), torch.zeros((rows, 32), device="cuda").bfloat16()
    marks = [0, (1 << 22) - 1, 1 << 22, (1 << 23) - 1, 1 << 23]  # around the joints of the launches
    gen = torch.Generator(device="cuda").manual_seed(0)
    for r in marks:
        w = torch.randn((1, 4096), generator=gen, device="cuda")
        for whole, row in zip((q, s, b), m.ops.quantize(w, 128, 2)):
            whole[r] = row[0]
    out = m.ops.dequantize(q, s, b, 128, 2)
    for r in marks:
        assert torch.equal(out[r:r + 1], m.ops.dequantize(q[r:r + 1], s[r:r + 1], b[r:r + 1], 128, 2))
    assert out[5].eq(0).all() and out[-5].eq(0).all()
    del q, s, b, out
    torch.cuda.empty_cache()
    w = torch.zeros((rows, 4096), device="cuda")
    for r in marks:
        w[r] = torch.randn(4096, generator=gen, device="cuda")
    got = m.ops.quantize(w, 128, 2)
    for r in marks:
        for whole, row in zip(got, m.ops.quantize(w[r:r + 1], 128, 2)):
            assert torch.equal(whole[r:r + 1], row)
    del w, got
    torch.cuda.empty_cache()
