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
