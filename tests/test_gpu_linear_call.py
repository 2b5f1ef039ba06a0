"""The call around a quantized linear layer in native code against the general path: the same results, and whatever it does not take
(subclasses, transforms, strides, alignment, refusals) still goes the general way."""
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def layer(n, k, dtype, group=64, bits=4, transpose=True):
    import mlx_rs_amd as m
    gen = torch.Generator(device="cuda").manual_seed(n + k)
    shape = (n, k) if transpose else (k, n)
    return m.ops.quantize(torch.randn(shape, generator=gen, device="cuda") * 0.02, group, bits, dtype)


@pytest.fixture
def general(monkeypatch):
    """Runs a call on the general path alone."""
    import mlx_rs_amd as m

    def run(fn):
        with monkeypatch.context() as c:
            c.setattr(m.ops, "_linear_call", lambda: lambda *a: None)
            return fn()
    return run


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("shape", [(1, 256), (3, 5, 256), (256,), (40, 256), (2, 0, 256)])
@pytest.mark.parametrize("transpose,bits,group", [(True, 4, 64), (True, 8, 32), (False, 4, 128), (True, 2, 64)])
def test_native_call_equals_the_general_path(shape, dtype, transpose, bits, group, general):
    import mlx_rs_amd as m
    q, s, b = layer(128, 256, dtype, group, bits, transpose)
    x = torch.randn(shape, generator=torch.Generator(device="cuda").manual_seed(1), device="cuda").to(dtype)
    lb = torch.ones(128, device="cuda", dtype=dtype) if transpose else None
    run = lambda: m.ops.quantized_linear(x, q, s, b, lb, transpose, group, bits)  # noqa: E731
    native, want = run(), general(run)
    assert native.shape == want.shape == (*shape[:-1], 128) and native.dtype == dtype and torch.equal(native, want)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        other = run()
    side.synchronize()
    assert torch.equal(other, want)


def test_what_is_not_plain_goes_the_general_way(general):
    import mlx_rs_amd as m
    call = m.ops._linear_call()
    q, s, b = layer(128, 256, torch.bfloat16)
    x = torch.randn((4, 256), device="cuda").to(torch.bfloat16)
    assert isinstance(call(x, q, s, b, None, True, 64, 4), torch.Tensor)

    class Sub(torch.Tensor):
        pass

    buf = torch.zeros(4 * 256 + 1, device="cuda", dtype=torch.bfloat16)
    for odd in (x.as_subclass(Sub), x.t().contiguous().t(), buf[1:].reshape(4, 256), x.cpu(), x.float(), x[:, :128].contiguous(), None):
        assert call(odd, q, s, b, None, True, 64, 4) is None
    for args in ((q.cpu(), s, b), (q, s.t(), b), (q, s[:64], b), (q, s, b.half()), (q[:, :16], s, b)):
        assert call(x, *args, None, True, 64, 4) is None
    assert call(x, q, s, b, None, True, 48, 4) is None and call(x, q, s, b, None, True, 64, 3) is None
    assert call(x, q, s, b, torch.ones(127, device="cuda", dtype=torch.bfloat16), True, 64, 4) is None
    seen = []
    torch.func.vmap(lambda v: (seen.append(call(v, q, s, b, None, True, 64, 4)), v)[1])(x)
    assert seen == [None]
    for bad, text in (((x.t().contiguous().t(), q, s, b), "contiguous"), ((x.cpu(), q, s, b), "device"), ((x, q, s[:64].contiguous(), b), "scales")):
        with pytest.raises(m.MoeError, match=text):
            m.ops.quantized_linear(*bad)


def test_native_call_under_capture():
    import mlx_rs_amd as m
    q, s, b = layer(1024, 512, torch.bfloat16)
    x = torch.randn((33, 512), device="cuda").to(torch.bfloat16)
    want = m.ops.quantized_linear(x, q, s, b)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        y = m.ops.quantized_linear(x, q, s, b)
    for _ in range(3):
        y.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, want)
        assert torch.equal(m.ops.quantized_linear(x, q, s, b), want)


def test_the_interpreter_is_let_go_around_the_launch():
    """The library's functions replaced by CPython's own question whether this thread holds the interpreter: 0, as a status, is a result."""
    import ctypes as C
    import mlx_rs_amd as m
    call = m.ops._linear_call()
    q, s, b = layer(128, 256, torch.bfloat16)
    x, lb = torch.randn((4, 256), device="cuda").to(torch.bfloat16), torch.ones(128, device="cuda", dtype=torch.bfloat16)
    held = C.cast(C.pythonapi.PyGILState_Check, C.c_void_p).value
    need = C.cast(m.load_library().mi_moe_quantized_matmul_workspace_size, C.c_void_p).value
    try:
        call.__self__.bind(held, held, need)
        assert isinstance(call(x, q, s, b, None, True, 64, 4), torch.Tensor) and isinstance(call(x, q, s, b, lb, True, 64, 4), torch.Tensor)
    finally:
        m.ops._linear_call.cache_clear()
        m.ops._linear_call()
    assert torch.equal(m.ops.quantized_linear(x, q, s, b, lb), (m.ops.quantized_linear(x, q, s, b).float() + 1).bfloat16())


@pytest.mark.parametrize("after", [0, 1])
def test_what_a_mode_raises_from_an_allocation_is_what_the_caller_sees(after, general):
    """From the result's allocation or the workspace's; the call after it is none the worse."""
    import mlx_rs_amd as m
    from torch.utils._python_dispatch import TorchDispatchMode

    class Refuses(TorchDispatchMode):
        left = after

        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            if "empty" in str(func):
                self.left -= 1
                if self.left < 0:
                    raise LookupError("no allocations here")
            return func(*args, **(kwargs or {}))

    q, s, b = layer(128, 256, torch.bfloat16)
    x = torch.randn((4, 256), device="cuda").to(torch.bfloat16)
    want = m.ops.quantized_linear(x, q, s, b)
    with pytest.raises(LookupError, match="no allocations here"), Refuses():
        m.ops.quantized_linear(x, q, s, b)
    with pytest.raises(LookupError, match="no allocations here"), Refuses():
        general(lambda: m.ops.quantized_linear(x, q, s, b))
    assert torch.equal(m.ops.quantized_linear(x, q, s, b), want)
