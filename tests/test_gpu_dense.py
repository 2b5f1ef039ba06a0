"""quantized_matmul / quantized_linear in bfloat16 with groups of 64 at the edges of the rules that pick its kernel, against
the float64 product of the dequantised matrix."""
import ctypes as C

import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

# one rounding of the result, and of the weights where the large tiles dequantise them: each at most 2^-8 of its values and
# typically 0.42 of that, so 0.6 * 2^-8 together in the 2-norm
BOUND = 2.0 ** -8
ROWS = [(m, 400, k) for k in (256, 4096) for m in (1, 3, 4, 15, 16, 17, 19, 20, 32, 33)]  # few rows, streamed, small tiles
TILES = [(1024, 4096, 128), (1280, 4096, 128), (1281, 4096, 128), (1300, 4112, 128), (1536, 4096, 192)]  # small, then large


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("rows,n,k", ROWS + TILES)
def test_dense_products(rows, n, k, bits):
    import mlx_rs_amd as m
    from test_gpu_codes import product
    if bits == 4 and k % 128:
        pytest.skip("4-bit rows are whole 128s")
    gen = torch.Generator(device="cuda").manual_seed(rows + k)
    q, s, b = m.ops.quantize(torch.randn((n, k), generator=gen, device="cuda") * 0.02, 64, bits)
    x = torch.randn((rows, k), generator=gen, device="cuda").bfloat16()
    lb = torch.randn(n, generator=gen, device="cuda").bfloat16()
    ref = product(x, q, s, b, 64, bits)
    y = m.ops.quantized_linear(x, q, s, b, bits=bits)
    assert float((y.double() - ref).norm() / ref.norm()) <= BOUND
    assert float((y[-1].double() - ref[-1]).norm() / ref[-1].norm()) <= BOUND  # (the last tile's last row)
    yb = m.ops.quantized_linear(x, q, s, b, lb, bits=bits)
    assert torch.equal(yb, (y.float() + lb.float()).bfloat16())


def test_what_needs_a_workspace_or_alignment_still_says_so():
    import mlx_rs_amd as m
    lib = m.load_library()
    q, s, b = m.ops.quantize(torch.randn((64, 256), device="cuda"), 64, 4)
    x, y = torch.randn((4, 256), device="cuda").bfloat16(), torch.zeros((4, 64), device="cuda").bfloat16()
    ws = torch.empty(1 << 16, dtype=torch.uint8, device="cuda")

    def call(sp, workspace, size):
        return lib.mi_moe_quantized_matmul(x.data_ptr(), q.data_ptr(), sp, b.data_ptr(), 4, 64, 256, 1, 64, 4, y.data_ptr(),
                                           workspace, size, C.c_void_p(torch.cuda.current_stream().cuda_stream))
    assert call(s.data_ptr(), None, 0) != 0 and b"workspace too small" in lib.mi_moe_last_error()
    assert call(s.data_ptr() + 2, ws.data_ptr(), ws.numel()) != 0 and b"aligned" in lib.mi_moe_last_error()
    assert call(s.data_ptr(), ws.data_ptr(), ws.numel()) == 0
