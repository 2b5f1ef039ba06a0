"""quantized_linear where its native call cannot be loaded: the general path takes the call."""
import os

import pytest

torch = pytest.importorskip("torch")


@pytest.fixture(params=["missing", "not a library", "wants what no library has", "another torch's"])
def without_native_call(request, tmp_path, monkeypatch):
    import mlx_rs_amd as m
    so = os.path.join(os.path.dirname(os.path.abspath(m.ops.__file__)), "_linear_call.so")
    there = tmp_path / "_linear_call.so"
    if request.param == "not a library":
        there.write_bytes(b"no ELF")
    elif request.param == "wants what no library has":
        data = open(so, "rb").read()
        assert b"THPVariableClass" in data
        there.write_bytes(data.replace(b"THPVariableClass", b"THPVariablfClass"))
    elif request.param == "another torch's":
        there.symlink_to(so)
        monkeypatch.setattr(torch, "__version__", "1.0.0+cpu")
    if request.param != "another torch's":
        monkeypatch.setattr(m.ops, "__file__", str(tmp_path / "ops.py"))
    m.ops._linear_call.cache_clear()
    yield m
    m.ops._linear_call.cache_clear()


def test_the_general_path_takes_the_call_with_one_warning(without_native_call):
    m = without_native_call
    x, q = torch.zeros((2, 64), dtype=torch.bfloat16), torch.zeros((64, 8), dtype=torch.int32)
    s = torch.zeros((64, 1), dtype=torch.bfloat16)
    with pytest.warns(RuntimeWarning, match="without its native call") as seen:
        for _ in range(2):
            with pytest.raises(m.MoeError, match="device tensor"):  # the general path's own refusal of these
                m.ops.quantized_linear(x, q, s, s)
    assert len([w for w in seen if "native call" in str(w.message)]) == 1


def test_it_loads_here():
    import warnings
    import mlx_rs_amd as m
    m.ops._linear_call.cache_clear()
    with warnings.catch_warnings():
        warnings.simplefilter("error")
        assert m.ops._linear_call().__name__ == "quantized_linear"
