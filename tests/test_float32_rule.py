"""Which dense float32 products go in tiles: csrc/dense_rule.hpp's rule, and what it means for a row's bits."""
import ctypes as C
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def tiles(tmp_path_factory):
    d = tmp_path_factory.mktemp("rule")
    (d / "rule.cpp").write_text('#include "dense_rule.hpp"\nextern "C" int tiles(long M, int N, int K, int bits) { return mi_moe::float32_tiles(M, N, K, bits); }\n')
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-shared", "-fPIC", "-I", os.path.join(ROOT, "mlx-rs_amd", "csrc"), str(d / "rule.cpp"), "-o", str(d / "rule.so")], check=True)
    lib = C.CDLL(str(d / "rule.so"))
    lib.tiles.argtypes = [C.c_long, C.c_int, C.c_int, C.c_int]
    return lib.tiles


# few tiles, whatever their K; few XCDs with any; a second round for a few of them
NARROW = [(64, 256, 16384), (72, 256, 8192), (64, 146, 16384), (64, 1024, 4096), (64, 512, 8192), (400, 64, 8192), (1000, 64, 4096), (2228, 104, 5632), (2510, 136, 1280), (6376, 104, 4096)]
MANY = [(64, 3072, 3072), (192, 1024, 4096), (116, 1176, 3712), (700, 1024, 4096), (1000, 3072, 3072), (1000, 4096, 4096), (700, 256, 8192)]


@pytest.mark.parametrize("bits", [4, 8])
def test_tiles_where_they_fill_the_chip(tiles, bits):
    """Each measured on both kernels: the plain one is 1.3 to 5 times as fast on the first ones, the tiles on the others."""
    assert not any(tiles(*shape, bits) for shape in NARROW)
    assert all(tiles(*shape, bits) for shape in MANY)
    assert not any(tiles(63, n, k, bits) or tiles(5000, n, 896, bits) for n in (64, 4096, 20000) for k in (1024, 16384))


@pytest.mark.gpu
@pytest.mark.parametrize("rows,n,k,bits", [(72, 256, 8192, 4), (64, 146, 4096, 8), (500, 64, 2048, 4)])
def test_narrow_products_keep_the_sums_of_a_row(rows, n, k, bits):
    import torch

    from test_gpu_float32_tiles import layer
    x, _, _, _, _, product = layer(rows, n, k, bits, 64)
    y = product(x)
    for i in range(0, rows, 7):
        assert torch.equal(y[i], product(x[i:i + 1].contiguous())[0]), i
