"""How the products on raw codes deal out their work: csrc/dense_rule.hpp, which needs no GPU, compiled and asked."""
import ctypes as C
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def rule(tmp_path_factory):
    d = tmp_path_factory.mktemp("rule")
    (d / "rule.cpp").write_text('#include "dense_rule.hpp"\n'
                                'extern "C" int share(int K, int n, int pairs) { return mi_moe::share_of_k(K, n, pairs != 0); }\n'
                                'extern "C" int tile(long M, int N, int K, int bits, int group, int bf16) { return (int)mi_moe::dense_tile(M, N, K, bits, group, bf16 != 0); }\n'
                                'extern "C" int longer(long M, int N, int K, int bits) { return mi_moe::long_tile_rows(M, N, K, bits); }\n')
    so = d / "rule.so"
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-shared", "-fPIC", "-I", os.path.join(ROOT, "mlx-rs_amd", "csrc"),
                    str(d / "rule.cpp"), "-o", str(so)], check=True)
    lib = C.CDLL(str(so))
    lib.tile.argtypes = [C.c_long, C.c_int, C.c_int, C.c_int, C.c_int, C.c_int]
    lib.longer.argtypes = [C.c_long, C.c_int, C.c_int, C.c_int]
    return lib


@pytest.mark.parametrize("n", [1, 2, 4])
def test_shares_of_k_are_as_even_as_whole_128s_can_be(rule, n):
    """The longest share sets the time: of 19 times 128 values four shares take 5, 5, 5 and 4, not 6, 6, 6 and 1."""
    for units in range(1, 200):
        share, pairs = rule.share(128 * units, n, 0), rule.share(128 * units, n, 1)
        assert share == 128 * -(-units // n)
        assert pairs % 256 == 0 and share <= pairs <= share + 128
    assert rule.share(2432, 4, 0) == 640


SMALL, REGISTERS_SMALL, COLUMNS, WIDE, REGISTERS, REGISTERS_SHARED = range(6)  # DenseTile


@pytest.mark.parametrize("shape,bits,group,want", [
    # rows, columns, K: launches of at most 256 tiles whose fullest XCD gets more than its 32 CUs hold at once
    ((567, 1280, 3840), 4, 64, REGISTERS_SHARED), ((367, 2304, 2944), 4, 64, REGISTERS_SHARED), ((221, 2080, 1408), 4, 32, COLUMNS),
    ((546, 1808, 4096), 8, 32, REGISTERS_SHARED), ((293, 3184, 1408), 8, 32, REGISTERS_SHARED), ((743, 2672, 3072), 8, 64, REGISTERS),
    # and those that fit
    ((77, 1680, 2432), 4, 32, SMALL), ((414, 1760, 2944), 4, 64, COLUMNS), ((661, 1488, 2432), 8, 64, SMALL), ((998, 1168, 3840), 4, 64, REGISTERS_SHARED),
    # 64 x 256: rows of few values, rounds that are not full
    ((991, 3392, 1024), 4, 64, REGISTERS), ((961, 3664, 4096), 4, 64, WIDE), ((1874, 2576, 4096), 4, 64, REGISTERS), ((3784, 3520, 4096), 4, 64, WIDE),
    ((2544, 2272, 4096), 8, 64, REGISTERS), ((3872, 1888, 2688), 8, 64, WIDE), ((3281, 2896, 2432), 8, 32, REGISTERS), ((777, 4096, 4096), 8, 64, REGISTERS),
])
def test_the_tile_follows_the_fullest_xcd(rule, shape, bits, group, want):
    """Each of these was measured with the other tiles too (dense_rule.hpp)."""
    assert rule.tile(*shape, bits, group, 0) == rule.tile(*shape, bits, group, 1) == want


@pytest.mark.parametrize("shape,bits,group,bf16,want", [((102, 1808, 3584), 8, 32, 1, REGISTERS_SMALL), ((29, 2176, 1920), 8, 32, 1, REGISTERS_SMALL), ((49, 1200, 1024), 8, 32, 1, SMALL),
                                                        ((258, 1744, 1408), 8, 32, 1, SMALL), ((102, 1808, 3584), 8, 32, 0, SMALL), ((102, 1808, 3584), 8, 64, 1, SMALL), ((102, 1808, 3584), 4, 32, 1, SMALL)])
def test_small_tiles_with_every_code_converted_stay_in_registers(rule, shape, bits, group, bf16, want):
    assert rule.tile(*shape, bits, group, bf16) == want


@pytest.mark.parametrize("shape,bits,want", [
    ((512, 4096, 4096), 8, 0), ((513, 4096, 4096), 8, 96), ((768, 4096, 4096), 4, 96), ((769, 4096, 4096), 8, 128), ((1024, 4096, 4096), 8, 128), ((1025, 4096, 4096), 8, 0),
    ((769, 4096, 4096), 4, 0), ((769, 4096, 2944), 8, 0), ((769, 4096, 3072), 8, 128), ((640, 4096, 896), 4, 0), ((640, 4096, 1024), 4, 96),
    ((640, 2304, 2304), 4, 0), ((641, 2304, 2304), 4, 96), ((960, 2304, 2304), 8, 96), ((961, 2304, 4096), 8, 128)])
def test_longer_tiles_where_they_are_one_round(rule, shape, bits, want):
    assert rule.longer(*shape, bits) == want
