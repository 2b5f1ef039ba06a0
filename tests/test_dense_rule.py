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
                                'extern "C" int share(int K, int n, int pairs) { return mi_moe::share_of_k(K, n, pairs != 0); }\n')
    so = d / "rule.so"
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-shared", "-fPIC", "-I", os.path.join(ROOT, "mlx-rs_amd", "csrc"),
                    str(d / "rule.cpp"), "-o", str(so)], check=True)
    return C.CDLL(str(so))


@pytest.mark.parametrize("n", [1, 2, 4])
def test_shares_of_k_are_as_even_as_whole_128s_can_be(rule, n):
    """The longest share sets the time: of 19 times 128 values four shares take 5, 5, 5 and 4, not 6, 6, 6 and 1."""
    for units in range(1, 200):
        share, pairs = rule.share(128 * units, n, 0), rule.share(128 * units, n, 1)
        assert share == 128 * -(-units // n)
        assert pairs % 256 == 0 and share <= pairs <= share + 128
    assert rule.share(2432, 4, 0) == 640
