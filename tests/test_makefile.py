"""The C library builds without torch or Python: what `make` would run in csrc/."""
import os
import subprocess
import sys

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "mlx-rs_amd", "csrc")


def planned(python):
    return subprocess.run(["make", "-C", CSRC, "--always-make", "--dry-run", f"PYTHON={python}"], check=True, capture_output=True, text=True)


@pytest.mark.parametrize("python", ["false", "/no/such/python", "bare"])
def test_the_library_alone_needs_no_torch(python, tmp_path):
    if python == "bare":  # a Python that finds no torch
        python = tmp_path / "python3"
        python.write_text(f"#!/bin/sh\nexec {sys.executable} -S -E \"$@\"\n")
        python.chmod(0o755)
    run = planned(python)
    assert "libmi_moe.so" in run.stdout and "linear_call.cpp" not in run.stdout and run.stderr == ""


def test_the_native_call_is_built_where_torch_is():
    pytest.importorskip("torch")
    assert "linear_call.cpp" in planned(sys.executable).stdout
