"""The copies from memory straight into LDS, as they stand in the built library: the wait states that the assembler does not add."""
import os
import re
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"


def test_every_copy_brings_its_wait_states(tmp_path):
    """Five between a vector instruction that writes a scalar register and a load that reads it, one between a write of m0 and the copy: the
    write of m0 is one, s_nop N is N + 1."""
    so = os.path.join(ROOT, "mlx-rs_amd", "libmi_moe.so")
    if not os.path.exists(OBJDUMP) or not os.path.exists(so):
        pytest.skip("no disassembler, or nothing built")
    (tmp_path / "lib.so").symlink_to(so)
    subprocess.run([OBJDUMP, "--offloading", "lib.so"], cwd=tmp_path, check=True, stdout=subprocess.DEVNULL)
    copies = 0
    for code in tmp_path.glob("lib.so.*gfx950"):
        text = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", str(code)], check=True, capture_output=True, text=True).stdout
        lines = [l.split("//")[0].strip() for l in text.splitlines()]
        for i, line in enumerate(lines):
            if line.startswith("buffer_load") and line.endswith(" lds"):
                copies += 1
                nop = re.fullmatch(r"s_nop (\d+)", lines[i - 1])
                assert nop and int(nop.group(1)) >= 3 and lines[i - 2].startswith("s_mov_b32 m0, "), lines[i - 3:i + 1]
    assert copies
