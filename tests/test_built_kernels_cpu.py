"""The instructions of the built library, where the source alone does not fix them."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "stochasticseriesexpansion.jl_amd", "libssegpu.so")
OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"


@pytest.mark.skipif(not os.path.exists(LIB) or not os.path.exists(OBJDUMP), reason="no built library or disassembler")
def test_write_back_is_waited_for(tmp_path):
    """A walker that passes between workgroups is given away by an atomic: the L2
    write-back ahead of it has to be waited for, in both work-queue kernels."""
    shutil.copy(LIB, tmp_path / "lib.so")
    subprocess.run([OBJDUMP, "--offloading", "lib.so"], cwd=tmp_path, check=True, stdout=subprocess.DEVNULL)
    code = [f for f in os.listdir(tmp_path) if f.endswith("gfx950")]
    assert len(code) == 1
    text = subprocess.run([OBJDUMP, "-d", "--mcpu=gfx950", code[0]], cwd=tmp_path, check=True,
                          capture_output=True, text=True).stdout
    lines = [ln.split("//")[0].strip() for ln in text.splitlines()]
    back = [k for k, ln in enumerate(lines) if ln.startswith("buffer_wbl2")]
    assert len(back) == 2
    for k in back:
        assert lines[k + 1].startswith("s_waitcnt vmcnt(0)"), lines[k:k + 6]
