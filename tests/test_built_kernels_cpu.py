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


@pytest.mark.skipif(not os.path.exists(LIB) or not os.path.exists(OBJDUMP), reason="no built library or disassembler")
def test_worm_steps_keep_no_array_in_scratch(tmp_path):
    """The worm's step is inlined into these kernels.  An array that it picks an element
    of must not end up in scratch memory: that is a store of all of it by 64 lanes and
    a load, in every step.  Such a load is the one with a register as its address."""
    shutil.copy(LIB, tmp_path / "lib.so")
    subprocess.run([OBJDUMP, "--offloading", "lib.so"], cwd=tmp_path, check=True, stdout=subprocess.DEVNULL)
    code = [f for f in os.listdir(tmp_path) if f.endswith("gfx950")]
    assert len(code) == 1
    text = subprocess.run([OBJDUMP, "-d", "--mcpu=gfx950", code[0]], cwd=tmp_path, check=True,
                          capture_output=True, text=True).stdout
    kernels, name, picked = set(), "", {}
    for ln in text.splitlines():
        if ln.endswith(">:"):
            name = ln[ln.index("<") + 1:-2]
        elif "worm_kernel" in name or "worm_measure_kernel" in name or "persist_kernel" in name:
            kernels.add(name)
            op = ln.split("//")[0].split(None, 1)
            if op and op[0].startswith("scratch_load"):
                _, vaddr, saddr = (a.split()[0] for a in op[1].split(","))
                if (vaddr, saddr) != ("off", "off"):
                    picked[name] = picked.get(name, 0) + 1
    assert len(kernels) == 5, kernels
    assert not picked, picked
