"""The built kernels' hand-written changes of the exec mask.

add_in (lu.hip) and fma_in (trsm.hip) set exec, run a few VALU instructions and
set it back in one asm text, which neither the register allocator's ordinary
rules nor the hazard pass look into.  In the machine code of the library built
here: no instruction of such a region reads a register that an earlier one of the
region wrote for another purpose, and two wait states follow the last of them
before anything else (a DPP read of a register needs two after its VALU write).
"""
import glob
import os
import re
import shutil
import subprocess

import pytest

from hpcc_fpga_amd.linpack import LIB_PATH

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"


@pytest.fixture(scope="module")
def regions(tmp_path_factory):
    if not (os.path.exists(OBJDUMP) and os.path.exists(LIB_PATH)):
        pytest.skip("needs the built library and llvm-objdump")
    d = tmp_path_factory.mktemp("code")
    so = shutil.copy(LIB_PATH, d)
    subprocess.run([OBJDUMP, "--offloading", so], check=True, capture_output=True)
    found = []
    for obj in glob.glob(so + ".*gfx950"):
        text = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", obj], check=True,
                              capture_output=True, text=True).stdout
        kernel, insts = None, []
        for line in text.splitlines():
            m = re.match(r"[0-9a-f]+ <(.*)>:", line)
            if m:
                kernel = m.group(1)
                continue
            inst = line.split("//")[0].strip()
            if inst:
                insts.append((kernel, inst))
        for i, (kernel, inst) in enumerate(insts):
            if re.match(r"s_mov_b32 exec_lo, (0x|[0-9])", inst):
                j = next(j for j in range(i, len(insts)) if insts[j][1] == "s_mov_b64 exec, -1")
                found.append((kernel, [x for _, x in insts[i + 2:j]], insts[j + 1][1]))
    return found


def test_regions_are_there(regions):
    kernels = {k for k, _, _ in regions}
    assert any("lu_diag_kernel" in k for k in kernels)
    assert any("prep_kernel" in k for k in kernels)


def test_no_input_is_overwritten_before_it_is_read(regions):
    for kernel, body, _ in regions:
        written = set()
        for inst in body:
            dst, *src = re.findall(r"\bv\d+\b", inst)
            assert not written & set(src) - {dst}, (kernel, body)
            assert dst not in written, (kernel, body)
            written.add(dst)


def test_two_wait_states_follow(regions):
    # the move back to exec is the first
    for kernel, body, after in regions:
        assert after.startswith("s_nop"), (kernel, body, after)
