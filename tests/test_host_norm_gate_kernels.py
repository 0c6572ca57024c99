"""The built norm_gate backward kernels (disassembled, no GPU).  Those whose rows share a wavefront hand their column sums from wavefront to
wavefront behind ONE barrier that every thread comes by.  A second one in the code means a barrier inside a branch on the lane, which
the language leaves undefined."""
import os
import re
import shutil
import subprocess

import pytest

from lightning_attn.ops.hip import _lib

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"
KERNEL = re.compile(r"<_ZN2la20norm_gate_bwd_kernelI(.*?)Li1ELi(\d+)ELb([01])EEEv.*>:$")


def barriers(lines):
    """{(element type, threads per row, few): barriers in the kernel}"""
    found, key = {}, None
    for line in lines:
        if line.endswith(">:"):
            m = KERNEL.search(line)
            key = (m[1], int(m[2]), m[3] == "1") if m else None
            if key:
                found[key] = 0
        elif key and "s_barrier" in line:
            found[key] += 1
    return found


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    if not os.path.exists(OBJDUMP):
        pytest.skip("no disassembler")
    tmp = tmp_path_factory.mktemp("norm_gate")
    shutil.copy(_lib.LIB_PATH, tmp / "lib.so")
    subprocess.run([OBJDUMP, "--offloading", "lib.so"], cwd=tmp, check=True, capture_output=True)
    found = {}
    for f in sorted(tmp.glob("lib.so.*gfx950")):
        text = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", "--no-leading-addr", f.name], cwd=tmp, check=True, capture_output=True, text=True).stdout
        found.update(barriers(text.split("\n")))
    return found


def test_one_barrier_where_rows_share_a_wavefront(kernels):
    shared = {k: n for k, n in kernels.items() if k[1] < 64}
    assert {k[1] for k in shared} == {8, 16, 32} and len({k[0] for k in shared}) == 3
    assert set(shared.values()) == {1}, shared


def test_no_kernel_that_no_launch_takes(kernels):
    """Workgroups of 256 threads for few rows: at most 16 (8) rows per CU where 16 (32) threads share a row - but rows are shared out
    like that beyond 16 per CU only."""
    assert not [k for k in kernels if k[2] and k[1] in (16, 32)]
    assert {k[1] for k in kernels if k[2]} == {8, 64, 128}
