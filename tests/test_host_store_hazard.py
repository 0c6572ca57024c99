"""The built kernels (disassembled, no GPU): no store of more than 8 bytes is followed at once by an instruction that overwrites its data
registers.  gfx950 reads them after the next instruction has issued; the compiler knows this for most forms of a store, not for
buffer stores whose uniform offset is a scalar register (csrc/la_common.h, buf_store16p)."""
import os
import re
import shutil
import subprocess

import pytest

from lightning_attn.ops.hip import _lib

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"
STORE = re.compile(r"\s(?:buffer_store_dwordx[34] v\[(\d+):(\d+)\]|(?:global|flat)_store_dwordx[34] \S+ v\[(\d+):(\d+)\])")
WRITE = re.compile(r"\s(v_\S+) v(?:\[(\d+):(\d+)\]|(\d+)),")


def overwrites(lines):
    """(function, store, next instruction) wherever the pair is found."""
    found, name, pending = [], "", None
    for line in lines:
        if line.endswith(">:"):
            name, pending = line, None
        elif line[:1] in " \t" and line.strip():
            w = WRITE.match(line)
            if pending and w and not w[1].startswith("v_cmp"):
                lo, hi = (int(w[2]), int(w[3])) if w[2] else (int(w[4]), int(w[4]))
                if lo <= pending[1] and hi >= pending[0]:
                    found.append((name, pending[2], line.strip()))
            s = STORE.match(line)
            pending = None
            if s:
                a, b = (s[1], s[2]) if s[1] else (s[3], s[4])
                pending = (int(a), int(b), line.strip())
    return found


def test_the_scan_finds_the_pair():
    good = ["\tbuffer_store_dwordx4 v[26:29], v36, s[16:19], s28 offen nt", "\ts_nop 1", "\tv_cndmask_b32_e32 v26, v45, v42, vcc"]
    assert not overwrites(good) and len(overwrites([good[0], good[2]])) == 1
    assert not overwrites([good[0], "\tv_cndmask_b32_e32 v30, v45, v42, vcc"])


@pytest.mark.skipif(not os.path.exists(OBJDUMP), reason="no disassembler")
def test_no_store_data_overwritten_at_once(tmp_path):
    shutil.copy(_lib.LIB_PATH, tmp_path / "lib.so")
    subprocess.run([OBJDUMP, "--offloading", "lib.so"], cwd=tmp_path, check=True, capture_output=True)
    stores = 0
    for f in sorted(tmp_path.glob("lib.so.*gfx950")):
        text = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", "--no-leading-addr", f.name], cwd=tmp_path, check=True, capture_output=True, text=True).stdout
        lines = text.split("\n")
        stores += sum(bool(STORE.match(x)) for x in lines)
        assert not overwrites(lines)
    assert stores > 100
