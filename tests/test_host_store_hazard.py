"""The built kernels (disassembled, no GPU): no store of more than 8 bytes is followed within two wait states by an instruction that
overwrites its data registers.  gfx950 reads them after later instructions have issued; the compiler knows this for most forms of a store, not
for buffer stores whose uniform offset is a scalar register (csrc/la_common.h, buf_store16p), so there are none of those."""
import os
import re
import shutil
import subprocess

import pytest

from lightning_attn.ops.hip import _lib

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"
WAIT_STATES = 2
STORE = re.compile(r"\s(?:buffer_store_dwordx[34] ([va])\[(\d+):(\d+)\]|(?:global|flat)_store_dwordx[34] \S+ ([va])\[(\d+):(\d+)\])")
WRITE = re.compile(r"\s(v_\S+) ([va])(?:\[(\d+):(\d+)\]|(\d+))(?:,|$|\s)")
SWAP = re.compile(r"\sv_(?:swap|permlane\d+_swap)\S* v(\d+), v(\d+)")
NOP = re.compile(r"\ss_nop (\d+|0x[0-9a-f]+)")
JUMP = re.compile(r"\s(s_c?branch\S*) .*<(\S+?)(?:\+0x([0-9a-f]+))?>")
ADDRESS = re.compile(r"// ([0-9A-F]+):")
HEAD = re.compile(r"^([0-9a-f]+) <(\S+)>:$")


def writes(line):
    """(register file, first, last) of each run of vector registers that a vector instruction writes."""
    s = SWAP.match(line)
    if s:
        return [("v", int(r), int(r)) for r in s.groups()]
    w = WRITE.match(line)
    if not w or w[1].startswith("v_cmp"):
        return []
    return [(w[2], int(w[3] or w[5]), int(w[4] or w[5]))]


def overwrites(lines):
    """(function, store, instruction that overwrites its data too early) wherever there is one, on either way out of a branch."""
    code, at, start, name = [], {}, {}, ""  # (instruction, function), address -> index, function -> address
    for line in lines:
        h = HEAD.match(line)
        if h:
            name = h[2]
            start[name] = int(h[1], 16)
        elif line[:1] in " \t" and line.strip():
            a = ADDRESS.search(line)
            if a:
                at[int(a[1], 16)] = len(code)
            code.append((line, name))

    def follow(i):
        """indices of what may run after instruction i"""
        j = JUMP.match(code[i][0])
        out = [] if code[i][0].split()[0] in ("s_branch", "s_endpgm", "s_setpc_b64") else [i + 1]
        if j and j[2] in start:
            out.append(at.get(start[j[2]] + int(j[3] or "0", 16), len(code)))
        return [k for k in out if k < len(code) and code[k][1] == code[i][1]]

    found = []
    for i, (line, name) in enumerate(code):
        s = STORE.match(line)
        if not s:
            continue
        file, lo, hi = (s[1], int(s[2]), int(s[3])) if s[1] else (s[4], int(s[5]), int(s[6]))
        todo = [(k, WAIT_STATES) for k in follow(i)]
        while todo:
            k, left = todo.pop()
            after = code[k][0]
            if any(f == file and a <= hi and b >= lo for f, a, b in writes(after)):
                found.append((name, line.strip(), after.strip()))
            n = NOP.match(after)
            left -= 1 + int(n[1], 0) if n else 1
            if left > 0:
                todo += [(x, left) for x in follow(k)]
    return found


def test_the_scan_finds_the_pair():
    store, other, clash = "\tbuffer_store_dwordx4 v[26:29], v36, s[16:19], s28 offen nt", "\tv_add_u32_e32 v30, 1, v30", "\tv_cndmask_b32_e32 v26, v45, v42, vcc"
    assert not overwrites([store, "\ts_nop 1", clash]) and not overwrites([store, other, other, clash]) and not overwrites([store, other, "\ts_nop 0", clash])
    assert len(overwrites([store, clash])) == len(overwrites([store, other, clash])) == len(overwrites([store, "\ts_nop 0", clash])) == 1
    assert not overwrites([store, "\tv_cndmask_b32_e32 v30, v45, v42, vcc", "\tv_cmp_gt_u32_e32 vcc, v26, v27"])
    assert len(overwrites([store, "\tv_mfma_f32_16x16x32_bf16 v[28:31], v[0:3], v[4:7], v[28:31]"])) == len(overwrites([store, "\tv_swap_b32 v1, v27"])) == 1
    assert not overwrites([store, "\tv_accvgpr_write_b32 a26, v1"]) and len(overwrites([store.replace("x4 v", "x4 a"), "\tv_accvgpr_write_b32 a26, v1"])) == 1
    # behind a branch, taken or not
    code = ["%016x <f>:" % 0x100] + ["%s // %012X: 00000000" % (t, 0x100 + 4 * i) for i, t in enumerate(
        [store, "\ts_cbranch_scc1 2", "\ts_nop 0", "\ts_endpgm", clash, "\ts_endpgm"])]
    assert not overwrites(code)
    code[2] += " <f+0x10>"
    assert len(overwrites(code)) == 1


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """the lines of each code object"""
    if not os.path.exists(OBJDUMP):
        pytest.skip("no disassembler")
    tmp = tmp_path_factory.mktemp("store_hazard")
    shutil.copy(_lib.LIB_PATH, tmp / "lib.so")
    subprocess.run([OBJDUMP, "--offloading", "lib.so"], cwd=tmp, check=True, capture_output=True)
    return [subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", f.name], cwd=tmp, check=True, capture_output=True, text=True).stdout.split("\n")
            for f in sorted(tmp.glob("lib.so.*gfx950"))]


def test_no_store_data_overwritten_at_once(kernels):
    for lines in kernels:
        assert not overwrites(lines)
    assert sum(bool(STORE.match(x)) for lines in kernels for x in lines) > 100
    assert sum(bool(JUMP.match(x)) for lines in kernels for x in lines) > 100


def test_no_store_with_a_scalar_offset(kernels):
    offsets = [m[1] for lines in kernels for x in lines for m in [re.match(r"\sbuffer_store_dwordx[34] [va]\[\S+ \S+ s\[\d+:\d+\], (\S+)", x)] if m]
    assert len(offsets) > 100 and set(offsets) == {"0"}
