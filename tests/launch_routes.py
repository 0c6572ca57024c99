"""Which launches the library maps attention calls onto, asked without a GPU (256 compute units assumed): the launching
functions are replaced by recorders (launch_recorder.hip) in a process of their own.  Calls go through la_fwd_carry and
la_bwd_carry with the buffers that the size queries ask for, as the operators make them.

    routes(shapes) -> per (bh, n, d, e, dtype) {"kept": bytes, "ws": bytes, "fwd": "...", "bwd": "..."}"""
import ctypes
import functools
import json
import os
import subprocess
import sys
import tempfile

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "lightning-attention_amd", "lightning_attn", "_C", "liblightning_attn_hip.so")


_folder = tempfile.TemporaryDirectory(prefix="la_routes_")  # (gone when this process ends)


@functools.lru_cache(None)
def _recorder():
    out = os.path.join(_folder.name, "recorder.so")
    hipcc = os.environ.get("HIPCC") or "/opt/rocm/bin/hipcc"
    subprocess.run([hipcc, "--offload-arch=gfx950", "-O1", "-fPIC", "-shared", "-std=c++17", "-Xclang", "-target-feature", "-Xclang",
                    "-packed-fp32-ops", "-Wno-unknown-warning-option", "-I", os.path.join(ROOT, "include"), "-I",
                    os.path.join(ROOT, "lightning-attention_amd", "csrc"), os.path.join(ROOT, "tests", "launch_recorder.hip"), "-o", out],
                   check=True, capture_output=True)
    return out


def routes(shapes, lib=LIB, decay=True, once=0, workspace=True):
    """`once`: that launch option (0: none given); `workspace`: whether the backward pass gets what it asks for, or none."""
    ask = json.dumps({"recorder": _recorder(), "lib": lib, "decay": decay, "once": once, "workspace": workspace, "shapes": [list(s) for s in shapes]})
    r = subprocess.run([sys.executable, os.path.abspath(__file__)], input=ask, capture_output=True, text=True, check=True)
    return {tuple(k): v for k, v in json.loads(r.stdout)}


def _main():
    ask = json.load(sys.stdin)
    rec = ctypes.CDLL(ask["recorder"], mode=ctypes.RTLD_GLOBAL)  # (before the library: its calls find these first)
    rec.recorded.restype = ctypes.c_char_p
    L = ctypes.CDLL(ask["lib"])
    i64, vp, sz, i32 = ctypes.c_int64, ctypes.c_void_p, ctypes.c_size_t, ctypes.c_int
    L.la_workspace_bytes_opts.restype = L.la_carry_bytes.restype = sz
    L.la_workspace_bytes_opts.argtypes = [i32] + [i64] * 5 + [i32, vp]
    L.la_carry_bytes.argtypes = [i64] * 5 + [i32, vp]
    L.la_fwd_carry.argtypes = [vp] * 6 + [i64] * 5 + [i32, vp, sz, vp, vp, sz, vp]
    L.la_bwd_carry.argtypes = [vp] * 9 + [i64] * 5 + [i32, vp, sz, vp, vp, sz, vp]
    opts = (ctypes.c_int32 * 5)(0, 0, 0, 0, ask["once"])
    op = ctypes.cast(opts, vp) if ask["once"] else None
    p = [0x10000 * (i + 1) for i in range(12)]  # (never read)
    s = p[11] if ask["decay"] else None
    out = []
    for bh, n, d, e, dtype in ask["shapes"]:
        dims = (1, bh, n, d, e, dtype)
        kept = L.la_carry_bytes(*dims, op)
        w0, w1 = (L.la_workspace_bytes_opts(i, *dims, op) for i in (0, 1))
        got = {"kept": kept, "ws": w1}
        w1 = w1 if ask["workspace"] else 0
        w0 = 0 if kept else w0
        assert L.la_fwd_carry(p[0], p[1], p[2], s, p[3], None, *dims, p[9] if w0 else None, w0, op, p[10] if kept else None, kept, None) == 0
        got["fwd"] = rec.recorded().decode()
        assert L.la_bwd_carry(*p[:3], s, *p[4:8], None, *dims, p[9] if w1 else None, w1, op, p[10] if kept else None, kept, None) == 0
        got["bwd"] = rec.recorded().decode()
        out.append([(bh, n, d, e, dtype), got])
    json.dump(out, sys.stdout)


if __name__ == "__main__":
    _main()
