"""The operators' timed cases: what a program built on this package has them do, over the range of sizes it
does it at.  Five kinds of call, each through the package's public functions:

  train      lightning_attn_func forward and backward (a training step of one attention layer)
  infer      lightning_attn_func without gradients (prefill of one attention layer)
  silu       lightning_attn_silu_func without gradients (prefill of the TNL attention block, which hands over its
             projections before their activation, as (b, h, n, d) views of (b, n, h * d) memory)
  rmsnorm    SimpleRMSNorm forward and backward (the norm of every layer)
  normgate   norm_gate forward and backward (the output norm and gate of the TNL attention block)

The listed cases are the sizes this repository's benchmarks and tests quote; draw() takes others from the ranges
around them: sequences of 1 to 65536 tokens (training: from 64), 1 to 8 in a batch, 4 to 64 heads of 16 to 256
features, every element type, with and without decay, heads before tokens in memory or after them; rows of 64 to
16384 elements."""
import math
import os
import sys

import torch

# (the working folder is the root of the tree whose code is run)
sys.path.insert(0, os.path.join(os.getcwd(), "lightning-attention_amd"))

from lightning_attn.ops import SimpleRMSNorm, lightning_attn_func, lightning_attn_silu_func  # noqa: E402
from lightning_attn.ops.hip import norm_gate  # noqa: E402
from lightning_attn.utils import _build_slope_tensor  # noqa: E402

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}


def _attn(name, kind, b, h, n, d, e=None, dtype="bf16", decay=True, tokens_first=False):
    return {"name": name, "kind": kind, "b": b, "h": h, "n": n, "d": d, "e": e or d, "dtype": dtype, "decay": decay,
            "tokens_first": tokens_first}


def _rows(name, kind, rows, cols, dtype="bf16"):
    return {"name": name, "kind": kind, "rows": rows, "cols": cols, "dtype": dtype}


def listed():
    return [
        # a short prompt through one layer: launch and call latency
        _attn("infer_short", "infer", 1, 8, 113, 64),
        # a small model in full precision (the size of the plain-PyTorch plumbing check)
        _attn("train_f32_1k", "train", 1, 8, 1024, 64, dtype="fp32"),
        # the odd length, the fp16 type and the d != e of the test matrix
        _attn("train_f16_ragged", "train", 6, 8, 1213, 128, 64, dtype="fp16"),
        # a feature dim that is no power of two
        _attn("train_d192", "train", 2, 12, 2048, 192),
        # training inside the attention block: heads as views of the projections' memory
        _attn("train_block_4k", "train", 4, 16, 4096, 128, tokens_first=True),
        # the size the speed of the operator is quoted at
        _attn("train_8k", "train", 4, 32, 8192, 128),
        # one long document, few heads, without decay
        _attn("train_one_long", "train", 1, 16, 32768, 128, decay=False),
        # the long end of the sequence sweep
        _attn("train_32k", "train", 4, 32, 32768, 128),
        # prefill inside the attention block, activation included
        _attn("silu_block_8k", "silu", 4, 32, 8192, 128, tokens_first=True),
        # norm of a model of width 4096 at the same number of tokens
        _rows("rmsnorm_32k", "rmsnorm", 32768, 4096),
        # a ragged batch at a width that is no power of two, in full precision
        _rows("rmsnorm_f32_odd", "rmsnorm", 2 * 913, 1000, "fp32"),
        # output norm and gate of the attention block at embedding width 2048
        _rows("normgate_16k", "normgate", 16384, 2048),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """A case of the same ranges, at most as large as the largest listed one (in bytes, and for float32 attention in
    the operations its slower matrix instructions have to do)."""
    kind = rng.choices(("train", "infer", "silu", "rmsnorm", "normgate"), (5, 3, 2, 2, 1))[0]
    while True:
        dtype = rng.choices(("bf16", "fp16", "fp32"), (6, 3, 1 if kind != "silu" else 0))[0]
        if kind in ("rmsnorm", "normgate"):
            c = {"kind": kind, "rows": _log_int(rng, 16, 131072), "cols": 8 * _log_int(rng, 8, 2048 if kind == "rmsnorm" else 1024), "dtype": dtype}
            if kind == "normgate" and dtype == "fp32":
                c["cols"] = min(c["cols"], 4096)
            limit = 3.2e9
        else:
            d = 8 * rng.choice((2, 4, 8, 8, 10, 12, 16, 16, 16, 16, 20, 24, 32))
            e = d if rng.random() < 0.75 else 8 * rng.choice((4, 8, 12, 16, 24))
            if dtype == "fp32" or kind == "silu":
                d, e = min(d, 128), min(e, 128)
            c = {"kind": kind, "b": rng.randint(1, 8), "h": rng.choice((4, 6, 8, 12, 16, 20, 24, 32, 40, 64)),
                 "n": _log_int(rng, 64 if kind == "train" else 1, 65536), "d": d, "e": e, "dtype": dtype,
                 "decay": kind == "silu" or rng.random() < 0.75,  # (the block always decays)
                 "tokens_first": kind == "silu" or (dtype != "fp32" and rng.random() < 0.4)}
            limit = 4e9
        w = work(c)
        if w["bytes"] <= limit and (dtype != "fp32" or w["flops"] <= 1e11):
            return c


def _tensor(gen, shape, dtype, tokens_first=False):
    if tokens_first:  # (b, h, n, c) as a view of (b, n, h * c) memory
        b, h, n, c = shape
        return torch.randn(b, n, h, c, generator=gen, dtype=dtype, device="cuda").transpose(1, 2)
    return torch.randn(*shape, generator=gen, dtype=dtype, device="cuda")


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    dt = DTYPES[case["dtype"]]
    kind = case["kind"]
    st = {"kind": kind}
    if kind == "rmsnorm":
        x = _tensor(gen, (case["rows"], case["cols"]), dt)
        # one element in a hundred fifty times as large, as trained activations have them
        x *= 1 + 49 * (torch.rand(x.shape, generator=gen, device="cuda", dtype=torch.float32) < 0.01).to(dt)
        st.update(x=x.requires_grad_(), dy=_tensor(gen, x.shape, dt), norm=SimpleRMSNorm(case["cols"]))
    elif kind == "normgate":
        shape = (case["rows"], case["cols"])
        st.update(o=_tensor(gen, shape, dt).requires_grad_(), g=_tensor(gen, shape, dt).requires_grad_(), dy=_tensor(gen, shape, dt),
                  weight=(1 + 0.1 * _tensor(gen, shape[1:], dt)).requires_grad_(), bias=(0.1 * _tensor(gen, shape[1:], dt)).requires_grad_())
    else:
        b, h, n, d, e = (case[k] for k in ("b", "h", "n", "d", "e"))
        q, k, v = (_tensor(gen, (b, h, n, c), dt, case["tokens_first"]) for c in (d, d, e))
        st.update(q=q, k=k, v=v, s=_build_slope_tensor(h).cuda() if case["decay"] else None)
        if kind == "train":
            for t in (q, k, v):
                t.requires_grad_()
            st["do"] = _tensor(gen, (b, h, n, e), dt, case["tokens_first"])
    return st


def run(st):
    kind = st["kind"]
    if kind == "train":
        o = lightning_attn_func(st["q"], st["k"], st["v"], st["s"])
        return (o,) + torch.autograd.grad(o, (st["q"], st["k"], st["v"]), st["do"])
    if kind == "infer":
        with torch.no_grad():
            return lightning_attn_func(st["q"], st["k"], st["v"], st["s"])
    if kind == "silu":
        with torch.no_grad():
            return lightning_attn_silu_func(st["q"], st["k"], st["v"], st["s"])
    if kind == "rmsnorm":
        y = st["norm"](st["x"])
        return (y,) + torch.autograd.grad(y, st["x"], st["dy"])
    y = norm_gate(st["o"], st["g"], st["weight"], st["bias"])
    return (y,) + torch.autograd.grad(y, (st["o"], st["g"], st["weight"], st["bias"]), st["dy"])


def work(case):
    """Every tensor once per call that takes or gives it (forward and backward are two calls, with all of the forward
    pass between the two uses of its inputs); attention's operations as the block recurrence of 64 tokens needs them,
    two per multiply-add."""
    elt = 4 if case["dtype"] == "fp32" else 2
    if case["kind"] in ("rmsnorm", "normgate"):
        tensors, per = (5, 9) if case["kind"] == "rmsnorm" else (8, 40)
        return {"bytes": tensors * case["rows"] * case["cols"] * elt, "flops": per * case["rows"] * case["cols"]}
    tokens, d, e = case["b"] * case["h"] * case["n"], case["d"], case["e"]
    block = min(64, case["n"])
    bytes_, flops = (2 * d + 2 * e) * elt, 2 * block * (d + e) + 4 * d * e
    if case["kind"] == "train":
        bytes_ += (4 * d + 3 * e) * elt
        flops += 2 * block * (3 * d + 2 * e) + 10 * d * e
    return {"bytes": bytes_ * tokens, "flops": flops * tokens}


def tolerance(case):
    """About four times the error measured against the same formula in 64 bits.  2-norm: attention 2.7e-3 (bf16), 3.3e-4
    (fp16), 2.8e-7 (fp32; 9.6e-7 over 4096 tokens without decay, growing with the root of the length); rows 1.7e-3,
    2.1e-4, 1.5e-7.  Largest: attention 3.1e-2, 2.7e-3, 8.7e-6; rows 3.9e-3, 4.9e-4, 1.7e-6."""
    dtype = case["dtype"]
    if case["kind"] in ("rmsnorm", "normgate"):
        return {"rel": {"bf16": 7e-3, "fp16": 9e-4, "fp32": 6e-7}[dtype], "max": {"bf16": 1.6e-2, "fp16": 2e-3, "fp32": 7e-6}[dtype]}
    grown = 1.0 if case["decay"] else max(1.0, math.sqrt(case["n"] / 4096))
    return {"rel": {"bf16": 1e-2, "fp16": 1.4e-3, "fp32": 4e-6 * grown}[dtype], "max": {"bf16": 0.12, "fp16": 1.2e-2, "fp32": 4e-5 * grown}[dtype]}
