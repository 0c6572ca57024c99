"""The warm-up walk of the chunked sweeps (the blocks before a chunk, state update only) in every form of a workgroup: with one block
to a chunk, workgroups run over 0, 1, 2, ... blocks before their own, which takes the walk through each of its register sets,
both tile buffers and each exit.  Ragged last blocks (walking backward, the first), feature dims short of the padded ones, columns short
of a slice, strided tensors, fp16.  The same operations in the same order as the walk in one piece, so bit for bit."""
import pytest
import torch

pytestmark = pytest.mark.gpu

from lightning_attn.ops import lightning_attn_func, lightning_attn_silu_func  # noqa: E402
from lightning_attn.ops.hip import _lib  # noqa: E402

FORMS = [(64, 64, None), (40, 24, None), (128, 64, None), (128, 128, False), (128, 128, True), (72, 120, True), (192, 192, False), (192, 192, True),
         (192, 192, "all"), (136, 160, "all"), (256, 256, False), (256, 256, True), (200, 136, None)]


def _tensors(n, d, e, dtype, tokens_first):
    g = torch.Generator().manual_seed(n + d + e)
    out = []
    for c in (d, d, e, e):
        t = torch.randn(2, 3, n, c, generator=g).to(dtype).cuda()
        out.append(t.transpose(1, 2).contiguous().transpose(1, 2) if tokens_first else t)
    return out


def _pass(q, k, v, do, s, **opts):
    with _lib.launch_opts(scan=False, **opts):
        ts = [t.detach().requires_grad_() for t in (q, k, v)]
        o = lightning_attn_func(*ts, s)
        return (o.detach(),) + torch.autograd.grad(o, ts, do)


@pytest.mark.parametrize("d,e,wide", FORMS)
@pytest.mark.parametrize("n,dtype,tokens_first,decay", [(130, torch.bfloat16, False, True), (383, torch.float16, True, True), (449, torch.bfloat16, True, False)])
def test_chunks_of_one_block_match_the_single_walk(d, e, wide, n, dtype, tokens_first, decay):
    q, k, v, do = _tensors(n, d, e, dtype, tokens_first)
    s = torch.tensor([0.01, 0.1, 0.7], device="cuda") if decay else None
    one = _pass(q, k, v, do, s, wide=wide, chunks=1)
    for once in (None, False):
        for a, b in zip(one, _pass(q, k, v, do, s, wide=wide, chunks=8, once=once)):
            assert torch.equal(a, b), once


@pytest.mark.parametrize("d,e,wide", FORMS[:6])
def test_silu_chunks_of_one_block(d, e, wide):
    q, k, v, _ = _tensors(327, d, e, torch.bfloat16, True)
    s = torch.tensor([0.01, 0.1, 0.7], device="cuda")
    got = []
    for chunks in (1, 8):
        with _lib.launch_opts(scan=False, wide=wide, chunks=chunks), torch.no_grad():
            got.append(lightning_attn_silu_func(q, k, v, s))
    assert torch.equal(got[0], got[1])
