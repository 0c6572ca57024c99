"""Backward pass with d != e whose three sweeps share a launch (few sequences, feature dims up to 128): against the same
sweeps in launches of their own, bit for bit (the same instantiations of the same body, warm-up chunks rebuild their
state in the same order), over both padded widths of d and of e, lengths around the 64-token blocks and the shortest
chunked walk, ragged column slices, both layouts; and against the formula in float32 on the same inputs (2e-2 of the
result's scale, as for every 16-bit case of the attention tests)."""
import pytest
import torch

import oracle
from util import assert_close_scaled

pytestmark = pytest.mark.gpu

from lightning_attn.ops import lightning_attn_func  # noqa: E402
from lightning_attn.ops.hip import _lib  # noqa: E402


@pytest.mark.parametrize("d,e", [(128, 64), (64, 128), (40, 24), (96, 128), (104, 8), (16, 112)])
@pytest.mark.parametrize("n", [1, 64, 65, 511, 513, 1213])
@pytest.mark.parametrize("dtype,decay,token_major", [(torch.bfloat16, True, False), (torch.float16, False, True)])
def test_one_launch_is_the_separate_launches(d, e, n, dtype, decay, token_major):
    b, h = 1, 5
    g = torch.Generator().manual_seed(n * 131 + d)

    def mk(c, scale=1.0):
        t = torch.randn(b, n, h, c, generator=g) * scale if token_major else torch.randn(b, h, n, c, generator=g) * scale
        return t.to(dtype).transpose(1, 2) if token_major else t.to(dtype)

    q, k, v, do = mk(d, d ** -0.5), mk(d, d ** -0.5), mk(e), mk(e)
    s = torch.tensor([0.01, 0.05, 0.2, 0.5, 0.9]) if decay else None

    def grads(**opts):
        with _lib.launch_opts(scan=False, **opts):
            ts = [t.cuda().requires_grad_() for t in (q, k, v)]
            o = lightning_attn_func(*ts, s.cuda() if decay else None)
            return torch.autograd.grad(o, ts, do.cuda())

    apart = grads(once=False, wide=False)
    for opts in ({}, {"once": True}, {"once": True, "chunks": 1}, {"once": True, "chunks": 3}):
        for a, c in zip(apart, grads(**opts)):
            assert torch.equal(a, c), opts
    want = oracle.linear_attn_fwd_bwd(q, k, v, s, do, torch.float32)[1:]
    for name, a, r in zip(("dq", "dk", "dv"), apart, want):
        assert_close_scaled(a, r, 2e-2, 2e-2, name)


# more than one 64-column workgroup per CU for the three sweeps: the library lets dQ and dK share a launch, dV follows
PAIRS = [(48, 130, 128, 96), (48, 700, 96, 128), (41, 513, 72, 128), (88, 200, 64, 40), (128, 65, 32, 64)]


@pytest.mark.parametrize("h,n,d,e", PAIRS)
@pytest.mark.parametrize("token_major", [False, True])
def test_dq_and_dk_sharing_a_launch_by_choice(h, n, d, e, token_major):
    g = torch.Generator(device="cuda").manual_seed(n)

    def mk(c):
        t = torch.randn(1, n, h, c, generator=g, device="cuda").bfloat16()
        return t.transpose(1, 2) if token_major else t.transpose(1, 2).contiguous()

    q, k, v, do = mk(d), mk(d), mk(e), mk(e)
    s = torch.linspace(0.01, 0.9, h, device="cuda")

    def grads(**opts):
        with _lib.launch_opts(**opts):
            ts = [t.detach().requires_grad_() for t in (q, k, v)]
            return torch.autograd.grad(lightning_attn_func(*ts, s), ts, do)

    for a, c in zip(grads(once=False, wide=False, scan=False), grads()):
        assert torch.equal(a, c)
    sel = [0, h - 1]
    want = oracle.linear_attn_fwd_bwd(*(t[:, sel].cpu() for t in (q, k, v)), s[sel].cpu(), do[:, sel].cpu(), torch.float32)[1:]
    for name, a, r in zip(("dq", "dk", "dv"), grads(), want):
        assert_close_scaled(a[:, sel].cpu(), r, 2e-2, 2e-2, name)
