"""float32 sweep: the forms a workgroup comes in (32 or 64 columns, one or two wavefronts to a slab of columns), each at its
edges: one and two blocks, a ragged last one, columns that fill no slab or half a slice, feature dims short of the padded ones
and of the half a wavefront takes; with few sequences (32 columns) and with more than there are CUs for (64).  Against the formula
in float64: float32 accumulation over at most 2 * 150 + 128 terms, 1e-5 of the largest result."""
import pytest
import torch

import oracle

pytestmark = pytest.mark.gpu

from lightning_attn.ops import lightning_attn_func  # noqa: E402


@pytest.mark.parametrize("h", [3, 136])
@pytest.mark.parametrize("d,e", [(64, 64), (24, 24), (40, 8), (64, 72), (128, 128), (72, 72), (104, 48), (120, 24)])
@pytest.mark.parametrize("n", [1, 64, 150])
def test_float32_forms(h, d, e, n):
    g = torch.Generator().manual_seed(1000 * d + e + n)
    q, k = (torch.randn(1, h, n, d, generator=g) * d ** -0.5 for _ in range(2))
    v, do = (torch.randn(1, h, n, e, generator=g) for _ in range(2))
    s = torch.logspace(-2, 0, h)
    want = oracle.linear_attn_fwd_bwd(q, k, v, s, do, torch.float64)
    ts = [t.cuda().requires_grad_() for t in (q, k, v)]
    o = lightning_attn_func(*ts, s.cuda())
    got = (o.detach(),) + torch.autograd.grad(o, ts, do.cuda())
    for w, x in zip(want, got):
        assert (x.cpu().double() - w).abs().max() <= 1e-5 * w.abs().max()
