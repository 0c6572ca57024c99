"""float32 sweep: the walk cut into warm-up chunks against the walk in one piece, at the sizes where its tile buffers
change hands: one warm-up block, an even and an odd number of them, a ragged last block, feature dims short of the
padded 64 / 128 and columns short of a slice.  The same operations in the same order, so bit for bit; and against the
formula in float64 (float32 accumulation over at most 1100 terms: 1e-5 of the largest result)."""
import pytest
import torch

import oracle

pytestmark = pytest.mark.gpu

from lightning_attn.ops import lightning_attn_func  # noqa: E402
from lightning_attn.ops.hip import _lib  # noqa: E402


def _run(q, k, v, s, do, chunks):
    with _lib.launch_opts(chunks=chunks):
        ts = [t.clone().requires_grad_() for t in (q, k, v)]
        o = lightning_attn_func(*ts, s)
        return (o.detach(),) + torch.autograd.grad(o, ts, do)


@pytest.mark.parametrize("n", [65, 128, 192, 257, 320, 1085])
@pytest.mark.parametrize("d,e", [(64, 64), (40, 72), (128, 128), (100, 20)])
@pytest.mark.parametrize("decay", [True, False])
def test_float32_chunks_match_the_single_walk(n, d, e, decay):
    b, h = 1, 3
    g = torch.Generator().manual_seed(n + d)
    q, k = (torch.randn(b, h, n, d, generator=g) * d ** -0.5 for _ in range(2))
    v, do = (torch.randn(b, h, n, e, generator=g) for _ in range(2))
    s = torch.tensor([0.02, 0.2, 0.9]) if decay else None
    want = oracle.linear_attn_fwd_bwd(q, k, v, s, do, torch.float64)
    dev = [t.cuda() for t in (q, k, v)]
    sd = s.cuda() if decay else None
    one = _run(*dev, sd, do.cuda(), 1)
    for w, x in zip(want, one):
        assert (x.cpu().double() - w).abs().max() <= 1e-5 * w.abs().max()
    for chunks in (0, 2, 3, 8):
        for a, c in zip(one, _run(*dev, sd, do.cuda(), chunks)):
            assert torch.equal(a, c), chunks
