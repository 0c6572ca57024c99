"""float32 sweep where the number of sweeps in a launch decides between forms of a workgroup that sum in different orders (64 columns, one
wavefront to a slab, and 32 columns, two): the launch options still change no bit of a result."""
import pytest
import torch

import oracle

pytestmark = pytest.mark.gpu

from lightning_attn.ops import lightning_attn_func  # noqa: E402
from lightning_attn.ops.hip import _lib  # noqa: E402


def _inputs(h, n, d):
    g = torch.Generator().manual_seed(100 * h + n + d)
    q, k = (torch.randn(1, h, n, d, generator=g) * d ** -0.5 for _ in range(2))
    v, do = (torch.randn(1, h, n, d, generator=g) for _ in range(2))
    return q, k, v, torch.logspace(-2, 0, h), do


def _pass(q, k, v, s, do, decay=True, **opts):
    with _lib.launch_opts(**opts):
        ts = [t.cuda().requires_grad_() for t in (q, k, v)]
        o = lightning_attn_func(*ts, s.cuda() if decay else None)
        return (o.detach(),) + torch.autograd.grad(o, ts, do.cuda())


# (32 columns in a sweep alone, 64 in three together; but 8 sequences, 32 in either, and d = 128, whose two forms give the same sums)
@pytest.mark.parametrize("h,n,d", [(16, 1024, 64), (24, 700, 40), (9, 700, 64), (40, 513, 56), (8, 1024, 64), (4, 2048, 128)])
@pytest.mark.parametrize("decay", [True, False])
def test_gradients_of_separate_launches_are_the_joint_launchs(h, n, d, decay):
    args = _inputs(h, n, d)
    together, apart = _pass(*args, decay=decay), _pass(*args, decay=decay, paired=False)
    for a, c in zip(together, apart):
        assert torch.equal(a, c)
    want = oracle.linear_attn_fwd_bwd(args[0], args[1], args[2], args[3] if decay else None, args[4], torch.float64)
    for w, x in zip(want, together):  # (float32 accumulation over at most 2048 + 128 terms)
        assert (x.cpu().double() - w).abs().max() <= 1e-5 * w.abs().max()


# (64 columns to a workgroup, of 256 CUs: the backward pass of the first six - of 48 sequences because 32 columns give more workgroups than CUs
# at any length - and the forward pass of the others)
@pytest.mark.parametrize("h,n,d", [(9, 700, 64), (24, 1085, 64), (24, 700, 40), (48, 65, 64), (48, 128, 40), (48, 192, 64),
                                   (49, 700, 64), (64, 1085, 40), (136, 257, 64), (136, 320, 40)])
@pytest.mark.parametrize("decay", [True, False])
def test_warm_up_of_the_64_column_form(h, n, d, decay):
    """Chunks behind no, one, an odd and an even number of warm-up blocks, ragged last blocks, against the walk in one piece."""
    args = _inputs(h, n, d)
    one = _pass(*args, decay=decay, chunks=1)
    for chunks in (0, 2, 3, 5, 8):
        for a, c in zip(one, _pass(*args, decay=decay, chunks=chunks)):
            assert torch.equal(a, c), chunks
    want = oracle.linear_attn_fwd_bwd(args[0], args[1], args[2], args[3] if decay else None, args[4], torch.float64)
    for w, x in zip(want, one):  # (float32 accumulation over at most 1085 + 128 terms)
        assert (x.cpu().double() - w).abs().max() <= 1e-5 * w.abs().max()


@pytest.mark.parametrize("h,n,d", [(90, 113, 24), (96, 200, 32), (264, 130, 8), (264, 64, 32)])
def test_rows_of_up_to_32_columns_in_more_workgroups_than_cus(h, n, d):
    """32 columns to a workgroup also beyond one round of them: together and apart, in one walk and cut up."""
    args = _inputs(h, n, d)
    one = _pass(*args)
    for opts in ({"paired": False}, {"chunks": 1}, {"chunks": 2}, {"chunks": 3, "paired": False}):
        for a, c in zip(one, _pass(*args, **opts)):
            assert torch.equal(a, c), opts
    want = oracle.linear_attn_fwd_bwd(*args, torch.float64)
    for w, x in zip(want, one):  # (float32 accumulation over at most 200 + 64 terms)
        assert (x.cpu().double() - w).abs().max() <= 1e-5 * w.abs().max()
