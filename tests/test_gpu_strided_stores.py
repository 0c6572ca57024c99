"""Token-major tensors against plain ones, in every form of a workgroup: the same products in the same order, so the same bits.  (The two
layouts have kernels of their own, whose stores address memory differently; a register of a store overwritten too early shows as
a few elements of one of them.)"""
import pytest
import torch

pytestmark = pytest.mark.gpu

from lightning_attn.ops import lightning_attn_func  # noqa: E402
from lightning_attn.ops.hip import _lib  # noqa: E402


@pytest.mark.parametrize("d,e,wide", [(64, 64, None), (40, 24, None), (128, 64, None), (128, 128, False), (128, 128, True), (72, 120, True), (192, 192, False),
                                      (192, 192, True), (192, 192, "all"), (136, 160, "all"), (256, 256, False), (256, 256, True)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("decay", [True, False])
def test_token_major_tensors_give_the_same_bits(d, e, wide, dtype, decay):
    g = torch.Generator().manual_seed(d + e)
    plain = [torch.randn(2, 3, 383, c, generator=g).to(dtype).cuda() for c in (d, d, e, e)]
    tokens_first = [t.transpose(1, 2).contiguous().transpose(1, 2) for t in plain]
    s = torch.tensor([0.01, 0.1, 0.7], device="cuda") if decay else None
    got = []
    for q, k, v, do in (plain, tokens_first):
        with _lib.launch_opts(wide=wide, chunks=1, scan=False):
            leaves = [t.detach().requires_grad_() for t in (q, k, v)]
            o = lightning_attn_func(*leaves, s)
            got.append((o.detach(),) + torch.autograd.grad(o, leaves, do))
    for a, b in zip(*got):
        assert torch.equal(a, b)
