"""Token-major tensors against plain ones, in every form of a workgroup: the same products in the same order, so the same bits.  (The two
layouts have kernels of their own, whose stores address memory differently; a register of a store overwritten too early shows as
a few elements of one of them.)"""
import ctypes

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


@pytest.mark.parametrize("d,e,wide", [(64, 64, 0), (128, 128, _lib.LA_OPT_OFF), (128, 128, _lib.LA_OPT_ON), (192, 192, _lib.LA_OPT_OFF), (192, 192, _lib.LA_OPT_ON),
                                      (192, 192, _lib.LA_OPT_ALL)])
@pytest.mark.parametrize("n,stride", [(1, 1 << 33), (2, 1 << 30), (3, 1 << 29), (5, 1 << 28), (9, 1 << 27), (17, 1 << 26), (33, 1 << 25)])
def test_rows_so_far_apart_that_those_beyond_the_last_would_wrap(d, e, wide, n, stride):
    """Few rows, `stride` bytes apart: a multiple of it that belongs to no row is 4 GiB, offset 0 in 32 bits."""
    g = torch.Generator().manual_seed(n + d)
    q, k, v = (torch.randn(1, 1, n, c, generator=g).bfloat16().cuda() for c in (d, d, e))
    opts = _lib.LaunchOpts(0, 0, wide, 0, 0)
    far = torch.empty((n - 1) * stride // 2 + e, dtype=torch.bfloat16, device="cuda")
    o = far.as_strided((1, 1, n, e), (far.numel(), far.numel(), stride // 2, 1)).fill_(7.0)
    want = torch.empty_like(v)
    strides = (ctypes.c_int64 * 12)(*(n * d, n * d, d) * 2, n * e, n * e, e, (n - 1) * stride // 2 + stride // 2, (n - 1) * stride // 2 + stride // 2, stride // 2)
    for out, st in ((want, None), (o, strides)):
        assert _lib.lib().la_fwd_opts(q.data_ptr(), k.data_ptr(), v.data_ptr(), None, out.data_ptr(), st, 1, 1, n, d, e, 0, None, 0, ctypes.byref(opts),
                                      torch.cuda.current_stream().cuda_stream) == 0
    assert torch.equal(o, want)
