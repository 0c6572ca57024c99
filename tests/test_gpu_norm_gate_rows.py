"""norm_gate backward where its walk over the rows can go wrong: row counts around a workgroup's group of rows (1024
threads: 16, 8, 4, 2 or 1 of them side by side) and around the whole grid's (256 workgroups: the second pass of some
workgroups only, whose rows were requested during the first), with widths short of the threads that share a row.
Tolerance: float64 formula, 5e-3 / 1e-3 / 2e-5 in the 2-norm (rounding of bf16 / fp16 / float32 results)."""
import pytest
import torch

import oracle
from util import rel_norm

pytestmark = pytest.mark.gpu

from lightning_attn.ops.hip import norm_gate  # noqa: E402


@pytest.mark.parametrize("cols,side", [(64, 16), (512, 16), (1000, 8), (2048, 4), (2056, 2), (8192, 1)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_row_counts_around_a_pass(cols, side, dtype):
    if dtype == torch.float32 and cols > 4096:
        pytest.skip("float32 rows beyond 4096 columns are not supported")
    lim = {torch.bfloat16: 5e-3, torch.float16: 1e-3, torch.float32: 2e-5}[dtype]
    for rows in sorted({1, max(1, side - 1), side + 1, 256 * side - 1, 256 * side, 256 * side + 1, 512 * side + 3}):
        g_ = torch.Generator().manual_seed(rows)
        o, g, dy = ((torch.randn(rows, cols, generator=g_) * 2).to(dtype) for _ in range(3))
        w, b = (torch.randn(cols, generator=g_).to(dtype) for _ in range(2))
        leaves = [t.cuda().requires_grad_() for t in (o, g, w, b)]
        y = norm_gate(*leaves, 1e-5)
        got = (y,) + torch.autograd.grad(y, leaves, dy.cuda())
        want = oracle.norm_gate_fwd_bwd(o, g, w, b, dy, 1e-5, torch.float64)
        for name, a, r in zip(("y", "d_o", "d_g", "d_weight", "d_bias"), got, want):
            assert rel_norm(a.detach().cpu(), r) < lim, (rows, name, rel_norm(a.detach().cpu(), r))


@pytest.mark.parametrize("cols,side", [(64, 4), (200, 4), (512, 4), (520, 2), (1024, 2)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_row_counts_around_the_small_workgroups(cols, side, dtype):
    """16-bit rows of one or two wavefronts: workgroups of 256 threads up to one group of rows per CU (256), of 1024 beyond."""
    lim = {torch.bfloat16: 5e-3, torch.float16: 1e-3}[dtype]
    for rows in (1, side - 1, side, side + 1, 255 * side + 1, 256 * side, 256 * side + 1):
        g_ = torch.Generator().manual_seed(rows + cols)
        o, g, dy = ((torch.randn(rows, cols, generator=g_) * 2).to(dtype) for _ in range(3))
        w, b = (torch.randn(cols, generator=g_).to(dtype) for _ in range(2))
        leaves = [t.cuda().requires_grad_() for t in (o, g, w, b)]
        y = norm_gate(*leaves, 1e-5)
        got = (y,) + torch.autograd.grad(y, leaves, dy.cuda())
        want = oracle.norm_gate_fwd_bwd(o, g, w, b, dy, 1e-5, torch.float64)
        for name, a, r in zip(("y", "d_o", "d_g", "d_weight", "d_bias"), got, want):
            assert rel_norm(a.detach().cpu(), r) < lim, (rows, name, rel_norm(a.detach().cpu(), r))


@pytest.mark.parametrize("cols", [8, 64, 72, 128, 136, 256])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_short_rows_side_by_side(cols, dtype):
    """Rows of up to 32 chunks of 16 bytes: 8, 4 or 2 of them to a wavefront - always in the forward pass, beyond 16 rows per CU
    (4096) in the backward pass; the last workgroup of a launch with one row, all but one or all of them."""
    lim = {torch.bfloat16: 5e-3, torch.float16: 1e-3, torch.float32: 2e-5}[dtype]
    for rows in (1, 31, 32, 33, 4096, 4097, 8193, 32768, 65537):
        g_ = torch.Generator().manual_seed(rows + cols)
        o, g, dy = ((torch.randn(rows, cols, generator=g_) * 2).to(dtype) for _ in range(3))
        w, b = (torch.randn(cols, generator=g_).to(dtype) for _ in range(2))
        leaves = [t.cuda().requires_grad_() for t in (o, g, w, b)]
        y = norm_gate(*leaves, 1e-5)
        got = (y,) + torch.autograd.grad(y, leaves, dy.cuda())
        want = oracle.norm_gate_fwd_bwd(o, g, w, b, dy, 1e-5, torch.float64)
        for name, a, r in zip(("y", "d_o", "d_g", "d_weight", "d_bias"), got, want):
            assert rel_norm(a.detach().cpu(), r) < lim, (rows, name, rel_norm(a.detach().cpu(), r))
