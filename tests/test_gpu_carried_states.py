"""la_fwd_carry / la_bwd_carry where the forward pass runs in chunks from scanned states: the dQ sweep starts from the
transposes of those states, and dK + dV from states collected once (dK from their transposes).

* o is la_fwd's with the same workspace, bit for bit; the gradients agree with la_bwd's without a workspace (warm-up
  chunks: states summed in the same order, operands rounded to the tensors' dtype in the other role: a few 1e-3 in the
  2-norm, as for la_bwd_saved) and with the formula on a few sequences;
* carry and workspace start as NaN: every slot that is read was written;
* too few bytes of carry: exactly la_bwd_opts;
* an altered carry shows in dQ after its first chunk and nowhere else, and shared states in the workspace: the launches under
  test are the ones that ran (which ones a shape takes: tests/test_host_launch_routes.py)."""
import ctypes

import pytest
import torch

import oracle
from util import assert_close_scaled, rel_norm

pytestmark = pytest.mark.gpu

from lightning_attn.ops import lightning_attn_func  # noqa: E402
from lightning_attn.ops.hip import _lib  # noqa: E402
from lightning_attn.utils import _build_slope_tensor  # noqa: E402

CODE = {torch.bfloat16: 0, torch.float16: 1}

CASES = [
    # b, h, n, d, e, dtype, decay, token_major
    (1, 16, 8192, 128, 128, torch.bfloat16, True, False),
    (1, 13, 9057, 128, 128, torch.bfloat16, True, False),   # ragged, a short last chunk, units short of a multiple of 8
    (2, 12, 6400, 96, 120, torch.float16, True, False),    # d != e: dQ alone
    (4, 16, 4096, 128, 128, torch.bfloat16, True, True),   # projection layout; dK + dV in single walks
    (4, 16, 6400, 128, 128, torch.bfloat16, True, True),   # projection layout; dK + dV: two chunks, four collected
    (3, 15, 6113, 72, 72, torch.bfloat16, False, True),    # no decay, d off the tiles
    (1, 16, 16384, 64, 64, torch.bfloat16, True, False),   # 64-column workgroups
    (1, 9, 9001, 48, 40, torch.float16, False, False),
]


def _strides(*ts):
    vals = []
    for t in ts:
        vals += list(t.stride())[:3]
    return (ctypes.c_int64 * len(vals))(*vals)


@pytest.mark.parametrize("b, h, n, d, e, dtype, decay, token_major", CASES)
def test_gradients_from_carried_states(b, h, n, d, e, dtype, decay, token_major):
    L = _lib.lib()
    code = CODE[dtype]
    g = torch.Generator().manual_seed(n)

    def mk(c):
        if token_major:
            return torch.randn(b, n, h, c, generator=g).to(dtype).cuda().transpose(1, 2)
        return torch.randn(b, h, n, c, generator=g).to(dtype).cuda()

    q, k, v, do = mk(d), mk(d), mk(e), mk(e)
    s = _build_slope_tensor(h).float().cuda().contiguous() if decay else None
    sp = s.data_ptr() if decay else None
    st = torch.cuda.current_stream().cuda_stream
    nbytes = L.la_carry_bytes(b, h, n, d, e, code, None)
    print("carry case", (b, h, n, d, e, dtype, decay, token_major), nbytes, flush=True)
    assert nbytes > 0 and L.la_saved_state_bytes(b, h, n, d, e, code, None) == 0
    assert nbytes == L.la_workspace_bytes(0, b, h, n, d, e, code)
    nan = lambda size: torch.full((max(size, 16) // 4,), float("nan"), device="cuda")  # noqa: E731
    carry, ws0 = nan(nbytes), nan(nbytes)
    wb = L.la_workspace_bytes(1, b, h, n, d, e, code)
    ws1 = nan(wb)

    def fwd(ws, cr, cb):
        o = torch.full_like(v, float("nan"))
        rc = L.la_fwd_carry(q.data_ptr(), k.data_ptr(), v.data_ptr(), sp, o.data_ptr(), _strides(q, k, v, o), b, h, n, d, e, code,
                            ws.data_ptr() if ws is not None else None, nbytes if ws is not None else 0, None,
                            cr.data_ptr() if cr is not None else None, cb, st)
        assert rc == 0, L.la_error_string(rc)
        return o

    def bwd(ws, cr, cb):
        gr = [torch.full_like(t, float("nan")) for t in (q, k, v)]
        rc = L.la_bwd_carry(q.data_ptr(), k.data_ptr(), v.data_ptr(), sp, do.data_ptr(), *(t.data_ptr() for t in gr),
                            _strides(q, k, v, do, *gr), b, h, n, d, e, code, ws.data_ptr() if ws is not None else None,
                            wb if ws is not None else 0, None, cr.data_ptr() if cr is not None else None, cb, st)
        assert rc == 0, L.la_error_string(rc)
        return gr

    o, o0 = fwd(None, carry, nbytes), fwd(ws0, None, 0)
    got, plain, short = bwd(ws1, carry, nbytes), bwd(None, None, 0), bwd(None, carry, nbytes - 4)
    torch.cuda.synchronize()
    assert torch.equal(o, o0)
    for a, p, sh in zip(got, plain, short):
        assert torch.equal(p, sh)
        assert rel_norm(a, p.float()) < 3e-3, rel_norm(a, p.float())
    sel = [0, h - 1]
    qs, ks, vs, ds = (t[-1:, sel].cpu().contiguous() for t in (q, k, v, do))
    want = oracle.linear_attn_fwd_bwd(qs, ks, vs, s.cpu()[sel] if decay else None, ds, torch.float32)
    for name, a, r in zip(("o", "dq", "dk", "dv"), [o] + got, want):
        assert_close_scaled(a[-1:, sel], r, 2e-2, 2e-2, "carried %s" % name)
        assert rel_norm(a[-1:, sel], r) < 1e-2, (name, rel_norm(a[-1:, sel], r))


def _prepared(b, h, n, d, e, dtype, decay, token_major):
    """Forward pass done; backward(workspace bytes, carry) -> dq, dk, dv; the carry, the workspace and the bytes it may have."""
    L = _lib.lib()
    code = CODE[dtype]
    g = torch.Generator(device="cuda").manual_seed(n)

    def mk(c):
        t = torch.randn(b, n, h, c, generator=g, device="cuda") if token_major else torch.randn(b, h, n, c, generator=g, device="cuda")
        return t.to(dtype).transpose(1, 2) if token_major else t.to(dtype)

    q, k, v, do = mk(d), mk(d), mk(e), mk(e)
    s = _build_slope_tensor(h).float().cuda().contiguous() if decay else None
    st = torch.cuda.current_stream().cuda_stream
    nbytes, wb = L.la_carry_bytes(b, h, n, d, e, code, None), L.la_workspace_bytes(1, b, h, n, d, e, code)
    assert nbytes > 0
    carry = torch.empty(nbytes // 4, device="cuda")
    ws = torch.full((max(wb, 16) // 4,), float("nan"), device="cuda")
    o = torch.empty_like(v)
    rc = L.la_fwd_carry(q.data_ptr(), k.data_ptr(), v.data_ptr(), s.data_ptr() if decay else None, o.data_ptr(), _strides(q, k, v, o), b, h, n, d, e, code, None, 0, None,
                        carry.data_ptr(), nbytes, st)
    assert rc == 0, L.la_error_string(rc)

    def backward(ws_bytes, cr):
        gr = [torch.full_like(t, float("nan")) for t in (q, k, v)]
        rc = L.la_bwd_carry(q.data_ptr(), k.data_ptr(), v.data_ptr(), s.data_ptr() if decay else None, do.data_ptr(), *(t.data_ptr() for t in gr), _strides(q, k, v, do, *gr),
                            b, h, n, d, e, code, ws.data_ptr() if ws_bytes else None, ws_bytes, None, cr.data_ptr(), nbytes, st)
        assert rc == 0, L.la_error_string(rc)
        return gr

    return backward, carry, ws, wb


@pytest.mark.parametrize("b, h, n, d, e, dtype, decay, token_major", CASES)
def test_the_launches_under_test_run(b, h, n, d, e, dtype, decay, token_major):
    backward, carry, ws, wb = _prepared(b, h, n, d, e, dtype, decay, token_major)
    got = backward(wb, carry)
    shared = d == e and (b, n) in ((1, 8192), (1, 9057), (1, 16384), (4, 6400))
    assert torch.isfinite(ws).any().item() == (shared or d != e)  # (d != e: dK and dV scan states of their own)
    other = backward(wb, torch.zeros_like(carry))
    assert torch.equal(got[1], other[1]) and torch.equal(got[2], other[2])
    same = (got[0] == other[0]).all(-1).all(0).all(0)  # per token
    chunk = int((~same).nonzero()[0])
    assert same[:chunk].all() and chunk % 64 == 0 and 0 < chunk < n and not same[chunk:chunk + 64].any()


@pytest.mark.parametrize("b, h, n, d", [(1, 16, 8192, 128), (4, 16, 6400, 128)])
@pytest.mark.parametrize("given", [0, 4096])
def test_carried_dq_without_a_backward_workspace(b, h, n, d, given):
    """No workspace, or one too small for the states of dK + dV: dQ from the carry as ever, dK and dV from warm-up blocks or single walks."""
    backward, carry, ws, wb = _prepared(b, h, n, d, d, torch.bfloat16, True, False)
    full, got = backward(wb, carry), None
    ws.fill_(float("nan"))
    got = backward(given, carry)
    assert not torch.isfinite(ws).any()
    assert torch.equal(got[0], full[0])
    for a, c in zip(got[1:], full[1:]):
        assert rel_norm(a, c.float()) < 3e-3


def test_carried_states_in_a_captured_step():
    """The operators under HIP graph capture, carry and workspaces in the graph's own memory: three replays over new inputs, eager work
    of the same kind and synchronisations between them, each equal to the eager result."""
    b, h, n, d = 1, 16, 4096, 128
    assert _lib.lib().la_carry_bytes(b, h, n, d, d, 0, None) > 0
    s = _build_slope_tensor(h).float().cuda()
    fresh = lambda: [torch.randn(b, h, n, d, device="cuda", dtype=torch.bfloat16) for _ in range(4)]  # noqa: E731
    q, k, v, do = fresh()
    ts = [t.requires_grad_() for t in (q, k, v)]

    def step(ts, do):
        o = lightning_attn_func(*ts, s)
        return (o,) + torch.autograd.grad(o, ts, do)

    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        step(ts, do)
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = step(ts, do)
    for _ in range(3):
        new = fresh()
        with torch.no_grad():
            for t, x in zip(ts + [do], new):
                t.copy_(x)
        graph.replay()
        torch.cuda.synchronize()
        want = step([t.clone().requires_grad_() for t in new[:3]], new[3])
        torch.cuda.synchronize()
        for a, c in zip(out, want):
            assert torch.equal(a, c)


def test_carried_states_through_autograd_twice():
    """The operators keep the states with the graph: a second backward pass over it gives the same gradients, and
    save_states=False keeps the inputs only."""
    q, k, v, do = (torch.randn(1, 16, 4096, 128, device="cuda", dtype=torch.bfloat16) for _ in range(4))
    s = _build_slope_tensor(16).float().cuda()
    ts = [t.requires_grad_() for t in (q, k, v)]
    assert _lib.lib().la_carry_bytes(1, 16, 4096, 128, 128, 0, None) > 0
    o = lightning_attn_func(*ts, s)
    g1 = torch.autograd.grad(o, ts, do, retain_graph=True)
    g2 = torch.autograd.grad(o, ts, do)
    assert all(torch.equal(a, c) for a, c in zip(g1, g2))
    with _lib.launch_opts(save_states=False):
        g3 = torch.autograd.grad(lightning_attn_func(*ts, s), ts, do)
    assert all(rel_norm(a, c.float()) < 3e-3 for a, c in zip(g1, g3))


def test_small_fp16_gradients_keep_their_bits():
    """Upstream gradients of 1e-5 in fp16 are subnormal numbers: scaled by a decay factor and rounded again they would lose
    bits that dK never lost.  dK + dV from states collected once: each within 5 % of the error (2-norm, against the block recurrence in
    64 bits) that the sweeps have on their own, the spread of either with the inputs being below 1 %."""
    b, h, n, d = 1, 16, 8192, 128
    L = _lib.lib()
    g = torch.Generator(device="cuda").manual_seed(3)
    q, k, v, do = (torch.randn(b, h, n, d, generator=g, device="cuda").half() for _ in range(4))
    do = (do.float() * 1e-5).half()
    s = _build_slope_tensor(h).float().cuda().contiguous()
    wb = L.la_workspace_bytes(1, b, h, n, d, d, 1)
    assert wb > 0

    def bwd(ws_bytes):
        gr = [torch.empty_like(q) for _ in range(3)]
        ws = torch.full((max(ws_bytes, 16) // 4,), float("nan"), device="cuda")
        rc = L.la_bwd(q.data_ptr(), k.data_ptr(), v.data_ptr(), s.data_ptr(), do.data_ptr(), *(t.data_ptr() for t in gr), b, h, n, d, d, 1,
                      ws.data_ptr() if ws_bytes else None, ws_bytes, torch.cuda.current_stream().cuda_stream)
        assert rc == 0, L.la_error_string(rc)
        return gr

    def reverse64(x, y, z):  # out_i = sum_{j>=i} lam^(j-i) (x_i . y_j) z_j, blocks of 64 from the end
        i = torch.arange(64, device="cuda", dtype=torch.float64)
        r = s.double().view(h, 1, 1)
        mask = torch.exp(-r * (i[None, :] - i[:, None]).clamp(min=0)) * (i[None, :] >= i[:, None])
        st, out = torch.zeros(h, d, d, device="cuda", dtype=torch.float64), torch.empty(h, n, d, device="cuda", dtype=torch.float64)
        for c in reversed(range(n // 64)):
            xs, ys, zs = (t[0, :, 64 * c:64 * c + 64].double().contiguous() for t in (x, y, z))
            out[:, 64 * c:64 * c + 64] = (torch.bmm(xs, ys.transpose(1, 2).contiguous()) * mask).bmm(zs) + torch.bmm(xs, st) * torch.exp(-r * (64 - i).view(1, 64, 1))
            st = st * torch.exp(-r * 64) + torch.bmm((ys * torch.exp(-r * i.view(1, 64, 1))).transpose(1, 2).contiguous(), zs)
        return out

    apart, shared = bwd(0), bwd(wb)
    for name, i, want in (("dk", 1, reverse64(v, do, q)), ("dv", 2, reverse64(k, q, do))):
        own, got = (((t[i][0].double() - want).norm() / want.norm()).item() for t in (apart, shared))
        assert got <= 1.05 * own, (name, got, own)
