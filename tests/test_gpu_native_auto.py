"""lightning_attn_func / lightning_attn_silu_func through one native call (attn_auto, attn_silu_auto) against the Python operators: every
form that the call takes as it is, every form that it hands back, and the errors of those that nobody takes."""
import pytest
import torch

pytestmark = pytest.mark.gpu

from lightning_attn.ops import SimpleRMSNorm, lightning_attn_func, lightning_attn_silu_func  # noqa: E402
from lightning_attn.ops.hip import _lib  # noqa: E402


def _t(shape, dtype, form="plain"):
    g = torch.Generator().manual_seed(sum(shape))
    t = torch.randn(*shape, generator=g).to(dtype).cuda()
    if form == "tokens_first":
        t = t.transpose(1, 2).contiguous().transpose(1, 2)
    elif form == "off_grid":  # dense, but not 16-byte aligned
        t = torch.cat([t.new_zeros(1), t.reshape(-1)])[1:].view(shape)
    elif form == "expanded":
        t = t[:, :1].expand(shape)
    return t


@pytest.mark.parametrize("form", ["plain", "tokens_first", "off_grid", "expanded"])
@pytest.mark.parametrize("dtype,d,e", [(torch.bfloat16, 64, 64), (torch.float16, 128, 40), (torch.float32, 32, 128), (torch.float32, 136, 16), (torch.bfloat16, 20, 64),
                                       (torch.bfloat16, 64, 264), (torch.float16, 264, 8), (torch.bfloat16, 200, 256)])
@pytest.mark.parametrize("decay", [True, False])
def test_same_as_the_python_operators(form, dtype, d, e, decay):
    q, k, v, do = (_t((2, 3, 70, c), dtype, form) for c in (d, d, e, e))
    s = torch.tensor([[0.1], [0.2], [0.5]], dtype=torch.float64) if decay else None  # (any shape, type and device with h elements)
    ops = _lib.native_ops()
    taken = ops.attn_auto(q, k, v, s) is not None
    widest = 128 if dtype == torch.float32 else 256
    assert taken == (d % 8 == 0 and e % 8 == 0 and d <= widest and e <= widest)
    got = []
    for native in (True, False):
        prev = _lib.use_native_ops(native)
        try:
            leaves = [t.detach().requires_grad_() for t in (q, k, v)]
            o = lightning_attn_func(*leaves, s)
            with torch.no_grad():
                got.append((o.detach(), lightning_attn_func(q, k, v, s), lightning_attn_silu_func(q, k, v, s)) + torch.autograd.grad(o, leaves, do))
        finally:
            _lib.use_native_ops(prev)
    for a, b in zip(*got):
        assert torch.equal(a, b) and a.stride() == b.stride()


def test_handed_back_and_refused():
    q, k, v = (_t((1, 2, 66, 64), torch.bfloat16) for _ in range(3))
    s = torch.tensor([0.1, 0.2], device="cuda")
    ops = _lib.native_ops()
    for a in ((q, k.float(), v, s), (q, k[:, :, :-1], v, s), (q, k, v[:, :1], s), (q, k, v, s[:1]), (q[0], k[0], v[0], s), (q.cpu(), k, v, s), (q.double(), k.double(), v.double(), s)):
        assert ops.attn_auto(*a) is None and ops.attn_silu_auto(*a) is None
        with pytest.raises((ValueError, TypeError, RuntimeError)):
            lightning_attn_func(*a)
    assert ops.attn_silu_auto(q.clone().requires_grad_(), k, v, s) is None and ops.attn_silu_auto(q.float(), k.float(), v.float(), s) is None
    with pytest.raises(AttributeError):
        lightning_attn_func(None, k, v, s)
    with _lib.launch_opts(chunks=2):
        assert _lib.plain_ops() is None
    assert lightning_attn_func(q[:, :, :0], k[:, :, :0], v[:, :, :0], s).shape == (1, 2, 0, 64)


@pytest.mark.parametrize("shape", [(7,), (3, 40), (2, 0, 16), (2, 3, 5, 24), (1, 1, 8)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_norm_of_any_number_of_dims(shape, dtype):
    for x in (_t(shape, dtype), _t(shape + (2,), dtype)[..., 0], _t(tuple(reversed(shape)), dtype).permute(*reversed(range(len(shape))))):
        got = []
        for native in (True, False):
            prev = _lib.use_native_ops(native)
            try:
                leaf = x.detach().requires_grad_()
                y = SimpleRMSNorm(shape[-1])(leaf)
                got.append((y.detach(),) + torch.autograd.grad(y, leaf, torch.ones_like(y)))
            finally:
                _lib.use_native_ops(prev)
        for a, b in zip(*got):
            assert a.shape == b.shape and torch.equal(a, b)


@pytest.mark.filterwarnings("ignore::torch.jit.TracerWarning", "ignore::DeprecationWarning")
def test_traced_calls():
    q, k, v, do = (_t((2, 3, 70, 64), torch.bfloat16) for _ in range(4))
    s = torch.tensor([0.1, 0.2, 0.5], device="cuda")
    leaves = [t.clone().requires_grad_() for t in (q, k, v)]
    traced = torch.jit.trace(lambda q, k, v, s: lightning_attn_func(q, k, v, s), (*leaves, s), check_trace=False)
    got, want = (f(*leaves, s) for f in (traced, lightning_attn_func))
    assert torch.equal(got, want)
    for a, b in zip(torch.autograd.grad(got, leaves, do), torch.autograd.grad(want, leaves, do)):
        assert torch.equal(a, b)
    with torch.no_grad():
        traced = torch.jit.trace(lambda q, k, v, s: lightning_attn_silu_func(q, k, v, s), (q, k, v, s), check_trace=False)
        assert torch.equal(traced(q * 2, k, v, s), lightning_attn_silu_func(q * 2, k, v, s))


@pytest.mark.filterwarnings("ignore:There is a performance drop")
def test_mapped_calls():
    q, k, v = (_t((4, 2, 3, 70, 64), torch.bfloat16).roll(i, 0) for i in range(3))
    s = torch.tensor([0.1, 0.2, 0.5], device="cuda")
    for f in (lightning_attn_func, lightning_attn_silu_func):
        got = torch.vmap(f, in_dims=(0, 0, 0, None))(q, k, v, s)
        assert torch.equal(got, torch.stack([f(q[i], k[i], v[i], s) for i in range(4)]))
