"""The differentiable first backward that runs without the interpreter
(``bwd_graph`` of the binding) against the Python Function of the same role,
which kernel timing takes: bitwise the same outputs, for whatever part of them
is differentiated, and the same autograd behaviour around them."""
import pytest
import torch

from testtimeideas_amd import _lib
from testtimeideas_amd.ttt_e2e.attention import gradgrad_attention, windowed_attention
from testtimeideas_amd.ttt_kernels.triton_attention import triton_attention

pytestmark = pytest.mark.gpu


def _inputs(t=193, d=64, dtype=torch.float16, seed=0):
    gen = torch.Generator().manual_seed(seed)
    return [torch.randn((1, 3, t, d), generator=gen).to(dtype).cuda() for _ in range(7)]


ATTEND = {
    "save_p": lambda q, k, v: triton_attention(q, k, v, causal=True, bwd_mode="save_p"),
    "recompute": lambda q, k, v: triton_attention(q, k, v, causal=False),
    "window": lambda q, k, v: windowed_attention(q, k, v, 64),
    "mask": lambda q, k, v: gradgrad_attention(q, k, v, torch.zeros(q.size(-2), device="cuda", dtype=q.dtype)),
}


def _step(xs, attend, pick=(0, 1, 2), want_gdo=True):
    q, k, v, do = (x.clone().requires_grad_(i < 3 or want_gdo) for i, x in enumerate(xs[:4]))
    o = attend(q, k, v)
    first = torch.autograd.grad(o, (q, k, v), do, create_graph=True)
    wrt = (q, k, v, do) if want_gdo else (q, k, v)
    second = torch.autograd.grad([first[i] for i in pick], wrt, [xs[4 + i] for i in pick])
    return [o, *first, *second]


@pytest.mark.parametrize("name", sorted(ATTEND))
@pytest.mark.parametrize("d", [64, 80])
@pytest.mark.parametrize("want_gdo", [False, True])
def test_same_as_python_function(name, d, want_gdo):
    xs = _inputs(d=d)
    for pick in ((0, 1, 2), (1,), (0, 2)):
        got = _step(xs, ATTEND[name], pick, want_gdo)
        assert "AttnBwdFn" not in type(got[1].grad_fn).__name__
        with _lib.kernel_timing():
            want = _step(xs, ATTEND[name], pick, want_gdo)
        assert type(want[1].grad_fn).__name__ == "_AttnBwdFnBackward"
        for a, b in zip(got, want):
            assert torch.equal(a, b)


def test_only_some_inputs_need_gradients():
    xs = _inputs()
    q, k, v = xs[0].requires_grad_(), xs[1], xs[2]
    o = triton_attention(q, k, v, causal=True)
    (dq,) = torch.autograd.grad(o, (q,), xs[3], create_graph=True)
    (gq,) = torch.autograd.grad(dq, (q,), xs[4])
    assert gq.shape == q.shape and torch.isfinite(gq).all()


def test_third_derivative_raises():
    xs = _inputs(t=70)
    q, k, v = (x.requires_grad_() for x in xs[:3])
    o = triton_attention(q, k, v, causal=True)
    dq, _, _ = torch.autograd.grad(o, (q, k, v), xs[3], create_graph=True)
    r = xs[4].requires_grad_()
    (gq,) = torch.autograd.grad(dq, (q,), r, create_graph=True)
    with pytest.raises(RuntimeError, match="differentiate twice"):
        gq.sum().backward()


def test_saved_tensor_hooks_see_the_saved_tensors():
    xs = _inputs(t=128)  # a multiple of 8: a copy of P then keeps the row stride the kernels take
    want = _step(xs, ATTEND["save_p"])
    seen = []

    def pack(t):
        seen.append(t.shape)
        return t.cpu()

    with torch.autograd.graph.saved_tensors_hooks(pack, lambda t: t.cuda()):
        got = _step(xs, ATTEND["save_p"])
    assert len(seen) >= 12  # the forward's and the first backward's
    for a, b in zip(got, want):
        assert torch.equal(a, b)


def test_freed_graph_raises():
    xs = _inputs(t=70)
    q, k, v = (x.requires_grad_() for x in xs[:3])
    o = triton_attention(q, k, v, causal=True)
    first = torch.autograd.grad(o, (q, k, v), xs[3], create_graph=True)
    torch.autograd.grad(first, (q, k, v), xs[4:])
    with pytest.raises(RuntimeError, match="second time"):
        torch.autograd.grad(first, (q, k, v), xs[4:])
