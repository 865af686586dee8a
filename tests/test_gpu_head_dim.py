"""Head dims that are neither 64 nor 128, run on rows of their own length: the
step (with GdO) against the float64 closed forms, with and without split
walks, from strided operands, and through a window and a mask."""
import pytest
import torch

from oracle import closed_form
from tests._util import check, check_f32_scaled, to_np
from testtimeideas_amd import _lib
from testtimeideas_amd.ttt_e2e.attention import gradgrad_attention, windowed_attention
from testtimeideas_amd.ttt_kernels.triton_attention import triton_attention

pytestmark = pytest.mark.gpu
NAMES = ("o", "dq", "dk", "dv", "gq", "gk", "gv", "gdo")


def _inputs(d, t, dtype, strided):
    gen = torch.Generator().manual_seed(d * 1000 + t)
    out = []
    for _ in range(7):
        x = torch.randn((2, t, 3, d) if strided else (2, 3, t, d), generator=gen).to(dtype)
        out.append(x.cuda().transpose(1, 2) if strided else x.cuda())
    return out


def _want(xs, causal, bias=None):
    n = [to_np(x) for x in xs]
    d = xs[0].size(-1)
    first = closed_form.backward(*n[:4], causal, d ** -0.5, bias)
    second = closed_form.double_backward(*n, causal, d ** -0.5, bias)
    return [first[k] for k in NAMES[:4]] + [second[k] for k in NAMES[4:]]


def _compare(xs, attend, want, dtype, what):
    q, k, v, do = (x.detach().requires_grad_() for x in xs[:4])
    o = attend(q, k, v)
    first = torch.autograd.grad(o, (q, k, v), do, create_graph=True)
    second = torch.autograd.grad(first, (q, k, v, do), xs[4:])
    for name, a, w in zip(NAMES, [o, *first, *second], want):
        assert a.shape == w.shape
        if dtype == torch.float32:
            check_f32_scaled(f"{name} {what}", a, w)
        else:
            check(f"{name} {what}", a, w, dtype)


@pytest.mark.parametrize("d", [8, 40, 72, 96, 120, 20])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("t,causal,strided", [(65, True, False), (130, False, True), (191, True, True)])
def test_step(d, dtype, t, causal, strided):
    xs = _inputs(d, t, dtype, strided)
    want = _want(xs, causal)
    for mode, split in (("recompute", 0), ("recompute", 1), ("save_p", 0), ("save_p", 2)):
        with _lib.split_chunk(split):
            _compare(xs, lambda q, k, v: triton_attention(q, k, v, causal=causal, bwd_mode=mode), want, dtype,
                     f"{mode} split {split}")


@pytest.mark.parametrize("d", [24, 88])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_window_and_mask(d, dtype):
    t, w = 150, 48
    xs = _inputs(d, t, dtype, False)
    i = torch.arange(t)
    hidden = (i[None] > i[:, None]) | (i[:, None] - i[None] >= w)
    m = torch.zeros(t, t).masked_fill(hidden, float("-inf"))
    want = _want(xs, False, to_np(m))
    _compare(xs, lambda q, k, v: windowed_attention(q, k, v, w, local=False), want, dtype, "window")
    _compare(xs, lambda q, k, v: gradgrad_attention(q, k, v, m.cuda().to(dtype)), want, dtype, "mask")
