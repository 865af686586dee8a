"""The double backward in the form of a step whose dO is a constant (GQ from the
first backward's dQ, no GdO), against the float64 closed forms: Tq != Tk, rows
of d < 128 columns, both at once, with and without split walks; and windows at
scales of either sign."""
import pytest
import torch

from oracle import closed_form, masks
from tests._util import ZERO_RMS, check, check_f32_scaled, to_np
from testtimeideas_amd import _lib
from testtimeideas_amd.ttt_e2e.attention import gradgrad_attention, windowed_attention
from testtimeideas_amd.ttt_kernels.triton_attention import triton_attention

pytestmark = pytest.mark.gpu
NAMES = ("o", "dq", "dk", "dv", "gq", "gk", "gv")


def _inputs(lq, lk, d, dtype):
    gen = torch.Generator().manual_seed(lq * 1000 + lk + d)
    return [torch.randn((2, 2, n, d), generator=gen).to(dtype) for n in (lq, lk, lk, lq, lq, lk, lk)], gen


def _want(xs, causal, scale, bias=None):
    n = [to_np(x) for x in xs]
    first = closed_form.backward(*n[:4], causal, scale, bias)
    second = closed_form.double_backward(*n, causal, scale, bias)
    return [first[k] for k in NAMES[:4]] + [second[k] for k in NAMES[4:]]


def _check_step(xs, attend, want, what, split=0, skip=()):
    q, k, v = (x.cuda().requires_grad_() for x in xs[:3])
    with _lib.split_chunk(split):
        o = attend(q, k, v)
        first = torch.autograd.grad(o, (q, k, v), xs[3].cuda(), create_graph=True)
        second = torch.autograd.grad(first, (q, k, v), [x.cuda() for x in xs[4:]])
    for name, a, w in zip(NAMES, [o, *first, *second], want):
        assert a.shape == w.shape
        if name in skip:
            continue
        if xs[0].dtype == torch.float32:
            check_f32_scaled(f"{name} {what}", a, w)
        else:
            check(f"{name} {what}", a, w, xs[0].dtype)


@pytest.mark.parametrize("lq,lk", [(1, 130), (64, 129), (200, 63), (300, 700), (700, 5), (130, 1)])
@pytest.mark.parametrize("dtype,d", [(torch.float32, 64), (torch.float32, 40), (torch.float16, 64),
                                     (torch.bfloat16, 128), (torch.bfloat16, 96), (torch.float16, 80),
                                     (torch.bfloat16, 24)])
@pytest.mark.parametrize("masked", [False, True])
def test_rectangular(lq, lk, dtype, d, masked):
    xs, gen = _inputs(lq, lk, d, dtype)
    mask = torch.randn((1, 2, lq, lk), generator=gen).to(dtype) if masked else None
    want = _want(xs, False, d ** -0.5, to_np(mask) if masked else None)
    # One key: P = 1, and dS, gS and gdP = P (gdS - E) cancel to 0, and with them dQ, dK, GQ, GK and GV.  In 16 bits
    # only what does not cancel is comparable (O, dV); in fp32 dQ and GQ too, each a single product of 2^-24 of the
    # terms that cancel, where dK, GK and GV sum one for every query.
    skip = () if lk > 1 else ("dk", "gk", "gv") if dtype == torch.float32 else ("dq", "dk", "gq", "gk", "gv")
    for mode, split in (("recompute", 0), ("recompute", 1), ("save_p", 0), ("save_p", 2)):
        _check_step(xs, lambda q, k, v: gradgrad_attention(q, k, v, None if mask is None else mask.cuda(),
                                                           bwd_mode=mode), want, f"{mode} split {split}", split, skip)


@pytest.mark.parametrize("t,causal", [(65, True), (191, False), (330, True)])
@pytest.mark.parametrize("dtype,d", [(torch.float16, 96), (torch.bfloat16, 72), (torch.float16, 120),
                                     (torch.bfloat16, 40), (torch.float32, 48)])
def test_square(t, causal, dtype, d):
    xs, _ = _inputs(t, t, d, dtype)
    want = _want(xs, causal, d ** -0.5)
    for mode, split in (("recompute", 0), ("recompute", 1), ("save_p", 0), ("save_p", 2)):
        _check_step(xs, lambda q, k, v: triton_attention(q, k, v, causal=causal, bwd_mode=mode), want,
                    f"{mode} split {split}", split)


@pytest.mark.parametrize("scale", [0.3, -0.2, 0.0])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("local", [True, False])
@pytest.mark.parametrize("mode", ["recompute", "save_p"])
def test_window_scales(scale, dtype, local, mode):
    t, w = 330, 100
    xs, _ = _inputs(t, t, 64, dtype)
    bias = masks.local_bias(t, w) if local else masks.window_bias(t, w)
    want = _want(xs, False, scale, bias)
    assert scale == 0.0 or all(float((x * x).mean()) ** 0.5 > ZERO_RMS for x in want)
    for split in (0, 1):
        _check_step(xs, lambda q, k, v: windowed_attention(q, k, v, w, local=local, scale=scale, bwd_mode=mode), want,
                    f"split {split}", split)


@pytest.mark.parametrize("t", [15, 17, 80, 97, 113, 129])  # last tiles of 15, 17, 16, 33, 49 and 1 keys
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("form", ["plain", "window", "bias"])
@pytest.mark.parametrize("mode", ["recompute", "save_p"])
def test_last_tiles_with_gdo(t, dtype, form, mode):
    """Head dim 128, whose streamed tiles load in four slices of 16 keys."""
    xs, gen = _inputs(t, t, 128, dtype)
    bias = masks.local_bias(t, 16) if form == "window" else None
    mask = torch.randn((1, 2, t, t), generator=gen).to(dtype) if form == "bias" else None
    n = [to_np(x) for x in xs]
    r = closed_form.double_backward(*n, False, 128 ** -0.5, to_np(mask) if mask is not None else bias)
    q, k, v, do = (x.cuda().requires_grad_() for x in xs[:4])
    if form == "window":
        o = windowed_attention(q, k, v, 16, local=True, scale=128 ** -0.5, bwd_mode=mode)
    else:
        o = gradgrad_attention(q, k, v, None if mask is None else mask.cuda(), bwd_mode=mode)
    first = torch.autograd.grad(o, (q, k, v), do, create_graph=True)
    gx = [x.cuda() for x in xs[4:]]
    second = torch.autograd.grad(first, (q, k, v, do), gx, retain_graph=True)
    no_gdo = torch.autograd.grad(first, (q, k, v), gx)
    for names, got in ((("gq", "gk", "gv", "gdo"), second), (("gq", "gk", "gv"), no_gdo)):
        for name, a in zip(names, got):
            if dtype == torch.float32:
                check_f32_scaled(f"{name} {len(got)}", a, r[name])
            else:
                check(f"{name} {len(got)}", a, r[name], dtype)
