"""Fewer or more keys than queries, run as they are: the step (with GdO)
through ``gradgrad_attention`` against the float64 closed forms, at the edges
of the 64-row tiles on either side, with and without split walks."""
import pytest
import torch

from oracle import closed_form
from tests._util import MAX_ABS_32, check, check_f32_scaled, to_np
from testtimeideas_amd import _lib
from testtimeideas_amd.ttt_e2e.attention import gradgrad_attention

pytestmark = pytest.mark.gpu


def _mask(kind, lq, lk, gen):
    if kind == "none":
        return None
    if kind == "padding":
        m = torch.zeros(2, 1, 1, lk)
        m[1, ..., (lk + 1) // 2:] = float("-inf")
        return m
    if kind == "full":
        return torch.randn((1, 2, lq, lk), generator=gen)
    q = torch.arange(lq)[:, None] + max(0, lk - lq)  # each query sees its own key and those before it
    return torch.zeros(lq, lk).masked_fill(torch.arange(lk)[None] > q, float("-inf"))


@pytest.mark.parametrize("lq,lk", [(1, 130), (65, 64), (64, 129), (200, 63), (3, 700), (700, 5), (130, 1)])
@pytest.mark.parametrize("dtype,d", [(torch.float32, 64), (torch.float16, 64), (torch.bfloat16, 128),
                                     (torch.float32, 128)])
@pytest.mark.parametrize("mask", ["none", "padding", "full", "causal"])
def test_rectangular_step(lq, lk, dtype, d, mask):
    gen = torch.Generator().manual_seed(lq * 1000 + lk)
    b, h = 2, 2
    rows = (lq, lk, lk, lq, lq, lk, lk)
    xs = [torch.randn((b, h, n, d), generator=gen).to(dtype) for n in rows]
    m = _mask(mask, lq, lk, gen)
    mt = None if m is None else m.to(dtype)
    n = [to_np(x) for x in xs]
    bias = None if m is None else to_np(mt)
    first = closed_form.backward(*n[:4], False, d ** -0.5, bias)
    second = closed_form.double_backward(*n, False, d ** -0.5, bias)
    want = [first[k] for k in ("o", "dq", "dk", "dv")] + [second[k] for k in ("gq", "gk", "gv", "gdo")]
    # One key in 16 bits: dS, gS and gdP are differences of rounded terms that cancel exactly, which only fp32 pins.
    cancel = ("dq", "dk", "gq", "gk", "gv") if lk == 1 and dtype != torch.float32 else ()
    dev = [x.cuda() for x in xs]
    for mode, split in (("recompute", 0), ("recompute", 1), ("save_p", 0), ("save_p", 2)):
        q, k, v, do = (x.clone().requires_grad_() for x in dev[:4])
        with _lib.split_chunk(split):
            o = gradgrad_attention(q, k, v, None if mt is None else mt.cuda(), bwd_mode=mode)
            if mode == "save_p":
                assert tuple(o.grad_fn.saved_probs[0].shape) == (b, h, lq, lk)
            f = torch.autograd.grad(o, (q, k, v), do, create_graph=True)
            g = torch.autograd.grad(f, (q, k, v, do), dev[4:])
        for name, a, w in zip(("o", "dq", "dk", "dv", "gq", "gk", "gv", "gdo"), [o, *f, *g], want):
            # With one key P = 1 and dS, gS cancel to 0.  In fp32 each query leaves 2^-24 of the products that
            # cancel (|dP|, |gP| up to ~30, times a cotangent), of random sign, and dK and GK sum lq of them.
            # Elsewhere the key gradients sum up to 700 queries for few keys and reach 10 and more: fp32's bound is
            # then relative to the largest.
            if name in cancel:
                continue
            if dtype == torch.float32:
                check_f32_scaled(f"{name} {mode} split {split}", a, w, MAX_ABS_32 * (lq ** 0.5 if lk == 1 else 1.0))
            else:
                check(f"{name} {mode} split {split}", a, w, dtype)
