"""Forced splits, kernel timing and tuning apply to the double backward as they
stand when it runs, whatever held when the first backward did."""
import pytest
import torch

from testtimeideas_amd import _lib, autotune
from testtimeideas_amd.ttt_kernels.triton_attention import triton_attention

pytestmark = pytest.mark.gpu


def test_double_backward_takes_the_state_it_finds():
    g = torch.Generator().manual_seed(3)
    xs = [torch.randn((1, 2, 512, 64), generator=g).to(torch.float16).cuda() for _ in range(7)]
    q, k, v = (x.requires_grad_() for x in xs[:3])

    def second(first_in, second_in):
        with first_in:
            o = triton_attention(q, k, v, causal=True)
            first = torch.autograd.grad(o, (q, k, v), xs[3], create_graph=True)
        with second_in:
            return torch.autograd.grad(first, (q, k, v), xs[4:])

    o = triton_attention(q, k, v, causal=True)
    first = torch.autograd.grad(o, (q, k, v), xs[3], create_graph=True)
    with _lib.kernel_timing() as rec:
        torch.autograd.grad(first, (q, k, v), xs[4:])
    assert set(rec) == {"ttt_attn_gg_row", "ttt_attn_gg_col"}
    # a split forced around the double backward alone: the Python Function's result under the same split
    got = second(_lib.split_chunk(0), _lib.split_chunk(1))
    want = second(_lib.kernel_timing(), _lib.split_chunk(1))
    whole = second(_lib.split_chunk(0), _lib.split_chunk(64))
    for a, b in zip(got, want):
        assert torch.equal(a, b)
    assert any(not torch.equal(a, b) for a, b in zip(got, whole))
    prev = autotune.enabled()
    o = triton_attention(q, k, v, causal=True)
    first = torch.autograd.grad(o, (q, k, v), xs[3], create_graph=True)
    autotune.enable(True)
    autotune.clear()
    try:
        torch.autograd.grad(first, (q, k, v), xs[4:])
        assert len(autotune.choices()) == 2
    finally:
        autotune.enable(prev)
        autotune.clear()
