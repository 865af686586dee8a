"""fp32 products formed from bf16 parts on the matrix cores: the full step
against the float64 closed forms, over tile edges and over operands whose
columns differ by many orders of magnitude."""
import pytest
import torch

from oracle import closed_form
from tests._util import MAX_ABS_32, to_np
from testtimeideas_amd.ttt_kernels.triton_attention import triton_attention

pytestmark = pytest.mark.gpu


def _step(xs, causal, mode):
    q, k, v = (x.clone().requires_grad_() for x in xs[:3])
    o = triton_attention(q, k, v, causal=causal, bwd_mode=mode)
    first = torch.autograd.grad(o, (q, k, v), xs[3], create_graph=True)
    return [o.detach(), *(g.detach() for g in first), *torch.autograd.grad(first, (q, k, v), xs[4:])]


# A product of length L carries at most (L + 2) 2^-24 of its terms' absolute
# sum in fp32; L <= 193 here and the terms are of random sign, so 2e-6 of the
# result's norm holds with room (measured: below 5e-7).
@pytest.mark.parametrize("d", [32, 64])
@pytest.mark.parametrize("t,causal", [(1, True), (63, False), (64, True), (65, True), (193, False)])
@pytest.mark.parametrize("mode", ["recompute", "save_p"])
def test_step_against_float64(d, t, causal, mode):
    g = torch.Generator().manual_seed(t + d)
    xs = [torch.randn((1, 2, t, d), generator=g) for _ in range(7)]
    got = _step([x.cuda() for x in xs], causal, mode)
    n = [to_np(x) for x in xs]
    first = closed_form.backward(*n[:4], causal, d ** -0.5)
    second = closed_form.double_backward(*n, causal, d ** -0.5)
    want = [first[k] for k in ("o", "dq", "dk", "dv")] + [second[k] for k in ("gq", "gk", "gv")]
    for name, a, b in zip(("o", "dq", "dk", "dv", "gq", "gk", "gv"), got, want):
        b = torch.from_numpy(b)
        err = a.double().cpu() - b
        if t == 1:  # dS, and with it dQ, dK, GQ and GK, cancels exactly: the suite's fp32 bound on what is left
            assert err.abs().max() <= MAX_ABS_32, (name, float(err.abs().max()))
        else:
            assert err.norm() <= 2e-6 * b.norm(), (name, float(err.norm()), float(b.norm()))


def test_columns_of_any_magnitude_keep_their_precision():
    # O's column j is P . V's column j, so each keeps fp32's relative precision whatever its scale.
    t, d = 130, 64
    g = torch.Generator().manual_seed(0)
    q, k, v = (torch.randn((1, 1, t, d), generator=g) for _ in range(3))
    mul = torch.ldexp(torch.ones(d), torch.linspace(-100, 100, d).round().to(torch.int32))
    v = v * mul
    o = triton_attention(q.cuda(), k.cuda(), v.cuda(), causal=True).double().cpu()
    s = (q.double() @ k.double().transpose(-1, -2)) * d ** -0.5
    s = s.masked_fill(torch.ones(t, t, dtype=torch.bool).triu(1), float("-inf"))
    want = torch.softmax(s, -1) @ v.double()
    rel = (o - want).norm(dim=-2) / want.norm(dim=-2)
    assert float(rel.max()) < 2e-6
