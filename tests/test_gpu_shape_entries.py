"""Key counts other than the query count and head dims other than 64 and 128
through the per-kernel entry points: kernel timing brackets every kernel and
autotuning tunes every family."""
import pytest
import torch

from oracle import math_path
from testtimeideas_amd import _lib, autotune
from testtimeideas_amd.ttt_e2e.attention import gradgrad_attention
from tests._util import check

pytestmark = pytest.mark.gpu
KERNELS = {"ttt_attn_fwd", "ttt_attn_bwd_dq", "ttt_attn_bwd_dkdv", "ttt_attn_gg_row", "ttt_attn_gg_col"}
NAMES = ("o", "dq", "dk", "dv", "gq", "gk", "gv")


def _inputs(lq, lk, d, dtype):
    g = torch.Generator().manual_seed(lq + lk + d)
    return [torch.randn((1, 2, n, d), generator=g).to(dtype) for n in (lq, lk, lk, lq, lq, lk, lk)]


def _step(xs, mode):
    q, k, v = (x.cuda().requires_grad_() for x in xs[:3])
    o = gradgrad_attention(q, k, v, bwd_mode=mode)
    first = torch.autograd.grad(o, (q, k, v), xs[3].cuda(), create_graph=True)
    return [x.detach() for x in (o, *first, *torch.autograd.grad(first, (q, k, v), [x.cuda() for x in xs[4:]]))]


SHAPES = [(200, 1000, 64, torch.float16), (700, 200, 128, torch.bfloat16), (600, 600, 80, torch.bfloat16),
          (500, 900, 40, torch.float32)]


@pytest.mark.parametrize("lq,lk,d,dtype", SHAPES)
@pytest.mark.parametrize("mode", ["recompute", "save_p"])
def test_every_kernel_is_timed(lq, lk, d, dtype, mode):
    xs = _inputs(lq, lk, d, dtype)
    want = _step(xs, mode)
    with _lib.kernel_timing() as rec:
        got = _step(xs, mode)
    torch.cuda.synchronize()
    assert set(rec) == KERNELS
    for name, a, b in zip(NAMES, got, want):
        check(name, a, b, dtype, rel_tol=5e-3)  # one call or two: the fused ones share a workspace and its split


@pytest.mark.parametrize("lq,lk,d,dtype", SHAPES)
@pytest.mark.parametrize("mode", ["recompute", "save_p"])
def test_autotuned(lq, lk, d, dtype, mode):
    xs = _inputs(lq, lk, d, dtype)
    ref = math_path.gradgrad_step(*(x.double() for x in xs), False, d ** -0.5)
    prev = autotune.enabled()
    autotune.enable(True)
    autotune.clear()
    try:
        first = _step(xs, mode)
        chosen = autotune.choices()
        assert len(chosen) == 5, chosen
        second, third = _step(xs, mode), _step(xs, mode)
        assert autotune.choices() == chosen
        # another key count is another problem
        _step([x[:, :, :70] if i in (1, 2, 5, 6) else x for i, x in enumerate(xs)], mode)
        assert len(autotune.choices()) == 10
    finally:
        autotune.enable(prev)
        autotune.clear()
    for name, a, b, c in zip(NAMES, first, second, third):
        check(name, a, ref[name], dtype)
        assert torch.equal(b, c), name
