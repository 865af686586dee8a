"""A saved P that passes through saved-tensor hooks comes back without the row
storage the forward gave it: rows that start on no 16-byte boundary, or that
end with their last element.  The step is bitwise the same."""
import pytest
import torch

from testtimeideas_amd import _lib
from testtimeideas_amd.ttt_e2e.attention import gradgrad_attention
from testtimeideas_amd.ttt_kernels.triton_attention import triton_attention

pytestmark = pytest.mark.gpu


def _step(xs, attend):
    q, k, v, do = (x.clone().requires_grad_() for x in xs[:4])
    o = attend(q, k, v)
    first = torch.autograd.grad(o, (q, k, v), do, create_graph=True)
    return [o, *first, *torch.autograd.grad(first, (q, k, v, do), xs[4:])]


# rows of 193 elements are unaligned in every type; fp32 rows of 196 are aligned, and their last run of eight is not
@pytest.mark.parametrize("dtype,tk", [(torch.float16, 193), (torch.bfloat16, 196), (torch.float32, 193),
                                      (torch.float32, 196), (torch.float16, 200)])
@pytest.mark.parametrize("lq", [None, 70])
@pytest.mark.parametrize("timed", [False, True])
def test_saved_p_in_another_layout(dtype, tk, lq, timed):
    gen = torch.Generator().manual_seed(tk)
    lq = lq or tk
    xs = [torch.randn((1, 3, n, 64), generator=gen).to(dtype).cuda() for n in (lq, tk, tk, lq, lq, tk, tk)]
    if lq == tk:
        attend = lambda q, k, v: triton_attention(q, k, v, causal=True, bwd_mode="save_p")
    else:
        attend = lambda q, k, v: gradgrad_attention(q, k, v, bwd_mode="save_p")
    want = _step(xs, attend)

    def run():
        with torch.autograd.graph.saved_tensors_hooks(lambda t: t.cpu().contiguous(), lambda t: t.cuda()):
            return _step(xs, attend)

    if timed:
        with _lib.kernel_timing():
            got = run()
    else:
        got = run()
    for a, b in zip(got, want):
        assert torch.equal(a, b)
