"""A key window against the same mask as an additive bias: both forwards shift
each row by its running maximum over the same tiles and round the scaled
scores alike, so O, LSE and P agree bit for bit, whatever the scale's sign."""
import pytest
import torch

from oracle import masks
from testtimeideas_amd import _lib

pytestmark = pytest.mark.gpu


# The O + LSE pass takes tiles one by one; the pass that writes P takes them in pairs, so there every row block's
# window starts on a pair: a local window of two tiles, of which T is a multiple.
@pytest.mark.parametrize("kind,t,w,want_p", [(_lib.WINDOW_LOCAL, 449, 128, False), (_lib.WINDOW_SLIDING, 449, 100, False),
                                             (_lib.WINDOW_LOCAL, 512, 128, True)])
@pytest.mark.parametrize("dtype,d", [(torch.bfloat16, 64), (torch.float16, 64), (torch.bfloat16, 128),
                                     (torch.float32, 64), (torch.float32, 128)])
@pytest.mark.parametrize("scale", [0.125, 0.3, -0.2, 0.0])
def test_window_is_its_additive_mask(kind, t, w, want_p, dtype, d, scale):
    g = torch.Generator().manual_seed(w + d)
    q, k, v = (torch.randn((1, 2, t, d), generator=g).to(dtype).cuda() for _ in range(3))
    bias = torch.from_numpy(masks.window_bias(t, w) if kind == _lib.WINDOW_SLIDING else masks.local_bias(t, w))
    bias = _lib.prep_bias(bias, 1, 2, t, dtype, "cuda")
    with _lib.split_chunk(64):  # whole walks
        o, lse, p = _lib.fwd(q, k, v, _lib.Mask(causal=True, window=w, window_kind=kind), scale, want_p)
        ob, lseb, pb = _lib.fwd(q, k, v, _lib.Mask(causal=True, bias=bias), scale, want_p)
    assert torch.isfinite(o).all() and torch.isfinite(lse).all()
    assert torch.equal(o, ob)
    assert torch.equal(lse, lseb)
    if want_p:
        seen = torch.isfinite(bias[0, 0])
        assert torch.equal(p[..., seen], pb[..., seen])
