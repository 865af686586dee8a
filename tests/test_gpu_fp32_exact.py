"""fp32 at head dims up to 64, whose products are formed from bf16 parts: one
term keeps fp32's relative precision, and infinities and NaN give what fp32
products give (the head dim 128 kernels, which form them, on the same operands
with zero columns behind them)."""
import pytest
import torch

from testtimeideas_amd import _lib
from testtimeideas_amd.ttt_kernels.triton_attention import triton_attention

pytestmark = pytest.mark.gpu


def test_one_term_products():
    # Queries with one nonzero column against one key: LSE = q k, one product.  The significands' low 16 bits
    # (0xff7f) give parts whose smallest products all have one sign and are as large as they come, so what is left
    # out of a product shows in the mean, where roundings do not: the constants log2(e) and ln(2) in fp32 leave
    # 1.1e-8 of it, products of parts below 2^-24 would leave up to 2.4e-7.
    h, t, d = 64, 64, 64
    g = torch.Generator().manual_seed(0)

    def values(shape):
        bits = (torch.randint(0, 8, shape, generator=g) << 16) + 0xFF7F
        x = 1.0 + bits.double() * 2.0 ** -23
        sign = torch.randint(0, 2, shape, generator=g) * 2 - 1
        return x * sign * 2.0 ** torch.randint(-2, 2, shape, generator=g)

    x, y = values((h, t)), values((h, 1))
    col = torch.randint(0, d, (h, 1, 1), generator=g)
    q = torch.zeros(1, h, t, d).scatter_(3, col.expand(h, t, 1)[None], x.float()[None, ..., None])
    k = torch.zeros(1, h, 1, d).scatter_(3, col[None], y.float()[None, ..., None])
    _, lse, _ = _lib.fwd(q.cuda(), k.cuda(), k.cuda(), _lib.Mask(causal=False), 1.0, False)
    want = x * y
    rel = (lse[0].double().cpu() - want) / want
    assert abs(float(rel.mean())) <= 2.0 ** -24
    # product, scaling, logarithm's sum, scaling back: four roundings and the constants
    assert float(rel.abs().max()) <= 4 * 2.0 ** -24 + 2e-8


def _step(xs, causal, mode, scale):
    q, k, v, do = (x.clone().requires_grad_() for x in xs[:4])
    o = triton_attention(q, k, v, causal=causal, scale=scale, bwd_mode=mode)
    first = torch.autograd.grad(o, (q, k, v), do, create_graph=True)
    return [x.detach() for x in (o, *first, *torch.autograd.grad(first, (q, k, v, do), xs[4:]))]


def _same(name, a, b, tol):
    assert torch.equal(torch.isnan(a), torch.isnan(b)), name
    assert torch.equal(torch.isinf(a), torch.isinf(b)), name
    inf = torch.isinf(a)
    assert torch.equal(a[inf], b[inf]), name
    fin = torch.isfinite(a)
    x, y = a[fin].double(), b[fin].double()
    if x.numel():
        assert float((x - y).norm()) <= tol * max(float(y.norm()), 1.0), name


@pytest.mark.parametrize("which", range(7), ids=["q", "k", "v", "do", "rq", "rk", "rv"])
@pytest.mark.parametrize("value", [float("inf"), float("-inf"), float("nan")])
@pytest.mark.parametrize("d,causal,mode", [(64, True, "recompute"), (64, False, "save_p"), (40, False, "recompute")])
def test_non_finite_operands(which, value, d, causal, mode):
    t = 150
    g = torch.Generator().manual_seed(which)
    xs = [torch.randn((1, 2, t, d), generator=g).cuda() for _ in range(7)]
    xs[which][0, 1, 70, 3] = value
    wide = [torch.nn.functional.pad(x, (0, 128 - d)) for x in xs]
    got = _step(xs, causal, mode, 0.125)
    want = _step(wide, causal, mode, 0.125)
    for name, a, b in zip(("o", "dq", "dk", "dv", "gq", "gk", "gv", "gdo"), got, want):
        _same(name, a[:, 0], b[:, 0, :, :d], 5e-6)  # the untouched slice
        _same(name, a, b[..., :d], 5e-6)
