"""fp32 at head dims up to 64, whose products are formed from bf16 parts: one
term keeps fp32's relative precision."""
import pytest
import torch

from testtimeideas_amd import _lib

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
