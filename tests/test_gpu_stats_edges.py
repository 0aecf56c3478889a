"""Softmax statistics and gradients of rows that start and end off a 16-byte boundary: vocabularies around the size of
one and of several passes of a block, rows cut out of wider ones (the packed result is then shifted against them),
and bases that are not aligned themselves - against float64."""
import pytest
import torch

from oracle import softmax_stats as osm
from tests.util import assert_close_rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("V,ld,offset", [(1, 1, 0), (7, 7, 3), (8, 9, 1), (255, 255, 0), (1031, 1040, 5), (4099, 4099, 2),
                                         (8192, 8193, 0), (33003, 33003, 1)])
def test_misaligned_rows(dev, dtype, V, ld, offset):
    from chatlearn_amd import ops
    R = 5
    g = torch.Generator().manual_seed(V + ld)
    flat = (torch.randn(offset + R * ld, generator=g) * 2).to(dtype).to(dev)
    z = torch.as_strided(flat, (R, V), (ld, 1), offset)
    y = torch.randint(0, V, (R,), generator=g)
    y[0], y[-1] = 0, V - 1
    glp, gen = torch.randn(R, generator=g), torch.randn(R, generator=g)
    lp, ent, lse = ops.softmax_stats(z, y.to(dev))
    zd = z.detach().cpu().double().requires_grad_(True)
    rlp, rent = osm.logprobs_from_logits(zd, y), osm.entropy_from_logits(zd)
    assert (lp.cpu().double() - rlp.detach()).abs().max() < 1e-5 * (1 + rlp.detach().abs().max())
    assert (ent.cpu().double() - rent.detach()).abs().max() < 1e-5 * (1 + rent.detach().abs().max())
    (rlp * glp.double() + rent * gen.double()).sum().backward()
    # the result is rounded once to the logits' dtype (bf16: 2^-9 of each entry); the arithmetic before that is fp32
    tol = 1e-5 if dtype == torch.float32 else 2 ** -8
    for kept in ({"lse": lse, "entropy": ent}, {}):
        d = ops.softmax_stats_backward(z, y.to(dev), glp.to(dev), gen.to(dev), **kept)
        if V > 1:
            assert_close_rel(d, zd.grad, tol, "dlogits")
        else:
            assert d.abs().max() < 1e-5
