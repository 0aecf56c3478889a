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


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("V,offset", [(40, 0), (1031, 0), (1031, 3), (4099, 2), (33003, 1)])
@pytest.mark.parametrize("where", ["head", "tail", "most"])
def test_entries_masked_with_the_lowest_value(dev, dtype, V, offset, where):
    """Vocabulary entries masked out with the type's lowest value, where they are all that a thread sees at first (or at
    all): in front of the row's first 16-byte boundary, behind its last one, and in whole pieces."""
    from chatlearn_amd import ops
    R = 4
    g = torch.Generator().manual_seed(V + offset)
    flat = (torch.randn(offset + R * V, generator=g) * 2).to(dtype)
    rows = flat[offset:].view(R, V)
    {"head": rows[:, :16], "tail": rows[:, -11:], "most": rows[:, 5:]}[where].fill_(torch.finfo(dtype).min)
    z = flat.to(dev)[offset:].view(R, V)
    y = torch.full((R,), 3 if where != "head" else 20)
    glp, gen = torch.randn(R, generator=g), torch.rand(R, generator=g)
    lp, ent, lse = ops.softmax_stats(z, y.to(dev))
    zd = rows.double().requires_grad_(True)
    rlp, rent = osm.logprobs_from_logits(zd, y), osm.entropy_from_logits(zd)
    assert_close_rel(lp, rlp, 1e-5, "logprob")
    assert_close_rel(ent, rent, 1e-5, "entropy")
    (rlp * glp.double() + rent * gen.double()).sum().backward()
    for kept in ({"lse": lse, "entropy": ent}, {}):
        d = ops.softmax_stats_backward(z, y.to(dev), glp.to(dev), gen.to(dev), **kept)
        assert_close_rel(d, zd.grad, 1e-5 if dtype == torch.float32 else 2 ** -8, "dlogits")
