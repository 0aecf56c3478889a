"""The GEMM tile and the forward's launch plan at the sizes where they can go wrong: K extents of one to five slabs
(fewer than three do not stream from tile to tile), ragged last tiles in every dimension, several tiles per
workgroup, and vocabulary splits from one to the most a single token block gets - against float64 on the device."""
import pytest
import torch

from tests.util import assert_close_rel, assert_rows_rel_l2

pytestmark = pytest.mark.gpu

# the contract's bounds: bf16 operands are exact here, results pass through at most two bf16 roundings (2^-9 each)
RTOL = {torch.float32: 1e-5, torch.bfloat16: 1e-2}


def _check(dev, T, H, V, dtype, keep, seed):
    from chatlearn_amd import ops
    g = torch.Generator(device=dev).manual_seed(seed)
    h = torch.randn(T, H, generator=g, device=dev).to(dtype)
    w = (torch.randn(V, H, generator=g, device=dev) * H ** -0.5).to(dtype)
    y = torch.randint(0, V, (T,), generator=g, device=dev)
    y[0], y[-1] = 0, V - 1
    glp, gen = torch.randn(T, generator=g, device=dev), torch.randn(T, generator=g, device=dev) * 0.1
    zbuf = ops.saved_logits_buffer(T, V, dtype, dev) if keep else None
    lp, ent, mx, lse = ops.lmhead_forward(h, w, y, 0.9, saved_logits=zbuf)
    base = torch.randn(V, H, generator=g, device=dev) * 1e-3
    dh, dw = ops.lmhead_backward(h, w, y, lse, ent, glp, gen, 0.9, saved_logits=zbuf, dweight=base.clone(), accumulate_dweight=True)
    z = h.double() @ w.double().t() / 0.9
    rlse = torch.logsumexp(z, 1)
    p = torch.exp(z - rlse[:, None])
    rent = rlse - (p * z).sum(1)
    r = RTOL[dtype]
    assert_close_rel(lp, z.gather(1, y[:, None])[:, 0] - rlse, r, "logprob")
    assert_close_rel(ent, rent, r, "entropy")
    assert_close_rel(mx, z.max(1).values, r, "rowmax")
    dz = -p * (glp.double()[:, None] + gen.double()[:, None] * (z - rlse[:, None] + rent[:, None]))
    dz.scatter_add_(1, y[:, None], glp.double()[:, None])
    dz /= 0.9
    assert_close_rel(dh, dz @ w.double(), r, "dhidden")
    # Row by row, and rows that are nobody's label by themselves: their softmax part is down to 1e-5 of a label's.  The bound on
    # a row: dz rounded to bf16 (2^-9) and kept logits below 8 to half (2^-9, times 1 / 0.9, in the probability) are 4.2e-3
    # of every term, 1e-2 with room for sums that cancel; fp32 logits and their exponential err by some 1e-6.
    labelled = torch.zeros(V, dtype=torch.bool, device=dev)
    labelled[y] = True
    got, want = dw.double() - base.double(), dz.t() @ h.double()
    for name, rows in (("labels", labelled), ("others", ~labelled)):
        if rows.any():
            assert_rows_rel_l2(got[rows], want[rows], r, f"dweight, {name}")


@pytest.mark.parametrize("keep", [False, True])
@pytest.mark.parametrize("dtype,H", [(torch.bfloat16, h) for h in (64, 128, 192, 320)] + [(torch.float32, h) for h in (32, 64, 96, 160)])
def test_k_extents_and_ragged_tiles(dev, dtype, H, keep):
    _check(dev, 5003, H, 9001, dtype, keep, seed=H)


@pytest.mark.parametrize("T", [1, 33, 256, 257, 900])
@pytest.mark.parametrize("V", [255, 4097, 120001])
def test_vocabulary_splits(dev, T, V):
    _check(dev, T, 192, V, torch.bfloat16, True, seed=T + V)


@pytest.mark.parametrize("H,V", [(64, 4097), (192, 33000), (448, 9001), (576, 20064), (1088, 9001)])
@pytest.mark.parametrize("T", [1, 16, 127, 128, 129, 257, 384, 385])
def test_dhidden_of_few_rows(dev, T, H, V):
    """Up to 384 rows with kept logits read W itself (128 columns per wave, 512 per workgroup, 128 rows, K ranges of at least
    8 slabs); H beyond a whole number of either, a vocabulary that ends inside a slab, rows on both sides of a block and of the limit."""
    _check(dev, T, H, V, torch.bfloat16, True, seed=T + H)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("V", [4097, 9001, 9020])
@pytest.mark.parametrize("T", [100, 385])
def test_what_lies_behind_the_operands_does_not_matter(dev, T, V, dtype):
    """W and the hidden states cut from the front of larger arrays that are not finite behind them; vocabularies that end
    inside a group of 8 rows, inside a step of 32 and inside a slab."""
    from chatlearn_amd import ops
    H = 192
    g = torch.Generator(device=dev).manual_seed(V)
    h, w = torch.randn(T, H, generator=g, device=dev).to(dtype), (torch.randn(V, H, generator=g, device=dev) * H ** -0.5).to(dtype)
    y = torch.randint(0, V, (T,), generator=g, device=dev)
    glp = torch.randn(T, generator=g, device=dev)
    behind = torch.full((256, H), float("nan"), dtype=dtype, device=dev)
    cut = (torch.cat([h, behind])[:T], torch.cat([w, behind])[:V])
    for keep in (True, False):
        out = []
        for hidden, weight in ((h, w), cut):
            z = ops.saved_logits_buffer(T, V, dtype, dev) if keep else None
            lp, ent, _, lse = ops.lmhead_forward(hidden, weight, y, saved_logits=z)
            out.append((lp, ent) + ops.lmhead_backward(hidden, weight, y, lse, None, glp, saved_logits=z))
        for a, b in zip(*out):
            assert a.isfinite().all() and torch.equal(a, b)
