"""Rows that carry a gradient picked by an order, at the sizes where the compact problem's tiles are ragged: none, one, a
tile less one, a tile, a tile and one, all but one and all of the rows unmasked - against the same step with every row
in the backward (masked rows have a zero upstream gradient there), in one chunk and in chunks of 256 kept rows."""
import pytest
import torch

from tests.util import assert_close_rel

pytestmark = pytest.mark.gpu

T, H, V = 613, 192, 1500


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("keep", ["auto", 256])
@pytest.mark.parametrize("n_live", [0, 1, 255, 256, 257, T - 1, T])
def test_step_with_an_order_equals_the_step_without(dev, n_live, keep, dtype):
    from chatlearn_amd.fused import grpo_head_step
    g = torch.Generator().manual_seed(n_live)
    mask = torch.zeros(T, dtype=torch.int32)
    mask[torch.randperm(T, generator=g)[:n_live]] = 1
    hidden, weight = torch.randn(T, H, generator=g).to(dtype).to(dev), (torch.randn(V, H, generator=g) * 0.07).to(dtype).to(dev)
    labels = torch.randint(0, V, (T,), generator=g).to(dev)
    old = (torch.randn(T, generator=g) * 0.1 - 7.5).to(dev)
    cu = torch.tensor([0, 100, 300, T], dtype=torch.int32)
    args = (hidden, weight, labels, old, old - 0.05, torch.randn(3, generator=g).to(dev), cu.to(dev), mask.to(dev))
    kw = dict(n_tokens_total=float(max(n_live, 1)), kl_coef=1e-2, entropy_coef=1e-2, temperature=0.9, keep_logits_chunk=keep,
              cu_seqlens_host=cu.tolist())
    base = torch.randn(V, H, generator=g).to(dev)
    full = grpo_head_step(*args, skip_masked_rows=False, dweight=base.clone(), accumulate_dweight=True, **kw)
    # summation orders differ (K ranges, chunks): fp32 1e-5; bf16 dhidden is rounded once more (2^-8 between neighbours)
    tol = 1e-5 if dtype == torch.float32 else 2 ** -8
    for lean in (False, True):
        got = grpo_head_step(*args, loss_mask_host=mask, skip_masked_forward=lean, dweight=base.clone(),
                             accumulate_dweight=True, **kw)
        live = mask.bool().to(dev)
        assert got["rows_projected_bwd"] == n_live
        assert (got["dhidden"][~live] == 0).all()
        for k in ("logprob", "entropy", "lse"):
            if n_live:
                assert_close_rel(got[k][live], full[k][live], 1e-5, k)
            if lean and n_live:
                assert (got[k][~live] == 0).all()
            else:
                assert_close_rel(got[k], full[k], 1e-5, k)
        assert_close_rel(got["dhidden"], full["dhidden"], tol, "dhidden")
        assert_close_rel(got["dweight"], full["dweight"], 1e-5 if dtype == torch.float32 else 1e-3, "dweight")
        assert float(got["total_loss"]) == pytest.approx(float(full["total_loss"]), rel=1e-5, abs=1e-7)


@pytest.mark.parametrize("host", [False, True])
@pytest.mark.parametrize("mask_dtype", [torch.bool, torch.int64, torch.bfloat16, torch.float32])
def test_mask_of_any_type(dev, mask_dtype, host):
    from chatlearn_amd.fused import grpo_head_step
    g = torch.Generator().manual_seed(1)
    mask = (torch.rand(T, generator=g) < 0.4).int()
    hidden, weight = torch.randn(T, H, generator=g).to(dev), (torch.randn(V, H, generator=g) * 0.07).to(dev)
    old = (torch.randn(T, generator=g) * 0.1 - 7.5).to(dev)
    cu = torch.tensor([0, 100, 300, T], dtype=torch.int32)
    out = []
    for m in (mask, mask.to(mask_dtype)):
        out.append(grpo_head_step(hidden, weight, torch.zeros(T, dtype=torch.int64, device=dev), old, old, torch.ones(3, device=dev),
                                  cu.to(dev), m.to(dev), n_tokens_total=float(mask.sum()), keep_logits_chunk=256,
                                  cu_seqlens_host=cu.tolist(), loss_mask_host=m if host else None))
    assert out[0]["rows_projected_bwd"] == out[1]["rows_projected_bwd"] == int(mask.sum())
    for k in ("total_loss", "dhidden", "dweight"):
        assert torch.equal(out[0][k], out[1][k])
