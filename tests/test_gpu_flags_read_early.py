"""The loss flags travel while the backward runs: they are those of all chunks, and nothing else depends on when they are read."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _inputs(dev, T=900, H=128, V=3000):
    g = torch.Generator().manual_seed(1)
    hidden, weight = torch.randn(T, H, generator=g).bfloat16().to(dev), (torch.randn(V, H, generator=g) * 0.1).bfloat16().to(dev)
    labels = torch.randint(0, V, (T,), generator=g).to(dev)
    old, ref = (torch.randn(2, T, generator=g) * 0.1 - 8).to(dev)
    mask = (torch.rand(T, generator=g) < 0.8).int()
    cu = torch.tensor([0, 300, T], dtype=torch.int32)
    args = [hidden, weight, labels, old, ref, torch.tensor([1.0, -0.5], device=dev), cu.to(dev), mask.to(dev)]
    return args, dict(n_tokens_total=float(mask.sum()), kl_coef=1e-3, cu_seqlens_host=cu.tolist(), loss_mask_host=mask)


WAYS = [dict(), dict(keep_logits_chunk=256), dict(keep_logits_chunk=None), dict(need_dhidden=False, _need_dweight=False)]


@pytest.mark.parametrize("way", WAYS)
@pytest.mark.parametrize("at", [5, 895])
def test_a_bad_token_of_any_chunk_is_reported(dev, way, at):
    from chatlearn_amd.fused import grpo_head_step
    args, kw = _inputs(dev)
    at = int(torch.nonzero(kw["loss_mask_host"])[(torch.nonzero(kw["loss_mask_host"]).flatten() - at).abs().argmin()])
    args[3] = args[3].clone()
    args[3][at] = float("nan")
    with pytest.raises(AssertionError, match="pg loss is nan"):
        grpo_head_step(*args, **kw, **way)


@pytest.mark.parametrize("way", WAYS)
def test_results_do_not_depend_on_the_check(dev, way):
    from chatlearn_amd.fused import grpo_head_step
    args, kw = _inputs(dev)
    a, b = (grpo_head_step(*args, **kw, **way, check_flags=check) for check in (True, False))
    for k in ("logprob", "entropy", "dhidden", "dweight", "total_loss", "num_masked", "g_logprob"):
        assert (a[k] is None and b[k] is None) or torch.equal(a[k], b[k]), k


def test_a_stale_host_mask_is_still_refused(dev):
    from chatlearn_amd.fused import grpo_head_step
    args, kw = _inputs(dev)
    kw["loss_mask_host"] = kw["loss_mask_host"].clone()
    kw["loss_mask_host"][3] ^= 1
    with pytest.raises(ValueError, match="stale"):
        grpo_head_step(*args, **kw)
