"""dW over several micro-batches in one contraction, and dW rounded to bf16 as it is written: against a contraction per
micro-batch added up in fp32, where the kept operands fill their place exactly, by less than a slab, overflow into a second
contraction, or one micro-batch is larger than the place; vocabulary and hidden sizes off the tiles."""
import pytest
import torch

from tests.util import assert_close_rel

pytestmark = pytest.mark.gpu

LIVE = [1, 200, 64, 0, 333]           # rows with a gradient of each micro-batch


def _batches(dev, dtype, H, V):
    g = torch.Generator().manual_seed(H + V)
    weight = (torch.randn(V, H, generator=g) * 0.07).to(dtype).to(dev)
    out = []
    for n_live in LIVE:
        T = n_live + 37
        mask = torch.zeros(T, dtype=torch.int32)
        mask[torch.randperm(T, generator=g)[:n_live]] = 1
        old = (torch.randn(T, generator=g) * 0.1 - 7.0).to(dev)
        cu = torch.tensor([0, T // 3, T], dtype=torch.int32)
        out.append((mask, cu.tolist(), (torch.randn(T, H, generator=g).to(dtype).to(dev), weight, torch.randint(0, V, (T,), generator=g).to(dev),
                    old, old - 0.05, torch.randn(2, generator=g).to(dev), cu.to(dev), mask.to(dev))))
    return weight, out, torch.randn(V, H, generator=g).to(dev)


@pytest.mark.parametrize("dtype,H,V", [(torch.bfloat16, 192, 1500), (torch.bfloat16, 64, 257), (torch.float32, 96, 700)])
@pytest.mark.parametrize("limit", [64, 256, 10 ** 6])
@pytest.mark.parametrize("with_buffer", [False, True])
def test_sum_over_micro_batches(dev, dtype, H, V, limit, with_buffer):
    from chatlearn_amd import ops
    from chatlearn_amd.fused import grpo_head_step
    weight, batches, base = _batches(dev, dtype, H, V)
    kw = dict(n_tokens_total=float(sum(LIVE)), kl_coef=1e-2, entropy_coef=1e-2)
    want = base.clone() if with_buffer else torch.zeros_like(base)
    buffer = base.clone() if with_buffer else None
    total = ops.DweightSum(weight, sum(n + 64 for n in LIVE), limit, buffer)
    for mask, cu, args in batches:
        a = grpo_head_step(*args, loss_mask_host=mask, cu_seqlens_host=cu, dweight=want, accumulate_dweight=True, **kw)
        b = grpo_head_step(*args, loss_mask_host=mask, cu_seqlens_host=cu, _dweight_sum=total, **kw)
        assert b["dweight"] is None and torch.equal(a["dhidden"], b["dhidden"])
        assert b["scratch_bytes"] >= total.bytes > 0
    got = total.finish(dtype)
    assert got.dtype == (torch.float32 if with_buffer else dtype) and (buffer is None or got is buffer)
    # the order of fp32 sums differs; a bf16 result is rounded once (2^-9 of each entry)
    assert_close_rel(got.float(), want, 1e-5 if got.dtype == torch.float32 else 2 ** -8, "dweight")


@pytest.mark.parametrize("T,H,V", [(1, 64, 50), (300, 192, 1500), (513, 2048, 33000)])
@pytest.mark.parametrize("keep", ["auto", None])
def test_bf16_dweight_is_the_rounded_fp32_one(dev, T, H, V, keep):
    from chatlearn_amd import ops
    g = torch.Generator().manual_seed(T)
    hidden, weight = torch.randn(T, H, generator=g).bfloat16().to(dev), (torch.randn(V, H, generator=g) * 0.05).bfloat16().to(dev)
    labels = torch.randint(0, V, (T,), generator=g).to(dev)
    g_lp = torch.randn(T, generator=g).to(dev)
    out = []
    for dt in (torch.float32, torch.bfloat16):
        z = ops.saved_logits_buffer(T, V, hidden.dtype, dev) if keep else None
        _, _, _, lse = ops.lmhead_forward(hidden, weight, labels, saved_logits=z)
        dh, dw = ops.lmhead_backward(hidden, weight, labels, lse, None, g_lp, saved_logits=z, dweight_dtype=dt)
        assert dw.dtype == dt
        out.append((dh, dw.bfloat16()))
    assert torch.equal(out[0][0], out[1][0]) and torch.equal(out[0][1], out[1][1])
