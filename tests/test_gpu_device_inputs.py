"""Advantages and lengths, lists in the reference, given as tensors that already are on the device: the same results."""
import copy

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _loss_inputs(dev, B=3, S=17):
    g = torch.Generator().manual_seed(2)
    lp = (torch.randn(B, S, generator=g) * 0.3 - 5).to(dev)
    return lp, lp + 0.1, torch.randn(B, generator=g)


def test_loss_gallery(dev):
    from chatlearn_amd.algorithm.grpo_utils.loss_gallery import calculate_grpo_loss, calculate_gspo_loss
    lp, old, adv = _loss_inputs(dev)
    mask = torch.ones(lp.shape, dtype=torch.int32, device=dev)
    assert torch.equal(calculate_grpo_loss(lp, old, adv.to(dev)), calculate_grpo_loss(lp, old, adv.tolist()))
    assert torch.equal(calculate_gspo_loss(lp, old, adv.to(dev), loss_mask=mask)[0],
                       calculate_gspo_loss(lp, old, adv.tolist(), loss_mask=mask)[0])


@pytest.mark.parametrize("put", [lambda x, dev: x, lambda x, dev: x.to(dev)])
def test_megatron_batch_and_loss_dict(dev, put):
    from types import SimpleNamespace
    from chatlearn_amd.algorithm.grpo_utils.megatron_utils import train_helper
    p, r, S = [3, 5], [6, 9], 14
    g = torch.Generator().manual_seed(3)
    batch = {"all_tokens": torch.randint(0, 50, (2, S), generator=g), "old_logprobs": torch.randn(2, S, generator=g) * 0.1 - 4,
             "ref_logprobs": torch.randn(2, S, generator=g) * 0.1 - 4}
    args = SimpleNamespace(packing=True, use_group_sequence_policy=False, diff_clip_ratio=10, pos_clip_ratio=0.2,
                           neg_clip_ratio=0.2, final_clip_ratio=3)
    adv = torch.tensor([0.5, -1.5])
    logits = (torch.randn(24, 1, 50, generator=g) * 2).to(dev)
    out = []
    for lists in (True, False):
        b = dict(batch, prompt_token_length=p if lists else put(torch.tensor(p), dev),
                 response_token_length=r if lists else put(torch.tensor(r), dev), advantages=adv.tolist() if lists else put(adv, dev))
        inp = train_helper.get_batch_packed(b, True, eod=0)
        z = logits[:inp["labels"].numel()]
        losses = train_helper._compute_all_losses(args, None, z, inp["labels"], inp)
        out.append((inp["all_tokens"], inp["all_token_loss_mask"], losses["pg_loss"], losses["kl_loss"]))
    for a, b in zip(*out):
        assert torch.equal(a, b)


@pytest.mark.parametrize("packing", [False, True])
def test_policy_step(dev, packing):
    from chatlearn_amd.algorithm.grpo_utils.policy_step import PolicyStep
    V, H = 300, 64
    g = torch.Generator().manual_seed(4)
    table = torch.randn(V, H, generator=g).to(dev)
    data = []
    for i in range(5):
        p, r = 3 + i, 9 + 2 * i
        data.append({"all_tokens": torch.randint(0, V, (p + r,), generator=g), "prompt_token_length": p, "response_token_length": r,
                     "old_logprobs": torch.full((p + r,), -5.7), "ref_logprobs": torch.full((p + r,), -5.7),
                     "advantages": np.float32(i - 2)})
    moved = copy.deepcopy(data)
    for s in moved:
        for key in ("prompt_token_length", "response_token_length", "advantages"):
            s[key] = torch.tensor([s[key]], device=dev)
    out = []
    for samples in (data, moved):
        weight = (torch.randn(V, H, generator=torch.Generator().manual_seed(6)) * 0.05).to(dev).requires_grad_(True)
        step = PolicyStep(lambda ids, pos: table[ids], weight, packing=packing, max_token_in_seq=64, train_micro_batch_size=2)
        out.append((step.train_step(copy.deepcopy(samples)), weight.grad))
    assert out[0][0] == out[1][0] and torch.equal(out[0][1], out[1][1])
