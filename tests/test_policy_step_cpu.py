"""Host side of PolicyStep, without a device."""
import pytest
import torch


def _step(device="cpu", **kw):
    from chatlearn_amd.algorithm.grpo_utils.policy_step import PolicyStep
    return PolicyStep(None, torch.empty(8, 4, device=device), **kw)


def test_tensors_of_another_device_are_moved():
    """Device tensors without a device: what one GPU left in a record must not reach kernels on another as it is."""
    from torch._subclasses import FakeTensorMode
    with FakeTensorMode():
        step = _step("cuda:0")
        here, there = torch.empty(3, device="cuda:0"), torch.empty(3, device="cuda:1")
        assert step._put(here) is here
        moved = step._to_device({"old_logprobs": there, "loss_mask_host": torch.empty(3), "n": 2})
        assert moved["old_logprobs"].device == torch.device("cuda:0")
        assert moved["loss_mask_host"].device == torch.device("cpu") and moved["n"] == 2


@pytest.mark.parametrize("packing", [False, True])
def test_host_mask_is_the_rolled_response_mask(packing):
    """All prompt and response lengths up to the row's end, empty ones among them, against a roll of the mask itself."""
    width = 5
    pairs = [(p, r) for p in range(width + 1) for r in range(width + 1 - p)]
    mask = torch.zeros(len(pairs), width, dtype=torch.int32)
    for row, (p, r) in zip(mask, pairs):
        row[p:p + r] = 1
    want = torch.roll(mask, -1, 1)
    want[:, -1] = 0
    want = torch.cat([row[:p + r] for row, (p, r) in zip(want, pairs)]) if packing else want.reshape(-1)
    plen, rlen = zip(*pairs)
    for given in (None, mask):
        assert torch.equal(_step(packing=packing)._shifted_mask_host(given, plen, rlen, width), want)


@pytest.mark.parametrize("packing", [False, True])
@pytest.mark.parametrize("extra", [-2, 0, 3])
def test_host_mask_of_a_record_has_the_record_s_width(packing, extra):
    """One sample whose tokens are padded wider than its own loss mask, or less wide: the device mask keeps the record's width."""
    given = torch.tensor([[0, 0, 1, 1, 0, 1]], dtype=torch.int32)
    want = torch.tensor([0, 1, 1, 0, 1, 0], dtype=torch.int32)[:5 if packing else None]
    assert torch.equal(_step(packing=packing)._shifted_mask_host(given, [2], [3], given.shape[1] + extra), want)
