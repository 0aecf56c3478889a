"""Host side of PolicyStep, without a device."""
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
