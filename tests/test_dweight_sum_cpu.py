"""Host side of ops.DweightSum, without a device."""
import pytest
import torch


def _sum(total, limit, V=500, H=128):
    from chatlearn_amd import ops
    return ops.DweightSum(torch.empty(V, H, dtype=torch.bfloat16, device="cuda:0"), total, limit)


def test_a_first_chunk_beyond_the_limit_contracts_nothing():
    """One chunk with more rows than the sum was to hold gets a larger place; there is no [V, H] tensor to clear before it."""
    from torch._subclasses import FakeTensorMode
    with FakeTensorMode():
        total = _sum(1000, 256)
        total._contract = lambda dtype: pytest.fail("contracted")
        total.place(700)
        assert total.bytes == 2 * 704 * (512 + 256)
        assert total.capacity == 704 and total.dzt.shape == (512, 704) and total.hidt.shape == (256, 704)


@pytest.mark.parametrize("keep,rows,want", [(640, "auto", 640), (640, 128, 128), (640, 10 ** 6, 1024 + 2 * 64), (640, None, None),
                                            (640, 0, None), (None, "auto", None), (None, 128, None)])
def test_rows_that_wait_for_dweight_have_a_bound_of_their_own(keep, rows, want):
    """PolicyStep: as many as keep their logits by default, never more than the mini-batch has, none without kept logits."""
    from chatlearn_amd.algorithm.grpo_utils.policy_step import PolicyStep
    step = PolicyStep(None, torch.empty(500, 64), keep_logits_chunk=keep, dweight_sum_rows=rows)
    total = step._dweight_sum([{"loss_mask_host": torch.ones(512, dtype=torch.int32)}] * 2)
    assert (total if total is None else total.capacity) == want
