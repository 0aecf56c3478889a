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
        assert total.capacity == 704 and total.dzt.shape == (512, 704) and total.hidt.shape == (256, 704)
