"""Logits around and beyond the size (160 MB) from which the statistics and gradients go around the last-level cache and the gradients
take the rows from the last one on: the same bits as the rows in calls of some ten megabytes each."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("R,V,ld,offset,dtype", [
    (552, 151936, 151936, 0, torch.bfloat16),      # 159.97 MB
    (553, 151936, 151936, 0, torch.bfloat16),      # 160.26 MB: the first that does
    (700, 151669, 151669, 3, torch.bfloat16),      # rows of every alignment, gradients on both sides of 128 MB
    (1400, 32003, 32003, 1, torch.float32),
    (1400, 32003, 32007, 0, torch.float32),        # rows cut out of wider ones
])
@pytest.mark.parametrize("with_entropy", [False, True])
def test_rows_are_those_of_small_calls(dev, R, V, ld, offset, dtype, with_entropy):
    from chatlearn_amd import ops
    g = torch.Generator(device=dev).manual_seed(R + V)
    flat = torch.randn(offset + R * ld, generator=g, device=dev, dtype=torch.float32).to(dtype)
    z = torch.as_strided(flat, (R, V), (ld, 1), offset)
    y = torch.randint(0, V, (R,), generator=g, device=dev)
    glp, gen = torch.randn(R, generator=g, device=dev), torch.randn(R, generator=g, device=dev)
    gen = gen if with_entropy else None

    def both(a, b):
        lp, ent, lse = ops.softmax_stats(z[a:b], y[a:b])
        kept = {"lse": lse, "entropy": ent}
        ge = None if gen is None else gen[a:b].contiguous()
        grads = [ops.softmax_stats_backward(z[a:b], y[a:b], glp[a:b].contiguous(), ge, **k) for k in (kept, {})]
        return [lp, ent, lse] + grads

    whole = both(0, R)
    for a in range(0, R, 100):
        b = min(a + 100, R)
        for got, want in zip(whole, both(a, b)):
            assert torch.equal(got[a:b], want), f"rows {a} to {b}"
