"""dhidden's row tiles (128, 192 or 256 rows): the launch follows its plan also where that plan needs no partial sums."""
import pytest
import torch

# (rows, H, V) -> (row tiles of 256 of a first launch, K ranges, rows per tile of the launch behind it)
PLANS = [((1537, 7168, 129280), (0, 1, 192)), ((1728, 7168, 300), (0, 1, 192)), ((3400, 3584, 32003), (0, 1, 192)),
         ((128, 4096, 151936), (0, 16, 128)), ((320, 2048, 151936), (0, 16, 192)), ((12126, 4096, 151936), (0, 1, 256)),
         ((12700, 4096, 151936), (48, 8, 256))]


@pytest.mark.parametrize("size,plan", PLANS)
def test_reported_tiles(lib, size, plan):
    from chatlearn_amd import ops
    assert ops.dhidden_tile_plan(*size, torch.bfloat16)[:3] == plan
    assert ops.dhidden_launch_plan(*size, torch.bfloat16) == plan[:2]
    assert ops.dhidden_tile_plan(*size, torch.float32)[2] == 256           # fp32 has no narrower tiles


def test_a_plan_without_partial_sums_is_launched_as_planned(lib):
    """Whatever the scratch memory holds for partial sums: nothing where neither contraction wants any."""
    from chatlearn_amd import _lib, ops
    out = (_lib.i32 * 4)()
    for rows, H in ((1537, 7168), (1728, 7168), (3329, 3584)):
        assert lib.clgrpo_lmhead_bwd_dhidden_tile_plan(rows, H, 129280, _lib.BF16, 256, 0, out) == 0
        assert tuple(out)[:3] == (0, 1, 192)
        # with memory for none, a plan that would like some still takes the best tile without a K split
        assert lib.clgrpo_lmhead_bwd_dhidden_tile_plan(128, H, 129280, _lib.BF16, 256, 0, out) == 0
        assert tuple(out)[:3] == (0, 1, 128)


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [1537, 1600, 1727, 1728])
@pytest.mark.parametrize("ordered", [False, True])
def test_tiles_of_192_rows_without_a_k_split(dev, rows, ordered):
    """28 column tiles of H = 7168 by 9 row tiles, the last one ragged.  Bound per entry: a kept logit is off by its half rounding
    (2^-11) and its fp32 sum, which moves its probability by that much of itself, twice with the shift of lse; d(logits) and the
    result are rounded to bf16 (2^-8 each); 300 terms are summed in fp32."""
    from chatlearn_amd import ops
    from chatlearn_amd.fused import grpo_head_step
    H, V = 7168, 300
    T = rows + (200 if ordered else 0)
    g = torch.Generator(device=dev).manual_seed(rows)
    hidden = torch.randn(T, H, generator=g, device=dev).bfloat16()
    weight = (torch.randn(V, H, generator=g, device=dev) * 0.02).bfloat16()
    labels = torch.randint(0, V, (T,), generator=g, device=dev)
    mask = torch.zeros(T, dtype=torch.int32, device=dev)
    mask[torch.randperm(T, generator=g, device=dev)[:rows]] = 1
    assert ops.dhidden_tile_plan(rows, H, V, torch.bfloat16)[:3] == (0, 1, 192)
    out = grpo_head_step(hidden, weight, labels, torch.full((T,), -6.0, device=dev), None, torch.ones(1, device=dev),
                         torch.tensor([0, T], dtype=torch.int32, device=dev), mask, n_tokens_total=1.0, loss_mask_host=mask.cpu())
    h64, w64, g64 = hidden.double(), weight.double(), out["g_logprob"].double()[:, None]
    z64 = h64 @ w64.t()
    p = torch.softmax(z64, -1)
    dz = g64 * (torch.nn.functional.one_hot(labels, V) - p)
    zerr = (h64.abs() @ w64.abs().t()) * H * 2.0 ** -24 + z64.abs() * 2.0 ** -11
    dzerr = g64.abs() * p * (2 * zerr.max(-1, keepdim=True).values + 2.0 ** -20)
    want = dz @ w64
    bound = 1.01 * dzerr @ w64.abs() + dz.abs() @ w64.abs() * (2.0 ** -8 + V * 2.0 ** -24) + want.abs() * 2.0 ** -8 + 1e-30
    live = mask.bool()
    assert (out["dhidden"][~live] == 0).all()
    err = (out["dhidden"].double() - want).abs()
    assert (err <= bound)[live].all(), float((err / bound)[live].max())
    # and the products of the same rows in tiles of another width, bit for bit: no K split either way
    some = torch.nonzero(live).flatten()[:700]
    assert ops.dhidden_tile_plan(700, H, V, torch.bfloat16)[1:3] in ((1, 128), (1, 256))
    z = ops.saved_logits_buffer(700, V, torch.bfloat16, dev)
    y, g_lp = labels[some], out["g_logprob"][some]
    lse = ops.lmhead_forward(hidden[some], weight, y, saved_logits=z)[3]
    assert torch.equal(lse, out["lse"][some])
    assert torch.equal(ops.lmhead_backward(hidden[some], weight, y, lse, None, g_lp, need_dweight=False, saved_logits=z)[0],
                       out["dhidden"][some])
