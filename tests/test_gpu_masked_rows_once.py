"""Rows without a gradient are cleared by one launch per chunk, also where a chunk's stages are enqueued by two calls: all of it
goes with the forward's then, and the backward's call leaves those rows alone."""
import pytest
import torch

pytestmark = pytest.mark.gpu

TOGETHER = 8        # clgrpo_head_step_args.stages


def _step(dev, T, H, V, live, dtype=torch.bfloat16):
    from chatlearn_amd import ops
    g = torch.Generator(device=dev).manual_seed(T)
    hidden = torch.randn(T, H, generator=g, device=dev).to(dtype)
    weight = (torch.randn(V, H, generator=g, device=dev) * 0.1).to(dtype)
    order = torch.randperm(T, generator=g, device=dev).to(torch.int32)
    mask = torch.zeros(T, dtype=torch.int32, device=dev)
    mask[order[:live].long()] = 1
    f = dict(dtype=torch.float32, device=dev)
    out = {k: torch.full((T,), float("nan"), **f) for k in ("logprob", "entropy", "lse", "g_logprob", "loss")}
    out["dhidden"] = torch.full((T, H), float("nan"), dtype=dtype, device=dev)
    out["dweight"] = torch.full((V, H), float("nan"), **f)
    z = ops.saved_logits_buffer(max(live, 1), V, dtype, dev)
    ws = torch.empty(ops.head_step_workspace_bytes(T, live, H, V, 1, dtype, True, False), dtype=torch.uint8, device=dev)
    scratch = torch.zeros(24, dtype=torch.float64, device=dev)
    step = ops.HeadStep(hidden, weight, torch.randint(0, V, (T,), generator=g, device=dev), torch.full((T,), -6.0, **f), None,
                        torch.ones(1, **f), torch.tensor([0, T], dtype=torch.int32, device=dev), mask, order, mode=0, temperature=1.0,
                        diff_clip_ratio=10, pos_clip_ratio=0.2, neg_clip_ratio=0.2, final_clip_ratio=3, kl_coef=0.0,
                        entropy_coef=0.0, grad_scale=1.0, kl=None, sums=scratch[14:22], flags=scratch[22:], result=scratch[:14],
                        workspace=ws, saved_logits=z, weight_t=None, **out)
    chunk = dict(lo=0, n=T, n_live=live, ordered=True, chunk=0, accumulate=False, weight_t_ready=False)
    return step, chunk, out, mask.bool()


@pytest.mark.parametrize("live_only", [False, True])
@pytest.mark.parametrize("T,live", [(300, 299), (300, 1), (65, 40)])
def test_two_calls_clear_once_and_give_what_one_call_gives(dev, T, live, live_only):
    results = []
    for calls in ((7,), (1, 2, 4), (3 | TOGETHER, 4 | TOGETHER)):
        step, chunk, out, mask = _step(dev, T, 128, 700, live)
        for stages in calls:
            step.enqueue(stages, forward_live_only=live_only, **chunk)
            if stages == 3 | TOGETHER:
                assert (out["dhidden"][~mask] == 0).all() and out["dhidden"][mask].isnan().all()
                out["dhidden"][~mask] = 7.0
            if stages == 4 | TOGETHER:
                assert (out["dhidden"][~mask] == 7.0).all()
                out["dhidden"][~mask] = 0.0
        results.append(out)
    for other in results[1:]:
        for k, v in results[0].items():
            assert torch.equal(v, other[k]), k


def test_no_row_with_a_gradient(dev):
    step, chunk, out, _ = _step(dev, 90, 128, 700, 0)
    step.enqueue(3 | TOGETHER, forward_live_only=False, **chunk)
    assert (out["dhidden"] == 0).all()
    step.enqueue(4 | TOGETHER, forward_live_only=False, **chunk)
    assert (out["dhidden"] == 0).all() and (out["dweight"] == 0).all() and out["logprob"].isfinite().all()
