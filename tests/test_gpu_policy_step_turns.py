"""train_step processes its micro-batches one by one where nothing in them can be refused later: the same bits as with all of them
processed in front, and what is refused is refused before the backbone is called."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _samples(n, seed, V):
    g = torch.Generator().manual_seed(seed)
    out = []
    for i in range(n):
        p, r = int(torch.randint(0, 9, (1,), generator=g)), int(torch.randint(1, 60, (1,), generator=g))
        T = p + r
        out.append({"all_tokens": torch.randint(0, V, (T,), generator=g), "prompt_token_length": p, "response_token_length": r,
                    "old_logprobs": torch.randn(T, generator=g) - 6, "ref_logprobs": torch.randn(T, generator=g) - 6,
                    "advantages": float(torch.randn(1, generator=g))})
    return out


def _step(dev, packing, cls=None, calls=None, V=1031, H=128, **kw):
    from chatlearn_amd.algorithm.grpo_utils.policy_step import PolicyStep
    g = torch.Generator(device=dev).manual_seed(5)
    table = torch.randn(V, H, generator=g, device=dev).bfloat16()
    weight = (torch.randn(V, H, generator=g, device=dev) * H ** -0.5).bfloat16().requires_grad_()
    calls = [] if calls is None else calls

    def backbone(ids, position_ids):
        calls.append(torch.nn.functional.embedding(ids.to(dev), table).requires_grad_())
        return calls[-1]

    return (cls or PolicyStep)(backbone, weight, packing=packing, max_token_in_seq=128, train_micro_batch_size=2, **kw), weight, calls


@pytest.mark.parametrize("packing", [False, True])
@pytest.mark.parametrize("n", [1, 7])
@pytest.mark.parametrize("own_mask", [False, True])
def test_the_same_bits_as_all_in_front(dev, packing, n, own_mask):
    from chatlearn_amd.algorithm.grpo_utils.policy_step import PolicyStep
    if packing and own_mask:
        pytest.skip("a packed sample's mask follows from its lengths")

    class AllInFront(PolicyStep):
        def preprocess_data_list(self, data_list, training):
            return super().preprocess_data_list(data_list=data_list, training=training)

    results = []
    for cls in (None, AllInFront):
        step, weight, hiddens = _step(dev, packing, cls)
        data = _samples(n, 3, 1031)
        if own_mask:
            for d in data:
                d["loss_mask"] = (torch.arange(d["all_tokens"].numel()) % 3 > 0).int()
        stats = step.train_step(data)
        results.append((stats, weight.grad, [h.grad for h in hiddens]))
        if cls is None:
            mbs = step._split(data, True)
            ahead = step._masks_ahead(mbs)
            assert (ahead is None) == own_mask
            if ahead is not None:
                want = [step._process(mb, True)["loss_mask_host"] for mb in mbs]
                assert all(torch.equal(a, b) for a, b in zip(ahead, want))
    (s0, w0, h0), (s1, w1, h1) = results
    assert s0 == s1 and torch.equal(w0, w1) and len(h0) == len(h1) and all(torch.equal(a, b) for a, b in zip(h0, h1))


def test_a_length_beyond_the_sample_is_refused_first(dev):
    step, weight, hiddens = _step(dev, True)
    data = _samples(7, 3, 1031)
    step.train_step([dict(d) for d in data])
    assert hiddens
    hiddens.clear()
    weight.grad = None
    for d in data:
        d["response_token_length"] += 200 if d is data[-1] else 0
    with pytest.raises(ValueError):
        step.train_step(data)
    assert not hiddens and weight.grad is None


@pytest.mark.parametrize("change", [lambda d: d.pop("advantages"), lambda d: d.update(extra=torch.ones(3)),
                                    lambda d: d.update(old_logprobs=d["old_logprobs"][:-1]),
                                    lambda d: d.update(ref_logprobs=d["ref_logprobs"].tolist())])
def test_samples_that_differ_are_processed_in_front(dev, change):
    step, _, _ = _step(dev, False)
    data = _samples(5, 3, 1031)
    assert step._masks_ahead(step._split(data, True)) is not None
    change(data[-1])
    assert step._masks_ahead(step._split(data, True)) is None
