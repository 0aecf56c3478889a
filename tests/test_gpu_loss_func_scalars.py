"""loss_func's results as a training schedule uses them: the loss is divided in place, the report stays as it was."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("needs_grad", [True, False])
def test_loss_divided_in_place_keeps_its_gradient_and_leaves_the_report(dev, needs_grad):
    from chatlearn_amd.algorithm.grpo_utils.megatron_utils import train_helper as th
    g = torch.Generator().manual_seed(0)
    pg = torch.randn(3, 40, generator=g, dtype=torch.float64).to(dev).requires_grad_(needs_grad)
    ent = torch.randn(3, 40, generator=g).to(dev)
    mask = (torch.rand(3, 40, generator=g) < 0.6).int().to(dev)
    total, n, report = th.loss_func({"all_token_loss_mask": mask}, {"pg_loss": pg, "entropy_loss": ent})
    want = (pg.detach().float().double() * mask).sum().float()       # entries as fp32, summed in fp64, rounded to fp32 once
    assert torch.allclose(total.detach(), want, rtol=2.0 ** -22, atol=0)
    total /= n
    total /= 4
    assert torch.allclose(report["pg_loss"], want, rtol=2.0 ** -22, atol=0) and not report["pg_loss"].requires_grad
    report["pg_loss"] += 1.0
    assert torch.allclose(total.detach(), want / n / 4, rtol=2.0 ** -21, atol=0)
    assert int(n) == int(mask.sum()) and int(report["num_tokens"]) == int(n) and int(report["num_samples"]) == 1
    if needs_grad:
        total.backward()
        assert torch.allclose(pg.grad, mask.double() / int(n) / 4, rtol=2.0 ** -21, atol=0)
