"""Products of the backward with more tiles than compute units, one workgroup per tile: every tile is made once, whichever
XCD it is handed to, round by round (dhidden, dW of up to 128 or from 2048 rows on) or an eighth of the launch each."""
import pytest
import torch

pytestmark = pytest.mark.gpu


# dhidden of 43 x 16 tiles of 192 rows (fp32: 33 x 16 of 256); dW of 36 x 16, of 64 x 28 with ragged edges, of 43 x 6, and one tile
# more than a round; beside them dW of 37 x 28, which workgroups walk
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("T,H,V,plain", [(8200, 4096, 300, "dhidden"), (130, 4096, 9000, "dW"), (2050, 1536, 11000, "dW"), (70, 7104, 16383, "dW"),
                                         (64, 256, 65793, "dW"),
                                         (70, 7104, 9217, None)])
def test_products_against_64_bits(dev, dtype, T, H, V, plain):
    """bf16: d(logits) rounded to 2^-8, the result once more; fp32: sums of at most 66000 products, 2^-16 of their norm."""
    from chatlearn_amd import ops
    bulk, k_ranges, rows, _ = ops.dhidden_tile_plan(T, H, V, dtype)
    n_ht = -(-H // 256)
    assert (plain == "dhidden") == (bulk == 0 and k_ranges == 1 and 256 < -(-T // rows) * n_ht < 1024)
    assert (plain == "dW") == (ops.dweight_launch_plan(T, H, V, dtype) == (0, 0, 1) and -(-V // 256) * n_ht > 256)
    g = torch.Generator(device=dev).manual_seed(T + V)
    hidden = torch.randn(T, H, generator=g, device=dev).to(dtype)
    weight = (torch.randn(V, H, generator=g, device=dev) * 0.02).to(dtype)
    labels = torch.randint(0, V, (T,), generator=g, device=dev)
    g_lp = torch.randn(T, generator=g, device=dev)
    z = ops.saved_logits_buffer(T, V, dtype, dev)
    _, _, _, lse = ops.lmhead_forward(hidden, weight, labels, saved_logits=z)
    dh, dw = ops.lmhead_backward(hidden, weight, labels, lse, None, g_lp, saved_logits=z)
    h64, w64 = hidden.double(), weight.double()
    dz = -torch.softmax(h64 @ w64.t(), -1)
    dz.scatter_add_(1, labels[:, None], torch.ones(T, 1, dtype=torch.float64, device=dev))
    dz *= g_lp.double()[:, None]
    tol = 3 * 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -16
    for got, want in ((dh.double(), dz @ w64), (dw.double(), dz.t() @ h64)):
        assert (got - want).norm() <= tol * want.norm()
        blocks = [(got - want)[r:r + 256].norm() <= 2 * tol * want[r:r + 256].norm() + 1e-12 for r in range(0, len(want), 256)]
        assert all(bool(b) for b in blocks)
