"""dW added to what the buffer holds: the tile's old contents are requested before the tile before is stored, and rows and
columns past a tile's end take part in neither."""
import pytest
import torch

pytestmark = pytest.mark.gpu


# one workgroup per tile; walks over many vocabulary tiles with a ragged last row and column tile; walks and a K-split tail behind them;
# the last dW (H = 960) that is added to through the last-level cache and the first that goes around it
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("T,H,V", [(1, 64, 3), (130, 192, 257), (200, 960, 66049), (70, 1024, 65537), (640, 1088, 70001),
                                   (1300, 960, 66049), (500, 320, 40000), (70, 960, 30583), (70, 960, 30584)])
def test_added_equals_overwritten_plus_old(dev, dtype, T, H, V):
    """The same products are summed in the same order, from the old value instead of from 0: each of at most T additions rounds
    to 2^-24 of a partial sum, which |old| + sum over t of |g_t| max|h_t| bounds."""
    from chatlearn_amd import ops
    n_walk, bulk, k_ranges = ops.dweight_launch_plan(T, H, V, dtype)
    assert (n_walk > 0) == (V > 60000) and (bulk > 0 and k_ranges > 1) == (T == 1300)
    g = torch.Generator(device=dev).manual_seed(T + V)
    hidden = torch.randn(T, H, generator=g, device=dev).to(dtype)
    weight = (torch.randn(V, H, generator=g, device=dev) * 0.05).to(dtype)
    labels = torch.randint(0, V, (T,), generator=g, device=dev)
    g_lp = torch.randn(T, generator=g, device=dev)
    old = torch.randn(V + 2, H, generator=g, device=dev)
    buf = old.clone()
    _, _, _, lse = ops.lmhead_forward(hidden, weight, labels)
    ops.lmhead_backward(hidden, weight, labels, lse, None, g_lp, dweight=buf[1:V + 1], accumulate_dweight=True)
    dw = ops.lmhead_backward(hidden, weight, labels, lse, None, g_lp, need_dhidden=False)[1]
    assert torch.equal(buf[0], old[0]) and torch.equal(buf[-1], old[-1])
    size = old.abs().max() + (g_lp.abs() * hidden.float().abs().amax(1)).sum()
    assert (buf[1:V + 1].double() - old[1:V + 1].double() - dw.double()).abs().max() <= 2 * (T + 1) * 2.0 ** -24 * size
