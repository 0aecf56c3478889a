"""Row tiles narrower than 256: the forward takes blocks of 128, 160, 192, 224 or 256 tokens, dhidden of 128, 192 or 256 rows,
whichever wastes least.  Every width at its edges, with and without kept logits, against 64 bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu


# (tokens, vocabulary, the block width that the plan takes)
CASES = [(1, 300, 128), (128, 9000, 128), (129, 70000, 160), (160, 70000, 160), (161, 70000, 192), (193, 70000, 224), (224, 70000, 224),
         (225, 70000, 256), (257, 70000, 160), (321, 70000, 192), (385, 70000, 224), (449, 70000, 256), (600, 70000, 128)]


@pytest.mark.parametrize("T,V,width", CASES)
@pytest.mark.parametrize("ordered", [False, True])
def test_forward_and_backward_of_every_width(dev, T, V, width, ordered):
    """Statistics: fp32 sums over V entries, 2^-16 relative of the magnitudes that meet in them.  Gradients: d(logits) rounded to
    bf16 and the softmax rebuilt from half logits (2^-8 each at most), the result rounded once more; the bound is on rows."""
    from chatlearn_amd import ops
    H = 128
    n_tb, _, _, planned, _ = ops.lmhead_forward_tile_plan(T, H, V, torch.bfloat16)
    assert planned == width and n_tb == -(-T // width)
    g = torch.Generator(device=dev).manual_seed(T + V)
    hidden = torch.randn(T, H, generator=g, device=dev).bfloat16()
    weight = (torch.randn(V, H, generator=g, device=dev) * 0.1).bfloat16()
    labels = torch.randint(0, V, (T,), generator=g, device=dev)
    g_lp = torch.randn(T, generator=g, device=dev)
    z = ops.saved_logits_buffer(T, V, torch.bfloat16, dev).fill_(float("nan"))
    row_map = torch.randperm(T, generator=g, device=dev).to(torch.int32) if ordered else None
    lp, ent, _, lse = ops.lmhead_forward(hidden, weight, labels, saved_logits=z, saved_row_map=row_map)
    lp2, ent2, _, lse2 = ops.lmhead_forward(hidden, weight, labels)
    assert torch.equal(lse, lse2) and torch.equal(lp, lp2) and torch.equal(ent, ent2)
    z64 = hidden.double() @ weight.double().t()
    ls64 = torch.log_softmax(z64, -1)
    p64 = ls64.exp()
    assert (lse.double() - torch.logsumexp(z64, -1)).abs().max() < 2.0 ** -16 * 32
    assert (lp.double() - ls64.gather(1, labels[:, None])[:, 0]).abs().max() < 2.0 ** -16 * 32
    assert (ent.double() + (p64 * ls64).sum(-1)).abs().max() < 2.0 ** -16 * 32
    kept = ops.saved_logits_rowmajor(z, T, V)
    want = z64 if row_map is None else torch.empty_like(z64).index_copy_(0, row_map.long(), z64)
    assert ((kept.double() - want).abs() <= 2.0 ** -10 * want.abs() + 1e-4).all()
    pick = slice(None) if row_map is None else torch.argsort(row_map)
    dh, dw = ops.lmhead_backward(hidden[pick], weight, labels[pick], lse[pick], None, g_lp[pick], saved_logits=z)
    dz = (-p64).scatter_add_(1, labels[:, None], torch.ones(T, 1, dtype=torch.float64, device=dev)) * g_lp.double()[:, None]
    dh64, dw64 = (dz @ weight.double())[pick], dz.t() @ hidden.double()
    err = (dh.double() - dh64).norm(dim=1) / dh64.norm(dim=1).clamp_min(1e-30)
    assert err.max() < 3 * 2.0 ** -8
    assert (dw.double() - dw64).norm() < 3 * 2.0 ** -8 * dw64.norm()


@pytest.mark.parametrize("rows,H,width", [(rows, 256, 128) for rows in (1, 127, 128, 129, 190, 192, 193, 257, 320, 384, 385)] +
                         [(1, 2048, 128), (128, 2048, 128), (129, 2048, 192), (192, 2048, 192), (193, 2048, 128), (256, 2048, 128),
                          (257, 2048, 192), (320, 2048, 192), (384, 2048, 192), (385, 2048, 256)])
def test_dhidden_of_few_rows_matches_itself_row_by_row(dev, rows, H, width):
    """dhidden's row tiles and K ranges depend on the number of rows; a row's gradient does not, but for the order of an fp32
    sum over 33000 entries and the rounding to bf16: 2^-8 of the row's norm."""
    from chatlearn_amd import ops
    V = 33000
    bulk, k_ranges, planned, _ = ops.dhidden_tile_plan(rows, H, V, torch.bfloat16)
    assert bulk == 0 and k_ranges > 1 and planned == width
    g = torch.Generator(device=dev).manual_seed(5)
    hidden = torch.randn(400, H, generator=g, device=dev).bfloat16()
    weight = (torch.randn(V, H, generator=g, device=dev) * 0.1).bfloat16()
    labels = torch.randint(0, V, (400,), generator=g, device=dev)
    g_lp = torch.randn(400, generator=g, device=dev)

    def grad(n):
        z = ops.saved_logits_buffer(n, V, torch.bfloat16, dev)
        _, _, _, lse = ops.lmhead_forward(hidden[:n], weight, labels[:n], saved_logits=z)
        return ops.lmhead_backward(hidden[:n], weight, labels[:n], lse, None, g_lp[:n], saved_logits=z, need_dweight=False)[0]
    got, want = grad(rows).double(), grad(400)[:rows].double()
    assert ((got - want).norm(dim=1) <= 2.0 ** -8 * want.norm(dim=1)).all()
