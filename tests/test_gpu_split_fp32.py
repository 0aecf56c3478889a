"""fp32 operands run on the 16-bit matrix cores as three parts each (SplitTile): exponents far from 1, and elements that have no
such parts - infinite and NaN ones, and finite ones whose first part rounds to infinity - which the fp32 instructions compute."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _inputs(dev, T, H, V, seed):
    g = torch.Generator(device=dev).manual_seed(seed)
    h = torch.randn(T, H, generator=g, device=dev)
    w = torch.randn(V, H, generator=g, device=dev) * H ** -0.5
    return h, w, torch.randint(0, V, (T,), generator=g, device=dev), torch.randn(T, generator=g, device=dev)


def _bound(K):
    """Relative error of a sum of K products: six additions to the fp32 sum per 32 of them, each off by half a unit in the last
    place of a sum that grows with the square root of its terms, the parts left out 2^-26 of a product; fourfold."""
    return 4 * (2.0 ** -24 * (6 * K / 32) ** 0.5 + 2.0 ** -25)


@pytest.mark.parametrize("H", [32, 64, 96, 1024])
@pytest.mark.parametrize("power", [-60, -20, 0, 40, 90])
def test_products_at_any_exponent(dev, H, power):
    """hidden * 2^power against W * 2^-power: the same logits; d(logits) and W, d(logits) and hidden at those exponents."""
    from chatlearn_amd import ops
    T, V = 300, 1300
    h, w, y, glp = _inputs(dev, T, H, V, H)
    h, w = h * 2.0 ** power, w * 2.0 ** -power
    z = ops.saved_logits_buffer(T, V, torch.float32, dev)
    lp, _, _, lse = ops.lmhead_forward(h, w, y, saved_logits=z)
    dh, dw = ops.lmhead_backward(h, w, y, lse, None, glp, saved_logits=z)
    zz = h.double() @ w.double().t()
    p = torch.softmax(zz, 1)
    dz = glp.double()[:, None] * (torch.nn.functional.one_hot(y, V) - p)
    want_lp = torch.log_softmax(zz, 1).gather(1, y[:, None])[:, 0]
    rel = lambda got, want: float((got.double() - want).norm() / want.norm())
    # logits of unit variance and their lse of about 7, in the exponent of a probability: twice the larger one's fp32 unit beside the sum's error
    small = _bound(H) + 2.0 ** -22
    assert rel(lp, want_lp) < small
    assert rel(dh, dz @ w.double()) < _bound(V) + 2 * small
    assert rel(dw, dz.t() @ h.double()) < _bound(T) + 2 * small


@pytest.mark.parametrize("value", [float("inf"), float("-inf"), float("nan"), 3.4e38])
@pytest.mark.parametrize("T,V", [(130, 700), (2048, 20000)])          # one tile a workgroup, runs of several
def test_forward_around_an_element_without_parts(dev, T, V, value):
    """An element of W in the middle of a workgroup's tiles: its logits are what fp32 makes of them, every other one is untouched."""
    from chatlearn_amd import ops
    H, v0 = 96, V // 2
    h, w, y, _ = _inputs(dev, T, H, V, T)
    h[:, 7] = h[:, 7].abs() + 0.1
    y[:] = torch.where(y == v0, v0 + 1, y)
    w[v0, 7] = value
    zz = h.double() @ w.double().t()
    lp, _, mx, lse = ops.lmhead_forward(h, w, y)
    if value == float("-inf"):                # probability 0
        assert torch.allclose(lp.double(), torch.log_softmax(zz, 1).gather(1, y[:, None])[:, 0], rtol=1e-5, atol=1e-5)
        assert torch.allclose(lse.double(), torch.logsumexp(zz, 1), rtol=1e-6)
    elif value == 3.4e38:                     # the row's largest logit, to fp32 (the statistics, in units of log 2, overflow on it)
        fits = zz[:, v0] < 3.4e38
        assert fits.any() and (mx.double()[fits] - zz[fits, v0]).abs().max() <= 1e-6 * 3.4e38
    else:
        assert not lse.isfinite().any()
    # a token of that kind leaves the others alone
    h, w, y, _ = _inputs(dev, T, H, V, T)
    clean = ops.lmhead_forward(h, w, y)
    h[5, 3] = value
    lp, ent, mx, lse = ops.lmhead_forward(h, w, y)
    rest = torch.arange(T, device=dev) != 5
    for a, b in zip((lp, ent, mx, lse), clean):
        assert torch.allclose(a[rest], b[rest], rtol=1e-5, atol=1e-5)
    assert value == 3.4e38 or not lse[5].isfinite()


@pytest.mark.parametrize("adds", [False, True])
@pytest.mark.parametrize("V,H", [(2100, 320), (151936, 512)])         # one workgroup per tile, walks over several
def test_gradients_around_elements_without_parts(dev, V, H, adds):
    """An infinite hidden state, and an infinite upstream gradient: infinities of the sign that the products have, in the column of
    the one and the token of the other, sums as ever beside them (also where they are added to what is there)."""
    from chatlearn_amd import ops
    T, t0, k0 = 160, 70, 290
    h, w, y, glp = _inputs(dev, T, H, V, V)
    y[:] = torch.arange(T, device=dev) * 3
    z = ops.saved_logits_buffer(T, V, torch.float32, dev)
    _, _, _, lse = ops.lmhead_forward(h, w, y, saved_logits=z)
    kept = z.clone()
    zz = h.double() @ w.double().t()
    dz = glp.double()[:, None] * (torch.nn.functional.one_hot(y, V) - torch.softmax(zz, 1))
    base = torch.full((V, H), 2.0, device=dev)
    run = lambda hid, g: ops.lmhead_backward(hid, w, y, lse, None, g, saved_logits=z.copy_(kept),
                                             dweight=base.clone() if adds else None, accumulate_dweight=adds)
    want = dz.t() @ h.double() + (2.0 if adds else 0.0)
    h_inf = h.clone()
    h_inf[t0, k0] = float("inf")
    dh, dw = run(h_inf, glp)
    cols = torch.arange(H, device=dev) != k0
    err = (dw[:, cols].double() - want[:, cols]).norm() / want[:, cols].norm()
    assert err < _bound(T) + 2.0 ** -19
    assert torch.equal(dw[:, k0], torch.sign(dz[t0]).float() * float("inf"))
    assert dh.isfinite().all()
    g_inf = glp.clone()
    g_inf[t0] = float("inf")
    dh, dw = run(h, g_inf)
    others = torch.arange(T, device=dev) != t0
    want_dh = dz @ w.double()
    assert not dh[t0].isfinite().any() and (dh[others].double() - want_dh[others]).norm() / want_dh[others].norm() < _bound(V) + 2.0 ** -19
    plain = torch.arange(V, device=dev) != y[t0]                       # the label's own row is inf - inf
    assert torch.equal(dw[plain], (-torch.sign(h[t0]) * float("inf")).expand(V, H)[plain])
