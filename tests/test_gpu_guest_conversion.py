"""dhidden's launches that convert the next launch's kept logits beside their matrix instructions: the d(logits) they leave are those
of the conversion by itself, bit for bit, whatever the rows, the vocabulary's end, the options and the K ranges of the first launch."""
import pytest
import torch

pytestmark = pytest.mark.gpu

# H = 7168: 9 row tiles of 256 fill a round (one piece per slab), H = 2816: 23 (two)
CASES = [
    (4608, 7168, 640),         # two whole rounds, whole units
    (4607, 7168, 1000),        # the last row of a unit masked out, a vocabulary that ends inside a unit
    (4545, 7168, 577),         # one row in the last unit, one entry in the last unit
    (6911, 7168, 1027),        # three rounds
    (2800, 7168, 9001),        # a first launch of two row tiles in nine K ranges
    (4800, 7168, 2000),        # of one, too short to convert a whole round beside it
    (9000, 2816, 1300),
    (6001, 2816, 9001),
    (11700, 2816, 640),
]


def _both(dev, T, H, V, entropy, gen):
    from chatlearn_amd import ops
    h = torch.randn(T, H, generator=gen, device=dev).bfloat16()
    w = (torch.randn(V, H, generator=gen, device=dev) * H ** -0.5).bfloat16()
    y = torch.randint(0, V, (T,), generator=gen, device=dev)
    y[0], y[-1] = 0, V - 1
    y[5] = V + 3                                            # nobody's label
    glp = torch.randn(T, generator=gen, device=dev)
    glp[::7] = 0.0
    ge = torch.randn(T, generator=gen, device=dev) * 1e-2 if entropy else None
    z = ops.saved_logits_buffer(T, V, torch.bfloat16, dev)
    z.zero_()
    _, ent, _, lse = ops.lmhead_forward(h, w, y, 0.9, saved_logits=z)
    apart = z.clone()
    _, dw_apart = ops.lmhead_backward(h, w, y, lse, ent, glp, ge, 0.9, saved_logits=apart, need_dhidden=False)
    dh, dw = ops.lmhead_backward(h, w, y, lse, ent, glp, ge, 0.9, saved_logits=z)
    return h, w, y, glp, ge, z, apart, dh, dw, dw_apart


@pytest.mark.parametrize("entropy", [False, True])
@pytest.mark.parametrize("T,H,V", CASES)
def test_the_same_bits(dev, T, H, V, entropy):
    from chatlearn_amd import ops
    gen = torch.Generator(device=dev).manual_seed(T + V)
    *_, z, apart, dh, dw, dw_apart = _both(dev, T, H, V, entropy, gen)
    assert torch.equal(z.view(torch.int16), apart.view(torch.int16))
    assert torch.equal(dw, dw_apart)
    assert dh.isfinite().all()


def test_these_sizes_are_hosted(dev):
    from chatlearn_amd import ops
    plans = {c: ops.dhidden_guest_plan(*c) for c in CASES}
    assert all(p[0] > 0 and p[2] == (9 if c[1] == 7168 else 23) for c, p in plans.items()), plans
    assert any(p[1] > 1 for p in plans.values()), plans                       # a first launch with K ranges
    assert ops.dhidden_guest_plan(2304, 7168, 4100)[0] == 0                   # one round: nothing to convert beside it
    assert ops.dhidden_guest_plan(12836, 2560, 32000, partial_bytes=0)[0] == 0    # 510 tiles are two rounds of 256, not of 250


@pytest.mark.parametrize("T,H,V", [CASES[1], CASES[4], CASES[7]])
def test_dhidden_against_products_of_the_same_gradients(dev, T, H, V):
    """The rows' d(logits), read back out of the units, contracted in 64 bits: the contraction's own error is the result's rounding to
    bf16 (2^-9) and fp32 sums (K 2^-24 of the terms at most)."""
    gen = torch.Generator(device=dev).manual_seed(T)
    _, w, _, _, _, z, _, dh, _, _ = _both(dev, T, H, V, False, gen)
    rows, ld = z.shape
    units = z.view(-1).view(torch.bfloat16).reshape(rows // 64, ld // 64, 64, 64)
    worst = 0.0
    for a in range(0, T, 2048):
        b = min(T, a + 2048)
        dz = units[a // 64:(b + 63) // 64].permute(0, 2, 1, 3).reshape(-1, ld)[:b - a, :V].double()
        want = dz @ w.double()
        bound = want.abs() * 2.0 ** -8 + (dz.abs() @ w.double().abs()) * (V * 2.0 ** -24) + 1e-30
        worst = max(worst, float(((dh[a:b].double() - want).abs() / bound).max()))
    assert worst <= 1.0, worst


def test_through_a_row_order_and_kept_operands(dev):
    """A whole step whose masked rows are left out by an order, and one that leaves both operands of dW to a sum: against the same
    step in chunks of one round each, where nothing is hosted."""
    from chatlearn_amd import ops
    from chatlearn_amd.fused import grpo_head_step
    T, H, V = 5100, 7168, 2000
    gen = torch.Generator(device=dev).manual_seed(3)
    hidden = torch.randn(T, H, generator=gen, device=dev).bfloat16()
    weight = (torch.randn(V, H, generator=gen, device=dev) * H ** -0.5).bfloat16()
    labels = torch.randint(0, V, (T,), generator=gen, device=dev)
    old, ref = torch.randn(2, T, generator=gen, device=dev) * 0.1 - 7
    mask = (torch.rand(T, generator=gen, device=dev) < 0.9).int()
    live = int(mask.sum())
    assert ops.dhidden_guest_plan(live, H, V)[0] > 0 and ops.dhidden_guest_plan(2304, H, V)[0] == 0
    cu = torch.tensor([0, T], dtype=torch.int32, device=dev)
    run = lambda **kw: grpo_head_step(hidden, weight, labels, old, ref, torch.ones(1, device=dev), cu, mask, n_tokens_total=float(live),
                                      kl_coef=1e-3, **kw)
    one, parts = run(), run(keep_logits_chunk=2304)
    assert len(one["token_chunks"]) == 1 and len(parts["token_chunks"]) == 2
    rel = lambda a, b: float((a.double() - b.double()).norm() / b.double().norm())
    # the same products: other fp32 sums (K up to V and T terms), results of dhidden rounded to bf16 once more or less (2^-9)
    assert rel(one["dhidden"], parts["dhidden"]) < 2.0 ** -9
    assert rel(one["dweight"], parts["dweight"]) < 1e-5
    assert torch.equal(one["dhidden"][mask == 0], torch.zeros_like(one["dhidden"][mask == 0]))
    total = ops.DweightSum(weight, T, 10 ** 6)
    kept = run(_dweight_sum=total)
    assert torch.equal(kept["dhidden"], one["dhidden"])
    assert rel(total.finish(), one["dweight"]) < 2.0 ** -8                     # a sum of one contraction is rounded to bf16
