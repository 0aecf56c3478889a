"""The backward's contractions read an operand across its rows: d(logits) for dW, W for dhidden.  Sizes around the edges of a
slab (64 bf16 / 32 fp32 rows), of a 128-byte piece of columns and of a tile of 256, with NaN wherever memory ends."""
import pytest
import torch

pytestmark = pytest.mark.gpu

SHAPES = [(1, 64, 1), (64, 64, 64), (65, 192, 63), (129, 256, 65), (257, 320, 255), (300, 832, 257), (448, 576, 1100)]
SHAPES_FP32 = [(1, 32, 31), (33, 96, 33), (64, 288, 64), (257, 544, 255), (290, 32, 1025)]


def _fenced(x):
    """x as the front of a buffer whose rest is NaN."""
    buf = torch.full((x.numel() + 70000,), float("nan"), dtype=x.dtype, device=x.device)
    buf[:x.numel()] = x.reshape(-1)
    return buf[:x.numel()].view(x.shape)


@pytest.mark.parametrize("T,H,V,dtype", [s + (torch.bfloat16,) for s in SHAPES] + [s + (torch.float32,) for s in SHAPES_FP32])
@pytest.mark.parametrize("keep", [True, False])
def test_contractions_at_the_edges(dev, T, H, V, dtype, keep):
    """Against the contractions in 64 bits.  Bounds: a logit is off by its half rounding (kept 16-bit ones, 2^-11) and its fp32
    sum, which moves its probability by that much of itself, twice with the shift of lse; d(logits) is rounded to the operand's type
    (half a unit in the last place: 2^-8 or 2^-24), so is the result, and K terms are summed in fp32."""
    from chatlearn_amd import ops
    g = torch.Generator().manual_seed(1000 * T + V)
    hidden = torch.randn(T, H, generator=g).to(dtype)
    weight = (torch.randn(V, H, generator=g) * 0.2).to(dtype)
    labels = torch.randint(0, V, (T,), generator=g)
    g_lp = torch.randn(T, generator=g)
    g_lp[::5] = 0.0
    h, w = _fenced(hidden.to(dev)), _fenced(weight.to(dev))
    z = None
    if keep:
        z = ops.saved_logits_buffer(T, V, dtype, dev)
        z.fill_(float("nan"))
    y, glp = labels.to(dev), g_lp.to(dev)
    _, _, _, lse = ops.lmhead_forward(h, w, y, saved_logits=z)
    dh, dw = ops.lmhead_backward(h, w, y, lse, None, glp, saved_logits=z)
    h64, w64 = hidden.double(), weight.double()
    zz = h64 @ w64.t()
    p = torch.softmax(zz, -1)
    dz = g_lp.double()[:, None] * (torch.nn.functional.one_hot(labels, V) - p)
    unit = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -24
    zerr = (h64.abs() @ w64.abs().t()) * H * 2.0 ** -24 + (zz.abs() * 2.0 ** -11 if keep and dtype == torch.bfloat16 else 0)
    dzerr = g_lp.double().abs()[:, None] * p * (2 * zerr.max(-1, keepdim=True).values + 2.0 ** -20)
    for got, want, err_in, terms, K, what in ((dh, dz @ w64, dzerr @ w64.abs(), dz.abs() @ w64.abs(), V, "dhidden"),
                                              (dw, dz.t() @ h64, dzerr.t() @ h64.abs(), dz.abs().t() @ h64.abs(), T, "dW")):
        err = (got.double().cpu() - want).abs()
        bound = 1.01 * err_in + terms * (unit + K * 2.0 ** -24) + want.abs() * unit + 1e-30
        assert torch.isfinite(got.float()).all(), what
        assert (err <= bound).all(), (what, float((err / bound).max()))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_weight_read_across_gives_the_products_of_its_transpose(dev, dtype):
    """dhidden with a kept W^T and with W itself: the same products in the same order, bit for bit."""
    from chatlearn_amd import ops
    T, H, V = 700, 320, 2100
    g = torch.Generator().manual_seed(3)
    h, w = torch.randn(T, H, generator=g).to(dtype).to(dev), (torch.randn(V, H, generator=g) * 0.1).to(dtype).to(dev)
    y, glp = torch.randint(0, V, (T,), generator=g).to(dev), torch.randn(T, generator=g).to(dev)
    out = []
    for wt in (None, ops.weight_t_buffer(w)):
        z = ops.saved_logits_buffer(T, V, dtype, dev)
        _, _, _, lse = ops.lmhead_forward(h, w, y, saved_logits=z)
        out.append(ops.lmhead_backward(h, w, y, lse, None, glp, saved_logits=z, weight_t=wt, need_dweight=False)[0])
    assert torch.equal(out[0], out[1])


def test_kept_operands_begin_at_any_64_rows(dev):
    """dW over chunks of 1, 65 and 200 rows, each behind the other's 64-row places, against one chunk of all of them."""
    from chatlearn_amd import ops
    from chatlearn_amd.fused import grpo_head_step
    H, V, sizes = 192, 900, (1, 65, 200)
    g = torch.Generator().manual_seed(8)
    T = sum(sizes)
    hidden = torch.randn(T, H, generator=g).bfloat16().to(dev)
    weight = (torch.randn(V, H, generator=g) * 0.1).bfloat16().to(dev)
    labels = torch.randint(0, V, (T,), generator=g).to(dev)
    old, ref = torch.randn(2, T, generator=g).to(dev) * 0.1 - 7
    total = ops.DweightSum(weight, T, 10 ** 6)
    total.place(512)
    total.dzt.fill_(float("nan")), total.hidt.fill_(float("nan"))
    dhidden, lo = [], 0

    def step(lo, n, **kw):
        cut = slice(lo, lo + n)
        return grpo_head_step(hidden[cut], weight, labels[cut], old[cut], ref[cut], torch.ones(1, device=dev),
                              torch.tensor([0, n], dtype=torch.int32, device=dev), None, n_tokens_total=float(T), kl_coef=1e-3, **kw)

    for n in sizes:
        dhidden.append(step(lo, n, _dweight_sum=total)["dhidden"])
        lo += n
    dw = total.finish()
    parts = [step(sum(sizes[:i]), n) for i, n in enumerate(sizes)]
    assert torch.equal(torch.cat(dhidden), torch.cat([o["dhidden"] for o in parts]))
    want = sum(o["dweight"].double() for o in parts)
    # the same products, summed in another order in fp32
    assert (dw.double() - want).abs().max() <= 2.0 ** -20 * T * want.abs().max()
