"""The router's path for many bf16 tokens: logits on the bf16 matrix cores with an error bound; the winners, and what the choice
hangs on, anew in fp64.  Indices are those of the exact logits and weights those of fp64 logits, whatever the tokens look like."""
import numpy as np
import pytest
import torch

from oracle import moe_oracle as orc

pytestmark = pytest.mark.gpu


def _screened(T, H, E, K, renorm=True, normed=False):
    import ctypes as C
    from on_device_sd_amd import _lib, ops
    return bool(_lib.load().odsd_router_screened(C.byref(ops.make_shape(T, H, E, K, 128, renorm, torch.bfloat16)), normed))


@pytest.mark.parametrize("T,H,E,K,renorm,screened", [
    (1700, 4096, 128, 8, True, True),
    (2317, 2048, 128, 8, True, True),      # ragged token tile
    (4100, 384, 224, 3, True, True),       # an odd number of steps, experts that do not fill a workgroup; four logits per lane
    (700, 2048, 512, 4, True, True),       # two steps in the first slice and the last
    (1500, 4096, 512, 16, True, True),     # most winners, eight logits per lane
    (8200, 4096, 66, 1, True, True),       # one winner and its runner-up
    (1500, 2048, 300, 6, True, True),      # eight logits per lane, some past the experts
    # and their neighbours in fp64
    (1000, 4096, 128, 8, True, False),
    (2017, 2048, 128, 8, False, False),
    (27500, 128, 128, 4, True, False),
    (5300, 384, 224, 3, False, False),
    (1300, 5248, 66, 63, True, False),
    (1100, 1024, 512, 1, False, False),
])
def test_indices_and_weights(dev, T, H, E, K, renorm, screened):
    from on_device_sd_amd import ops
    print("router screen", T, H, E, K, renorm, flush=True)
    assert _screened(T, H, E, K, renorm) == screened
    g = torch.Generator().manual_seed(T + E)
    x = torch.randn(T, H, generator=g).to(torch.bfloat16)
    wg = (torch.randn(E, H, generator=g) * 0.02).to(torch.bfloat16)
    # exact ties and ties up to the last bit of one weight, among the popular experts as well
    wg[E // 2] = wg[1]
    wg[E - 1] = wg[3]
    wg[E - 1, 5] = wg[3, 5] * (1 + 2.0 ** -7)
    wg[2] = wg[4]
    wg[2, H - 1] = wg[4, H - 1] * (1 + 2.0 ** -7)
    x[0] = 0.0                                            # every logit is zero
    x[1] = x[1] * 1e-30                                   # squares vanish, the row has not
    x[2] = x[2] * 2.0 ** 124                              # sums beyond fp32
    x[3, 7] = 3000.0                                      # an outlier
    x[4, 1:] = 0.0                                        # one product per logit
    x[5] = x[6]
    x[T - 1] = x[T - 1] * 1e-20
    idx, w, idx64, x16 = ops.router_topk(x.to(dev), wg.to(dev), K, renorm, want_f16=True, want_int64=True)
    lo = orc.router_logits(x, wg)
    idx_o, w_o = orc.route(lo, K, renorm)
    assert np.array_equal(idx.cpu().numpy(), idx_o)
    assert np.array_equal(idx64.cpu().numpy(), idx_o.astype(np.int64))
    # the oracle's weights are fp32 from fp64 logits: half a unit each, one for exp, and the logits' own error
    np.testing.assert_allclose(w.cpu().numpy(), w_o, rtol=2e-6, atol=1e-7)
    sel = lo.double().numpy()[np.arange(T)[:, None], idx_o]
    p = np.exp(sel - sel[:, :1])
    p /= p.sum(1, keepdims=True) if renorm else np.exp(lo.double().numpy() - sel[:, :1]).sum(1, keepdims=True)
    err = np.linalg.norm(w.cpu().numpy() - p, axis=1) / np.linalg.norm(p, axis=1)
    print("weights against 64 bits, worst token %.2e" % err.max(), flush=True)
    # K - 1 additions, exp's unit, the division, and a logit's distance from the largest in fp32 (under 17 where a weight counts)
    assert np.all(err[np.arange(T) != 2] < (K + 2 + 2 * 17) * 2.0 ** -24) and err[2] < 1e-6
    assert torch.equal(x16.cpu(), torch.clamp(x.float(), -65504.0, 65504.0).to(torch.float16))
    again = ops.router_topk(x.to(dev), wg.to(dev), K, renorm)
    assert torch.equal(again[0], idx) and torch.equal(again[1].view(torch.int32), w.view(torch.int32))


# What the tokens and the router have in common in a trained model, and what makes a sum of 32 columns in fp32 lose the rest.
def _rows(kind, T, H, E):
    g = torch.Generator().manual_seed(T + H + E + len(kind))
    x, wg = torch.randn(T, H, generator=g), torch.randn(E, H, generator=g) * 0.02
    if kind == "residual_stream":
        x *= 8
    elif kind == "large_columns":
        x[:, [12, 99]] *= 1000.0
    elif kind == "common_component":
        x += 1.0
        wg += 0.02 * torch.randn(H, generator=g).abs()
    elif kind == "shared_column":                         # that all experts weight alike
        x[:, 33] = 300.0 * (1 + 0.1 * torch.randn(T, generator=g))
        wg[:, 33] = 0.5
    elif kind == "cancelling":
        # Two columns of every 32 cancel exactly and take the last bits of the others, which make the choice, with them; so
        # large that half of the neighbours are closer than what the screen leaves open, 35 * 2^-22 |x||w|, and half a few times that apart.
        for c in range(0, H, 32):
            x[:, c + 3], x[:, c + 20] = 10300 / H ** 0.5, -10300 / H ** 0.5
            wg[:, c + 3] = wg[:, c + 20] = 0.125
    elif kind == "swallowed":
        # One product of 1 in every 32, the others below half a unit in its last place in fp32 and all that tells the experts apart:
        # what a sum of 32 loses at most, which the bound has to leave open.
        x, wg = 2.0 ** -13 * (1 + torch.rand(T, H, generator=g)), 2.0 ** -12 * torch.rand(E, H, generator=g)
        x[:, ::32] = wg[:, ::32] = 1.0
    return x.to(torch.bfloat16), wg.to(torch.bfloat16)


@pytest.mark.parametrize("kind", ["residual_stream", "large_columns", "common_component", "shared_column", "cancelling", "swallowed"])
@pytest.mark.parametrize("T,H,E,K", [(1700, 4096, 128, 8), (4100, 384, 224, 3), (2100, 1024, 512, 8)])
def test_weights_are_those_of_fp64_logits(dev, T, H, E, K, kind):
    from on_device_sd_amd import ops
    print("router screen, weights", T, H, E, K, kind, flush=True)
    assert _screened(T, H, E, K)
    x, wg = _rows(kind, T, H, E)
    x, wg = x.to(dev), wg.to(dev)
    idx, w, _, _ = ops.router_topk(x, wg, K, True)
    lo = x.double() @ wg.double().t()
    val, pos = lo.topk(K, dim=1)
    sel = lo.gather(1, idx.long())
    # (two fp64 sums of H products may order neighbours differently only within their own rounding)
    slack = H * 2.0 ** -53 * (x.double().abs() @ wg.double().abs().t()).amax(1, keepdim=True)
    assert ((sel - val).abs() <= slack).all()
    # Each weight against 64 bits.  num: the difference rounded to fp32 and exp's own unit; den: the same of its terms, weighted, and
    # K - 1 additions; the division.  In units of 2^-24 of the weight.
    d = sel - sel[:, :1]
    p = d.exp()
    p = p / p.sum(1, keepdim=True)
    units = d.abs() + 2 + (p * (d.abs() + 2)).sum(1, keepdim=True) + (K - 1) + 1
    err = (w.double() - p).abs()
    print("worst weight %.2e of itself" % (err / p).max().item(), flush=True)
    assert (err <= p * (units * 2.0 ** -24) + 2.0 ** -149).all()
    # the call that returns the logits has them in fp64: a weight differs only where their last bits turn a rounding
    lg = torch.empty(T, E, dtype=torch.float64, device=dev)
    idx2, w2, _, _ = ops.router_topk(x, wg, K, True, logits_out=lg)
    assert torch.equal(idx, idx2)
    assert (w.view(torch.int32) != w2.view(torch.int32)).sum().item() <= 1e-4 * T * K


def test_tokens_that_are_not_finite_leave_the_others_alone(dev):
    from on_device_sd_amd import ops
    T, H, E, K = 1600, 4096, 128, 8
    assert _screened(T, H, E, K)
    g = torch.Generator().manual_seed(3)
    x = torch.randn(T, H, generator=g).to(torch.bfloat16)
    wg = (torch.randn(E, H, generator=g) * 0.02).to(torch.bfloat16)
    x[7, 9] = float("nan")
    x[8, 11] = float("inf")
    idx, w, _, _ = ops.router_topk(x.to(dev), wg.to(dev), K, True)
    good = np.r_[0:7, 9:T]
    idx_o, w_o = orc.route(orc.router_logits(x[good], wg), K, True)
    assert np.array_equal(idx.cpu().numpy()[good], idx_o)
    np.testing.assert_allclose(w.cpu().numpy()[good], w_o, rtol=2e-6, atol=1e-7)
    assert idx.min() >= 0 and idx.max() < E
    assert idx[7].tolist() == list(range(K))              # every logit is a NaN: a tie
    pos = (wg[:, 11].float() > 0).nonzero().flatten()[:K].tolist()
    assert idx[8].tolist() == pos                         # and here every logit is one of the infinities


# (an odd number of winners: the last group of a token's experts is not full)
@pytest.mark.parametrize("T,H,E,K,I", [(3601, 4096, 128, 8, 128), (2501, 4096, 512, 11, 128)])
def test_norm_folded_in_gives_the_same_bits(dev, T, H, E, K, I):
    """The RMSNorm applied on the fly from row statistics against the stand-alone one in front of the router."""
    import on_device_sd_amd as odsd
    from on_device_sd_amd import ops
    assert _screened(T, H, E, K) and _screened(T, H, E, K, normed=True)
    g = torch.Generator().manual_seed(12)
    x = torch.randn(T, H, generator=g).to(torch.bfloat16).to(dev)
    gate = (0.02 * torch.randn(E, H, generator=g)).to(torch.bfloat16).to(dev)
    gate[9] = gate[4]
    norm = (1 + 0.1 * torch.randn(H, generator=g)).to(torch.bfloat16).to(dev)
    bank = odsd.W4ExpertBank(E, H, I, dev)
    for e in range(E):
        bank.load_expert(e, *(0.02 * torch.randn(*s, generator=g) for s in ((I, H), (I, H), (H, I))))
    plan = ops.MoeForwardPlan(T, H, E, K, I, True, torch.bfloat16, dev)
    ss = ops.row_stats(T, H, dev)
    h1, a, b = torch.empty_like(x), torch.empty_like(x), torch.empty_like(x)
    plan.run(x, gate, bank.table(), norm, 1e-6, add_residual=True, out_act=h1, row_sumsq_out=ss)
    ra = plan.run(h1, gate, bank.table(), norm, 1e-6, add_residual=True, out_act=a)
    idx_a, w_a = ra.idx.clone(), ra.w.clone()
    rb = plan.run(h1, gate, bank.table(), norm, 1e-6, add_residual=True, out_act=b, row_sumsq_in=ss)
    assert torch.equal(idx_a, rb.idx) and torch.equal(w_a.view(torch.int32), rb.w.view(torch.int32)) and torch.equal(a, b)
