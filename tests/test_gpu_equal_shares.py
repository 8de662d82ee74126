"""Calls of few rows per expert at the edges of the equal-share kernel: fewer units than workgroups, shares that end
inside an expert, experts with 16, 17 and more rows (further passes), experts without rows and without weights, every
split of the two reductions that it has, the most experts and pairs it takes, the last average row count of its rule;
with the routing (up to 8 tokens) and the dispatch inside (whole block) and with caller-made dispatch arrays (stage calls)."""
import numpy as np
import pytest
import torch

from oracle import moe_oracle as orc
from tests.helpers import canon_to_oracle, check_output_relative

pytestmark = pytest.mark.gpu


def _bank(dev, H, E, I, g, distinct=6, w_down=0.05):
    """Bank of E experts; the weights repeat after `distinct` of them (the oracle then quantises few)."""
    import on_device_sd_amd as odsd
    bank = odsd.W4ExpertBank(E, H, I, dev)
    mk = lambda r, c, scale=0.05: torch.randn(r, c, generator=g) * scale  # noqa: E731
    ws = [(mk(I, H), mk(I, H), mk(H, I, w_down)) for _ in range(min(E, distinct))]
    experts = {}
    for e in range(E):
        if e < distinct:
            experts[e] = canon_to_oracle(bank.load_expert(e, *ws[e], keep_canonical=True))
        else:
            bank.load_expert(e, *ws[e % distinct])
            experts[e] = experts[e % distinct]
    return bank, experts


@pytest.mark.parametrize("T,H,E,K,I,crowd", [
    (1, 2048, 4, 1, 768, 0),         # one expert: 48 and 16 units for 256 workgroups
    (33, 2048, 16, 2, 768, 16),      # one expert with exactly 16 rows
    (33, 2048, 16, 2, 768, 17),      # ... and with 17: a second pass of one row
    (96, 2048, 16, 2, 1536, 96),     # six passes over one expert; 12 rows on average, the last of the rule; 4 x 3 groups
    (7, 4096, 12, 3, 2048, 0),       # 32 groups in gate_up; 16 in down
    (8, 2048, 128, 8, 768, 5),       # the most tokens that it routes for itself, and the most experts
    (9, 2048, 65, 8, 768, 0),        # one token more
    (8, 2048, 65, 64, 768, 0),       # the most choices per token
    (20, 4096, 8, 2, 4096, 18),      # two splits of the down reduction
    (40, 4096, 8, 2, 14336, 0),      # seven splits: 252 workgroups
    (64, 2048, 512, 8, 768, 3),      # the most experts
    (511, 2048, 384, 8, 768, 40),    # nearly the most pairs
    (8, 3072, 8, 2, 512, 0),         # 24 groups in gate_up, the top-k inside; 2 x 2 in down
    (6, 3072, 96, 8, 1024, 4),       # more than 64 experts to choose from; 4 x 2
    (70, 3072, 64, 8, 512, 17),      # 560 pairs
    (200, 3072, 256, 8, 512, 33),    # 1600 pairs
    (40, 2048, 16, 2, 3072, 21),     # 8 x 3 groups
    (9, 3072, 16, 2, 2304, 0),       # 2 x 3 groups and three splits: 255 workgroups
    (20, 4096, 8, 2, 2560, 17),      # 2 x 2 groups and five splits
    (33, 2048, 16, 2, 4608, 16),     # 4 x 3 groups and three splits
    (12, 2048, 8, 2, 1280, 0),       # ten groups: no split of theirs; the other plan
])
def test_equal_shares(dev, T, H, E, K, I, crowd):
    from on_device_sd_amd import ops
    print("equal shares", T, H, E, K, I, crowd, flush=True)
    g = torch.Generator().manual_seed(T + H + E + K + I + crowd)
    wg = (torch.randn(E, H, generator=g) * 0.02).to(torch.bfloat16)
    x = torch.randn(T, H, generator=g).to(torch.bfloat16)
    if crowd:
        # exactly the first `crowd` tokens choose expert E - 2: it alone looks at column 0
        wg[:, 0] = 0.0
        wg[E - 2] = 0.0
        wg[E - 2, 0] = 1.0
        x[:, 0] = -40.0
        x[:crowd, 0] = 40.0
    bank, experts = _bank(dev, H, E, I, g)
    xd, wgd, table = x.to(dev), wg.to(dev), bank.table()
    out = ops.moe_forward(xd, wgd, table, K, I, renorm=True)
    ref, idx, w = orc.moe_block(x, wg, experts, K, True)
    counts, offsets, perm, _ = orc.dispatch(idx, E)
    assert not crowd or counts[E - 2] == crowd
    assert np.array_equal(out.idx.cpu().numpy(), idx)
    assert np.array_equal(out.counts.cpu().numpy(), counts)
    assert np.array_equal(out.offsets.cpu().numpy(), offsets)
    assert np.array_equal(out.perm.cpu().numpy(), perm)
    assert np.allclose(out.w.cpu().numpy(), w, rtol=2e-6, atol=0)    # fp32 softmax of fp64 logits: a few units in the last place
    # h is rounded to fp16 once (2^-11): well inside the helper's 1e-2 of the largest and 2e-3 of the mean output
    check_output_relative(out.out_f32, ref)
    again = ops.moe_forward(xd, wgd, table, K, I, renorm=True)
    assert torch.equal(again.out_f32, out.out_f32)
    # the same kernels on caller-made dispatch arrays, one expert's weights missing
    gone = int(idx[0, 0])
    hole = table.clone()
    hole[gone] = 0
    x16, i32, wd = ops.to_f16(xd), torch.from_numpy(idx.astype(np.int32)).to(dev), torch.from_numpy(w).to(dev)
    disp = ops.dispatch(i32, E)
    got, _ = ops.experts_w4(x16, hole, i32, wd, disp, I, torch.bfloat16, want_f32=True, want_act=False)
    ref_hole = orc.moe_forward(x, idx, np.where(idx == gone, 0.0, w).astype(np.float32), experts)
    check_output_relative(got, ref_hole)


@pytest.mark.parametrize("T,H,E,K,I", [
    (8, 2048, 8, 2, 2048),       # one slice of sums where the reduction was to be split
    (16, 4096, 16, 2, 2048),
    (5, 4096, 8, 2, 14336),      # seven slices
])
def test_few_tokens_keep_fp32_sums(dev, T, H, E, K, I):
    """Expert outputs far beyond fp16's largest value: fp32 sums carry them, fp16 ones would be clamped to 65504."""
    from on_device_sd_amd import ops
    print("equal shares, large outputs", T, H, E, K, I, flush=True)
    g = torch.Generator().manual_seed(T + H + I)
    wg = (torch.randn(E, H, generator=g) * 0.02).to(torch.bfloat16)
    x = torch.randn(T, H, generator=g).to(torch.bfloat16)
    bank, experts = _bank(dev, H, E, I, g, distinct=3, w_down=8000.0)
    out = ops.moe_forward(x.to(dev), wg.to(dev), bank.table(), K, I, renorm=True)
    ref, idx, _ = orc.moe_block(x, wg, experts, K, True)
    assert np.array_equal(out.idx.cpu().numpy(), idx)
    assert (ref.abs() > 65504).float().mean() > 0.5       # (weights of at most 1: the sums themselves are larger still)
    check_output_relative(out.out_f32, ref)
