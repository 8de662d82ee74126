"""The 48-row streaming kernel at its edges: experts with 1, 16, 17, 32, 33, 48, 49 and more rows (every number of token
blocks, a second and a third pass), without rows and without weights, the ends of its rule, weight rows that end inside a
workgroup's 16 blocks, unsplit and split down reductions, splits of unequal length; and the 32- and 64-row kernel where
several workgroups share an expert's passes, at the edges of those."""
import numpy as np
import pytest
import torch

from oracle import moe_oracle as orc
from tests.helpers import check_output_relative
from tests.test_gpu_equal_shares import _bank

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,H,E,K,I,crowd", [
    (104, 4096, 8, 1, 4224, (1, 16, 17, 0, 32)),     # 13 rows on average, the first of the rule; 33 groups in down, splits of 9 and 6
    (272, 4096, 8, 1, 4224, (33, 48, 49, 97, 0)),    # 34 rows, the last; passes of one row and three passes
    (129, 4096, 64, 9, 128, (100,)),                 # 1161 pairs: more than the other kernel scans; one group in down
    (600, 4224, 40, 2, 256, (47, 16)),               # 33 groups; 264 blocks of output rows: the last workgroup has 8
    (100, 8192, 4, 1, 4608, (31, 2)),                # 64 groups
    (600, 512, 32, 2, 384, (600, 257, 256, 65)),     # 64-row passes: ten, five, four and two of them for four workgroups
    (600, 512, 96, 2, 384, (129, 128, 33, 32)),      # 32-row passes
    (65, 512, 8, 4, 384, (65, 64)),                  # two workgroups in down, the dispatch inside gate_up
])
def test_mid_rows(dev, T, H, E, K, I, crowd):
    from on_device_sd_amd import ops
    print("48-row streaming", T, H, E, K, I, crowd, flush=True)
    g = torch.Generator().manual_seed(T + H + E + K + I)
    wg = (torch.randn(E, H, generator=g) * 0.02).to(torch.bfloat16)
    x = torch.randn(T, H, generator=g).to(torch.bfloat16)
    # expert c is chosen by `crowd[c]` tokens: it alone looks at column c
    n = len(crowd)
    wg[:, :n] = 0.0
    at = 0
    for c, rows in enumerate(crowd):
        wg[c] = 0.0
        wg[c, c] = 1.0
        x[:, c] = -40.0
        x[(at + torch.arange(rows)) % T, c] = 40.0      # one after the other, round and round: at most K of them per token
        at += rows
    bank, experts = _bank(dev, H, E, I, g, distinct=3)
    xd, wgd, table = x.to(dev), wg.to(dev), bank.table()
    out = ops.moe_forward(xd, wgd, table, K, I, renorm=True)
    ref, idx, w = orc.moe_block(x, wg, experts, K, True)
    counts, offsets, perm, _ = orc.dispatch(idx, E)
    assert tuple(counts[:n]) == crowd
    assert np.array_equal(out.idx.cpu().numpy(), idx)
    assert np.array_equal(out.counts.cpu().numpy(), counts)
    # h and the sums are rounded to fp16 (2^-11): well inside the helper's 1e-2 of the largest and 2e-3 of the mean output
    check_output_relative(out.out_f32, ref)
    again = ops.moe_forward(xd, wgd, table, K, I, renorm=True)
    assert torch.equal(again.out_f32, out.out_f32)
    # one expert's weights missing
    gone = int(idx[0, 0])
    hole = table.clone()
    hole[gone] = 0
    got = ops.moe_forward(xd, wgd, hole, K, I, renorm=True)
    ref_hole = orc.moe_forward(x, idx, np.where(idx == gone, 0.0, w).astype(np.float32), experts)
    check_output_relative(got.out_f32, ref_hole)
