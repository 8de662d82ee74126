"""Whole-block calls with at most 16 tokens at the edges of their plan: the number of pairs from which gate_up
goes through LDS and dispatches for itself (48), reductions of fewer groups than the pipeline is deep, the
shortest reductions on either side of the down projection's rule (3 and 4 groups), one and two weight blocks
per wavefront, split reductions, every token on the same experts."""
import numpy as np
import pytest
import torch

from oracle import moe_oracle as orc
from tests.helpers import canon_to_oracle, check_output_relative

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,H,E,K,I", [
    (16, 256, 16, 3, 128),      # 48 pairs: the first with the dispatch inside; one group in the down reduction
    (15, 256, 16, 3, 384),      # 45 pairs: the last without; 3 groups
    (16, 128, 3, 3, 512),       # a single group in the gate_up reduction, 16 rows on every expert; 4 groups
    (7, 640, 40, 7, 640),       # 49 pairs, 5 groups either way
    (16, 384, 24, 8, 896),      # 3 and 7 groups
    (16, 2048, 64, 8, 1024),    # equal shares: 4 parts of 2 groups in the down projection
    (16, 2176, 64, 8, 1024),    # two weight blocks per wavefront in the down projection
    (5, 1024, 8, 2, 4608),      # too many workgroups per expert to dispatch inside; split down reduction
    (1, 512, 64, 48, 512),      # one token with 48 pairs
])
def test_few_tokens(dev, T, H, E, K, I):
    import on_device_sd_amd as odsd
    from on_device_sd_amd import ops
    print("few tokens", T, H, E, K, I, flush=True)
    g = torch.Generator().manual_seed(T + H + E + K + I)
    wg = (torch.randn(E, H, generator=g) * 0.02).to(torch.bfloat16)
    bank = odsd.W4ExpertBank(E, H, I, dev)
    mk = lambda r, c: torch.randn(r, c, generator=g) * 0.05  # noqa: E731
    experts = {e: canon_to_oracle(bank.load_expert(e, mk(I, H), mk(I, H), mk(H, I), keep_canonical=True)) for e in range(E)}
    x = torch.randn(T, H, generator=g).to(torch.bfloat16)
    out = ops.moe_forward(x.to(dev), wg.to(dev), bank.table(), K, I, renorm=True)
    ref, idx, _ = orc.moe_block(x, wg, experts, K, True)
    assert np.array_equal(out.idx.cpu().numpy(), idx)
    counts, offsets, perm, _ = orc.dispatch(idx, E)
    assert np.array_equal(out.counts.cpu().numpy(), counts)
    assert np.array_equal(out.offsets.cpu().numpy(), offsets)
    assert np.array_equal(out.perm.cpu().numpy(), perm)
    # weights and h are rounded to fp16 once each (2^-11): the largest error stays within the helper's 1e-2 of the
    # largest output and the mean within its 2e-3 of the mean output
    check_output_relative(out.out_f32, ref)
