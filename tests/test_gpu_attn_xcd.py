"""The tile form's units and shares are dealt to the XCDs in groups: counts that leave a broken period or an uneven eighth, few
and many row groups, against the oracle."""
import pytest
import torch

from tests.test_gpu_attn_stream import _case

pytestmark = pytest.mark.gpu

# heads, KV heads, head size, (context_len, q_len) per sequence
CASES = {
    # unsplit, 2 and 3 row groups bounded, some sequences with fewer: 37 * 3 and 11 * 5 groups
    "2_row_groups": (24, 3, 64, [(16 + (i * 53) % 600, 1 + (i * 5) % 16) for i in range(37)]),
    "3_row_groups": (60, 5, 64, [(16 + (i * 53) % 250, 1 + (i * 7) % 16) for i in range(11)]),
    # fewer units than one period
    "one_broken_period": (48, 1, 128, [(200, 3), (130, 2)]),
    # unsplit through the list, 9 row groups: groups of 8
    "list_9_row_groups": (8, 1, 64, [(256 - i, 66 + i) for i in range(7)]),
    # split: from a few shares up to all
    "few_shares": (16, 1, 64, [(700, 8), (300, 5)]),
    "odd_shares": (32, 2, 64, [(1300, 8), (1000, 3), (900, 1), (777, 6)]),
    "all_shares": (16, 2, 64, [(1990 - 100 * i, 8) for i in range(16)]),
}


@pytest.mark.parametrize("name", list(CASES))
def test_units_and_shares_by_xcd(dev, name):
    import on_device_sd_amd as odsd
    H, KVH, HD, seqs = CASES[name]
    print("attention by XCD", name, flush=True)
    q, kc, vc, ctx, mq, ref = _case(dev, torch.bfloat16, H, KVH, HD, 32, seqs, seed=len(name))
    out = odsd.paged_attention(q, kc, vc, ctx, KVH, 32, max_q_len=mq)
    # probabilities and output are rounded to bf16: 2^-9 of values up to ~4
    assert (out.float().cpu() - ref).abs().max().item() <= 2e-2
