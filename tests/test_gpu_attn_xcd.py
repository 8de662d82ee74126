"""The tile form's units and shares are dealt to the XCDs in groups: counts that leave a broken period or an uneven eighth, few
and many row groups, shares of one step and of many, against the oracle."""
import pytest
import torch

from tests.test_gpu_attn_stream import _case

pytestmark = pytest.mark.gpu

BF16, F16 = torch.bfloat16, torch.float16
# dtype, heads, KV heads, head size, (context_len, q_len) per sequence
UNSPLIT = {
    # 2 and 3 row groups bounded, some sequences with fewer: 37 * 3 and 11 * 5 groups
    "2_row_groups": (BF16, 24, 3, 64, [(16 + (i * 53) % 600, 1 + (i * 5) % 16) for i in range(37)]),
    "3_row_groups": (BF16, 60, 5, 64, [(16 + (i * 53) % 250, 1 + (i * 7) % 16) for i in range(11)]),
    # fewer units than one period
    "one_broken_period": (BF16, 48, 1, 128, [(200, 3), (130, 2)]),
    # through the list, 9 row groups, groups of 8: one broken period; two whole ones and a broken one
    "list_9_row_groups": (BF16, 8, 1, 64, [(256 - i, 66 + i) for i in range(7)]),
    "list_135_units": (BF16, 8, 1, 64, [(256 - i, 66 + i % 7) for i in range(15)]),
    "list_hd128_f16": (F16, 8, 1, 128, [(256 - i, 66 + i % 7) for i in range(15)]),
}
SPLIT = {
    # shares of one step: a few, an odd number, 170
    "few_shares": (BF16, 16, 1, 64, [(700, 8), (300, 5)]),
    "odd_shares": (BF16, 32, 2, 64, [(1300, 8), (1000, 3), (900, 1), (777, 6)]),
    "shares_170": (BF16, 16, 2, 64, [(1990 - 100 * i, 8) for i in range(16)]),
    # shares of many steps, which begin and end inside units: one row group, two, three for some sequences
    "many_steps": (F16, 32, 8, 64, [(1990 - 61 * i, 7) for i in range(16)]),
    "many_steps_hd128": (BF16, 32, 4, 128, [(1990 - 31 * i, 8) for i in range(24)]),
    "many_steps_2_row_groups": (BF16, 64, 8, 128, [(1990 - 37 * i, 12) for i in range(8)]),
    "many_steps_mixed_row_groups": (F16, 64, 8, 128, [(1700 - 37 * i, 1 + (i * 11) % 20) for i in range(10)]),
}


def _units(H, KVH, seqs):
    return [KVH * -(-q * (H // KVH) // 64) for _, q in seqs]


def _share(H, KVH, seqs):
    """(steps per share, shares) of a split launch: steps of 32 keys when 512 workgroups get 8 each, otherwise of 256."""
    for g in (32, 256):
        total = sum(u * -(-L // g) for u, (L, _) in zip(_units(H, KVH, seqs), seqs))
        if total >= 8 * 512:
            break
    share = -(-total // 512)
    return share, -(-total // share)


def _check(dev, name, dtype, H, KVH, HD, seqs):
    import on_device_sd_amd as odsd
    print("attention by XCD", name, flush=True)
    q, kc, vc, ctx, mq, ref = _case(dev, dtype, H, KVH, HD, 32, seqs, seed=len(name))
    out = odsd.paged_attention(q, kc, vc, ctx, KVH, 32, max_q_len=mq)
    # probabilities and output are rounded to the storage type: 2^-9 (bf16) or 2^-11 of values up to ~4
    assert (out.float().cpu() - ref).abs().max().item() <= (2e-2 if dtype == BF16 else 5e-3)


@pytest.mark.parametrize("name", list(UNSPLIT))
def test_units_by_xcd(dev, name):
    _, H, KVH, _, seqs = UNSPLIT[name]
    if name.startswith("list_"):                          # (the units of the list, row groups by their largest number)
        rg = max(_units(H, KVH, seqs)) // KVH
        assert rg >= 8 and (len(seqs) * KVH * rg >= 64) == (name != "list_9_row_groups")
    _check(dev, name, *UNSPLIT[name])


@pytest.mark.parametrize("name", list(SPLIT))
def test_shares_by_xcd(dev, name):
    _, H, KVH, _, seqs = SPLIT[name]
    share, used = _share(H, KVH, seqs)
    if name.startswith("many_steps"):
        assert share > 4 and 448 < used < 512 and used % 8
    else:
        assert share == 1 and used < 512
    _check(dev, name, *SPLIT[name])
