"""The prefill attention kernel against the oracle at the edges of its tiles: 64 / 65 query rows, key
counts around a multiple of 64, head groups that do not divide a row block, both head sizes, launches
below and above the bound between its two forms, and calls that stay with the decode / verify kernel."""
import numpy as np
import pytest
import torch

from oracle import moe_oracle as orc

pytestmark = pytest.mark.gpu

CASES = [
    # dtype, H, KVH, HD, (q_len, k_len) per sequence
    (torch.bfloat16, 32, 4, 128, [(9, 9), (8, 8)]),                          # 72 rows: one full block and 8 rows
    (torch.bfloat16, 32, 4, 128, [(63, 63), (64, 64), (65, 65), (128, 129)]),
    (torch.float16, 12, 4, 128, [(100, 100), (43, 43), (1, 1)]),             # 3 heads per group: rows of a token split over blocks
    (torch.float16, 6, 1, 64, [(191, 191), (193, 320)]),                     # chunked: more keys than queries
    (torch.bfloat16, 2, 2, 64, [(300, 300), (65, 40), (70, 0)]),             # queries without a visible key: zeros
    (torch.bfloat16, 32, 8, 128, [(513, 513), (200, 200), (385, 385)]),      # 24 x 17 workgroups: the 128-row form
    (torch.float16, 16, 8, 64, [(1300, 1300), (64, 64)]),                    # the same, head size 64
    (torch.bfloat16, 16, 2, 128, [(10, 1500), (3, 700)]),                    # few rows on many keys: the other kernel
]


@pytest.mark.parametrize("dtype,H,KVH,HD,seqs", CASES)
def test_prefill_attention_vs_oracle(dev, dtype, H, KVH, HD, seqs):
    import on_device_sd_amd as odsd
    print("prefill attention", dtype, H, KVH, HD, seqs, flush=True)
    g = torch.Generator().manual_seed(H * 1000 + HD + len(seqs))
    cu_q = np.concatenate([[0], np.cumsum([a for a, _ in seqs])]).astype(np.int32)
    cu_k = np.concatenate([[0], np.cumsum([b for _, b in seqs])]).astype(np.int32)
    q = torch.randn(int(cu_q[-1]), H, HD, generator=g)
    q[::7] *= 6.0                                    # peaked rows: the reference point of the exponentials moves
    q = q.to(dtype)
    k = torch.randn(int(cu_k[-1]), KVH, HD, generator=g).to(dtype)
    v = torch.randn(int(cu_k[-1]), KVH, HD, generator=g).to(dtype)
    args = (q.to(dev), k.to(dev), v.to(dev), torch.from_numpy(cu_q).to(dev), torch.from_numpy(cu_k).to(dev),
            max(a for a, _ in seqs), max(b for _, b in seqs))
    out = odsd.varlen_attention(*args)
    ref = orc.varlen_attention(q, k, v, cu_q, cu_k, HD ** -0.5)
    err = (out.float().cpu() - ref).abs()
    # probabilities and output are rounded to the storage type: 2^-9 (bf16) or 2^-12 of values up to ~4
    tol = 2e-2 if dtype == torch.bfloat16 else 3e-3
    print(f"  max-abs error {err.max().item():.3e}", flush=True)
    assert err.max().item() <= tol
    assert torch.equal(out, odsd.varlen_attention(*args))
