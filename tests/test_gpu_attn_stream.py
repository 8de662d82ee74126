"""The decode / verify attention kernels against the oracle where their division of the work can go wrong:
16 / 17, 32 / 33 and 64 / 65 query rows per KV head, contexts around the 32-key tiles, the 128-key turns and
the bounds below which nothing is split, pieces that begin and end inside a sequence, more than 64 sequences
(the list is laid out 64 at a time), sequences without queries or without keys, and table widths that choose
the two-row-block form."""
import numpy as np
import pytest
import torch

from oracle import moe_oracle as orc

pytestmark = pytest.mark.gpu


def _case(dev, dtype, H, KVH, HD, bs, seqs, pad_blocks=0, seed=0):
    """seqs: (context_len, q_len) per sequence; returns what the call needs and the oracle's answer."""
    g = torch.Generator().manual_seed(seed)
    nbs = [max(1, -(-L // bs)) for L, _ in seqs]
    perm = torch.randperm(sum(nbs) + 2, generator=g).tolist()
    tables, at = [], 0
    for nb in nbs:
        tables.append(perm[at:at + nb]); at += nb
    mb = max(nbs) + pad_blocks
    bt = torch.tensor([t + [-1] * (mb - len(t)) for t in tables], dtype=torch.int32)
    D = KVH * HD
    kc = torch.randn((sum(nbs) + 2) * bs, D, generator=g).to(dtype)
    vc = torch.randn((sum(nbs) + 2) * bs, D, generator=g).to(dtype)
    qls = [q for _, q in seqs]
    q = torch.randn(sum(qls), H, HD, generator=g)
    q[::5] *= 5.0                                    # peaked rows: the reference point of the exponentials moves
    q = q.to(dtype)
    ref = orc.paged_attention(q, kc, vc, bt.tolist(), [L for L, _ in seqs], qls, KVH, bs, HD ** -0.5)
    ctx = {"block_tables": bt.to(dev), "context_lens": torch.tensor([L for L, _ in seqs], dtype=torch.int32, device=dev),
           "verify_query_lens": torch.tensor(qls, dtype=torch.int32, device=dev)}
    return q.to(dev), kc.to(dev), vc.to(dev), ctx, max(qls), ref


def _edges(lens, q):
    return [(max(L, q), q) for L in lens]


CASES = {
    # rows per KV head either side of the forms' bounds
    "rows16": (torch.bfloat16, 16, 1, 128, 32, _edges([600, 33, 1300], 1), 0),
    "rows17": (torch.bfloat16, 17, 1, 128, 32, _edges([600, 33, 1300], 1), 0),
    "rows33": (torch.float16, 11, 1, 64, 32, _edges([700, 5, 901], 3), 0),
    "rows64": (torch.bfloat16, 16, 2, 128, 64, _edges([257, 1024, 255, 700], 8), 0),
    "rows65": (torch.float16, 13, 1, 128, 16, _edges([900, 300], 5), 0),
    # contexts at the tiles' and turns' edges, everything whole / something split
    "whole512": (torch.bfloat16, 8, 2, 128, 32, _edges([1, 31, 32, 33, 127, 128, 129, 511, 512], 1), 0),
    "split513": (torch.bfloat16, 8, 2, 128, 32, _edges([1, 31, 32, 33, 127, 128, 129, 512, 513], 1), 0),
    "tile256": (torch.bfloat16, 16, 2, 128, 32, _edges([9, 31, 64, 65, 255, 256], 6), 0),
    "tile257": (torch.bfloat16, 16, 2, 128, 32, _edges([9, 31, 64, 65, 255, 257], 6), 0),
    # table entries of single keys (block sizes that are no multiple of 32)
    "block16": (torch.float16, 8, 2, 128, 16, _edges([1000, 17, 129, 640], 1), 0),
    "block3_hd64": (torch.bfloat16, 8, 4, 64, 3, _edges([800, 95, 1, 333], 2), 0),
    # many sequences: the list is scanned 64 at a time; shares that span several of them
    "seqs150": (torch.bfloat16, 4, 2, 64, 32, [(1 + (i * 37) % 900, 1) for i in range(150)], 0),
    "seqs70_tile": (torch.float16, 16, 1, 64, 32, [(8 + (i * 53) % 700, 1 + i % 5) for i in range(70)], 0),
    # 128 units and more with few keys, 2048 and more: nothing is split
    "some": (torch.bfloat16, 4, 4, 64, 32, [(1 + (i * 37) % 1000, 1) for i in range(33)], 0),
    "some_tile": (torch.bfloat16, 36, 4, 64, 32, [(9 + (i * 53) % 370, 2 + i % 5) for i in range(32)], 0),
    "many": (torch.bfloat16, 8, 8, 64, 32, [(1 + (i * 37) % 700, 1) for i in range(256)], 0),
    "many_tile": (torch.float16, 40, 8, 64, 32, [(7 + (i * 53) % 400, 1 + i % 7) for i in range(257)], 0),
    # unsplit with more keys than are looked up at a time (1024)
    "long_unsplit": (torch.bfloat16, 36, 4, 64, 32, [(1300 - i if i % 40 == 0 else 9 + (i * 53) % 200, 4 + i % 4) for i in range(128)], 0),
    # no keys, no queries, fewer keys than queries
    "holes": (torch.bfloat16, 8, 2, 128, 32, [(0, 2), (700, 1), (3, 4), (40, 0), (1200, 2), (0, 1)], 0),
    "holes_tile": (torch.bfloat16, 24, 1, 128, 32, [(0, 2), (700, 3), (40, 0), (2, 3), (1200, 2), (0, 1)], 0),
    # a table wide enough for 96 MB of keys: 17 to 32 rows in two row blocks
    "wide": (torch.bfloat16, 32, 8, 128, 64, _edges([1500, 300, 129, 77], 5), 256),
    "wide_block48": (torch.float16, 24, 8, 64, 48, _edges([1500, 300, 129, 77], 8), 800),
}


@pytest.mark.parametrize("name", list(CASES))
def test_paged_attention_shares(dev, name):
    import on_device_sd_amd as odsd
    dtype, H, KVH, HD, bs, seqs, pad = CASES[name]
    print("attention shares", name, flush=True)
    q, kc, vc, ctx, mq, ref = _case(dev, dtype, H, KVH, HD, bs, seqs, pad, seed=len(name))
    out = odsd.paged_attention(q, kc, vc, ctx, KVH, bs, max_q_len=mq)
    err = (out.float().cpu() - ref).abs()
    # probabilities and output are rounded to the storage type: 2^-9 (bf16) or 2^-12 of values up to ~4
    tol = 2e-2 if dtype == torch.bfloat16 else 3e-3
    print(f"  max-abs error {err.max().item():.3e}", flush=True)
    assert err.max().item() <= tol
    assert torch.equal(out, odsd.paged_attention(q, kc, vc, ctx, KVH, bs, max_q_len=mq))


@pytest.mark.parametrize("q_len,lens", [(1, [100, 64]), (1, [640, 640, 300]), (7, [640, 640, 300]), (8, [256, 90])])
def test_context_longer_than_its_table(dev, q_len, lens):
    """A context_len beyond the table's width: the positions past it read slot 0, as documented for entries
    beyond the cache, and the other sequences are what they are without it.  Tables below and above the lengths
    that keep units whole, both forms of the kernel; the list of shares is sized from the tables."""
    import on_device_sd_amd as odsd
    KVH, bs, HD, long = 2, 32, 128, 1500
    q, kc, vc, ctx, mq, _ = _case(dev, torch.bfloat16, 8 * KVH, KVH, HD, bs, _edges(lens, q_len))
    over = [long] + lens[1:]
    ctx["context_lens"] = torch.tensor(over, dtype=torch.int32, device=dev)
    print("context longer than its table", q_len, lens, flush=True)
    out = odsd.paged_attention(q, kc, vc, ctx, KVH, bs, max_q_len=mq).float().cpu()
    bt = ctx["block_tables"].cpu()
    slots = []
    for s, L in enumerate(over):
        pos = torch.arange(L)
        here = pos // bs < bt.shape[1]
        slots.append(torch.where(here, bt[s][(pos // bs).clamp(max=bt.shape[1] - 1)].long() * bs + pos % bs, 0))
    rows = torch.cat(slots)
    k, v = kc.cpu()[rows].view(-1, KVH, HD), vc.cpu()[rows].view(-1, KVH, HD)
    cu_q = np.arange(len(over) + 1, dtype=np.int32) * q_len
    cu_k = np.concatenate([[0], np.cumsum(over)]).astype(np.int32)
    ref = orc.varlen_attention(q.cpu(), k, v, cu_q, cu_k, HD ** -0.5)
    assert (out - ref).abs().max().item() <= 2e-2


@pytest.mark.parametrize("keys", [200, 1500])
def test_query_longer_than_its_bound(dev, keys):
    """A query length above max_q_len: its rows past the launch's row groups are not computed (documented), every
    other row is, of all KV heads and of the sequences after it."""
    import on_device_sd_amd as odsd
    KVH, bs = 3, 32
    for rows, mq in ((16, 2), (64, 8)):               # query rows per unit and max_q_len, 8 heads per KV head
        seqs = [(keys, mq), (keys, mq + 7), (keys - 30, mq), (keys, 1)]
        q, kc, vc, ctx, _, ref = _case(dev, torch.bfloat16, 8 * KVH, KVH, 64, bs, seqs)
        print("query longer than its bound", keys, rows, flush=True)
        out = odsd.paged_attention(q, kc, vc, ctx, KVH, bs, max_q_len=mq).float().cpu()
        sure = torch.ones(q.shape[0], dtype=torch.bool)
        sure[mq + rows // 8:2 * mq + 7] = False       # the long query's tokens past the first row group
        assert (out - ref)[sure].abs().max().item() <= 2e-2


@pytest.mark.parametrize("name,seqs", [("units512", [(1040 - (i * 37) % 1000, 1) for i in range(256)]),
                                       ("keys480", [(480, 9), (300, 9)])])
def test_calls_that_can_do_without_a_workspace(dev, name, seqs):
    """512 units, or at most 480 keys per sequence: a call without a workspace is carried out unsplit."""
    from on_device_sd_amd import _lib
    H, KVH, HD, bs = 8, 2, 64, 32
    q, kc, vc, ctx, mq, ref = _case(dev, torch.bfloat16, H, KVH, HD, bs, seqs)
    lib, bt, out = _lib.load(), ctx["block_tables"], torch.empty_like(q)
    assert lib.odsd_paged_attention_workspace_bytes(len(seqs), mq, H, KVH, HD, bs, bt.shape[1]) > 256
    print("attention without workspace", name, flush=True)
    rc = lib.odsd_paged_attention(q.data_ptr(), kc.data_ptr(), vc.data_ptr(), bt.data_ptr(), ctx["context_lens"].data_ptr(),
                                  ctx["verify_query_lens"].data_ptr(), len(seqs), mq, H, KVH, HD, bs, bt.shape[1],
                                  kc.shape[0], HD ** -0.5, _lib.DT_BF16, out.data_ptr(), None, 0, None)
    torch.cuda.synchronize()
    assert rc == 0
    assert (out.float().cpu() - ref).abs().max().item() <= 2e-2


# long queries: (heads, KV heads, head size, (context_len, q_len) per sequence); row groups of 64 rows see more keys one after
# the other, and their steps in the list follow
LONG = {
    "whole_sequences": (8, 1, 64, [(900, 900), (333, 333), (64, 64)]),
    "75_row_groups": (16, 2, 64, [(1500, 600), (700, 300), (1200, 1)]),
    "3_heads": (6, 2, 128, [(1100, 400), (600, 23)]),
    "more_queries_than_keys": (8, 1, 64, [(150, 400), (0, 70), (700, 500), (5, 130)]),
    "coarse": (16, 2, 128, [(2000, 12), (1000, 40)]),
    "unsplit": (16, 2, 64, [(250, 250), (100, 17), (256, 90)]),
}


@pytest.mark.parametrize("name", list(LONG))
def test_paged_attention_long_queries(dev, name):
    import on_device_sd_amd as odsd
    H, KVH, HD, seqs = LONG[name]
    print("attention, long queries", name, flush=True)
    q, kc, vc, ctx, mq, ref = _case(dev, torch.bfloat16, H, KVH, HD, 32, seqs, seed=len(name))
    out = odsd.paged_attention(q, kc, vc, ctx, KVH, 32, max_q_len=mq)
    # probabilities and output are rounded to bf16: 2^-9 of values up to ~4
    assert (out.float().cpu() - ref).abs().max().item() <= 2e-2
    again = odsd.paged_attention(q, kc, vc, ctx, KVH, 32)        # the default bound on the query lengths: all tokens
    assert (again.float().cpu() - ref).abs().max().item() <= 2e-2


def test_merge_with_a_loose_bound_on_the_queries(dev):
    """Split units under a bound that allows for 38 row groups each: the merge walks the bounds of the shares."""
    import on_device_sd_amd as odsd
    seqs = [(40 + (i * 397) % 1500, 1 + (i * 7) % 20) for i in range(16)] + [(0, 3), (1500, 0), (7, 9)]
    q, kc, vc, ctx, _, ref = _case(dev, torch.bfloat16, 16, 2, 64, 32, seqs, pad_blocks=160)
    print("merge, loose bound on the queries", flush=True)
    out = odsd.paged_attention(q, kc, vc, ctx, 2, 32, max_q_len=300)
    assert (out.float().cpu() - ref).abs().max().item() <= 2e-2
    assert torch.equal(out, odsd.paged_attention(q, kc, vc, ctx, 2, 32, max_q_len=300))


def test_more_units_than_workgroups(dev):
    """16896 units in one unsplit call: a workgroup takes two of them in turn."""
    import on_device_sd_amd as odsd
    n, H, KVH, HD, bs, q_len = 64, 64, 8, 64, 32, 264
    lens = [q_len + (i * 5) % 40 for i in range(n)]
    nbs = [-(-L // bs) for L in lens]
    first = np.concatenate([[0], np.cumsum(nbs)])
    bt = torch.full((n, max(nbs)), -1, dtype=torch.int32)
    for i in range(n):
        bt[i, :nbs[i]] = torch.arange(first[i], first[i + 1]).flip(0)
    g = torch.Generator(device=dev).manual_seed(7)
    mk = lambda *s: torch.randn(*s, generator=g, device=dev).to(torch.bfloat16)
    q, kc, vc = mk(n * q_len, H, HD), mk(int(first[-1]) * bs, KVH * HD), mk(int(first[-1]) * bs, KVH * HD)
    ctx = {"block_tables": bt.to(dev), "context_lens": torch.tensor(lens, dtype=torch.int32, device=dev),
           "verify_query_lens": torch.full((n,), q_len, dtype=torch.int32, device=dev)}
    print("more units than workgroups", flush=True)
    out = odsd.paged_attention(q, kc, vc, ctx, KVH, bs, max_q_len=q_len)
    kc, vc = kc.cpu(), vc.cpu()
    for s in (0, 31, 63):
        rows = slice(s * q_len, (s + 1) * q_len)
        ref = orc.paged_attention(q[rows].cpu(), kc, vc, [bt[s].tolist()], [lens[s]], [q_len], KVH, bs, HD ** -0.5)
        assert (out[rows].float().cpu() - ref).abs().max().item() <= 2e-2


@pytest.mark.parametrize("keys", [250, 700])
def test_rows_do_not_touch_keys_past_their_group(dev, keys):
    """A row group stops at the 32-key tile of its last visible key: an infinity in a later V row does not reach it
    as 0 x inf (unsplit, and in shares)."""
    import on_device_sd_amd as odsd
    q, kc, vc, ctx, mq, _ = _case(dev, torch.bfloat16, 8, 1, 64, 32, [(keys, keys)])
    bt = ctx["block_tables"].cpu()[0]
    last = keys // 32 * 32 + 1                        # a key of the last tile
    vc[int(bt[last // 32]) * 32 + last % 32] = float("inf")
    out = odsd.paged_attention(q, kc, vc, ctx, 1, 32, max_q_len=mq)
    print("infinity in V at key", last, flush=True)
    assert torch.isfinite(out[:keys // 32 * 32 - 8].float()).all()


# (q_len, k_len) per sequence; 8 heads per KV head
PACKED = {
    "stream_whole": (2, [(1, 300), (2, 64), (1, 512)]),
    "stream_split": (1, [(1, 1500), (2, 700), (0, 90), (1, 40), (2, 1100)]),
    "tile_whole": (2, [(7, 200), (8, 33), (5, 256)]),
    "tile_split": (1, [(7, 1500), (8, 700), (0, 90), (3, 40), (8, 1100)]),
    "prefill": (4, [(300, 300), (65, 129), (200, 200)]),
}


@pytest.mark.parametrize("name", list(PACKED))
def test_packed_offsets_that_do_not_begin_at_zero(dev, name):
    """Part of a batch's offsets: rows are the absolute ranges of cu_seqlens, in every kernel, and rows
    outside them are left alone."""
    import on_device_sd_amd as odsd
    from on_device_sd_amd import _lib
    KVH, seqs = PACKED[name]
    H, HD, q_first, k_first = 8 * KVH, 128, 13, 45
    g = torch.Generator().manual_seed(len(name))
    cu_q = np.concatenate([[0], np.cumsum([a for a, _ in seqs])]).astype(np.int32)
    cu_k = np.concatenate([[0], np.cumsum([b for _, b in seqs])]).astype(np.int32)
    nq, nk = int(cu_q[-1]), int(cu_k[-1])
    q = torch.randn(nq + 2 * q_first, H, HD, generator=g).to(torch.bfloat16)
    k = torch.randn(nk + 2 * k_first, KVH, HD, generator=g).to(torch.bfloat16)
    v = torch.randn(nk + 2 * k_first, KVH, HD, generator=g).to(torch.bfloat16)
    mq, mk = max(a for a, _ in seqs), max(b for _, b in seqs)
    lib = _lib.load()
    nbytes = lib.odsd_varlen_attention_workspace_bytes(len(seqs), mq, mk, H, KVH, HD)
    assert name == "prefill" or (nbytes > 256) == name.endswith("split")
    ws = torch.empty(nbytes, dtype=torch.uint8, device=dev)
    qd, kd, vd = q.to(dev), k.to(dev), v.to(dev)
    cq, ck = torch.from_numpy(cu_q + q_first).to(dev), torch.from_numpy(cu_k + k_first).to(dev)
    out = torch.full_like(qd, 77.0)
    print("packed attention, offsets from", q_first, k_first, name, flush=True)
    _lib.check(lib.odsd_varlen_attention(qd.data_ptr(), kd.data_ptr(), vd.data_ptr(), cq.data_ptr(), ck.data_ptr(), len(seqs), mq,
                                         mk, H, KVH, HD, HD ** -0.5, _lib.DT_BF16, out.data_ptr(), ws.data_ptr(), nbytes, None),
               "odsd_varlen_attention")
    torch.cuda.synchronize()
    ref = orc.varlen_attention(q[q_first:q_first + nq], k[k_first:k_first + nk], v[k_first:k_first + nk], cu_q, cu_k, HD ** -0.5)
    out = out.float().cpu()
    assert (out[q_first:q_first + nq] - ref).abs().max().item() <= 2e-2
    assert (out[:q_first] == 77.0).all() and (out[q_first + nq:] == 77.0).all()
    part = odsd.varlen_attention(qd, kd, vd, cq, ck, mq, mk).float().cpu()
    assert torch.equal(part[q_first:q_first + nq], out[q_first:q_first + nq])
