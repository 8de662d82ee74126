"""The workspace that an attention call asks for is the one that its launch uses (host side only, no GPU):
sizes around the bounds where the kernel form and the splitting of units change."""
import random

import pytest
import torch

from on_device_sd_amd import _lib

ERR_NULL, ERR_WORKSPACE, ERR_LAUNCH = 1, 5, 6
NOTHING = 256                                       # the answer where nothing is split


def _shapes():
    """(n_seqs, max_q, max_k, heads, kv_heads, head_dim): keys either side of 96 MB, and of the lengths below
    which units stay whole, none of them a multiple of 32."""
    out = []
    for heads, kvh, hd in ((32, 4, 128), (32, 8, 128), (16, 2, 128), (16, 8, 64), (12, 4, 64)):
        for n in (1, 3, 25, 50, 51, 100, 130, 200, 400):
            edge = (96 << 20) // (n * kvh * hd * 4)
            for k in {edge - 1, edge, edge + 1, (edge + 31) // 32 * 32 - 1, 257, 479, 481, 513, 983, 1025, 1966}:
                for q in (1, 2, 3, 4, 6, 9):
                    out.append((n, q, max(k, 1), heads, kvh, hd))
    return out


def test_packed_and_paged_calls_of_one_shape_ask_for_the_same():
    lib = _lib.load()
    for n, q, k, heads, kvh, hd in _shapes():
        packed = lib.odsd_varlen_attention_workspace_bytes(n, q, k, heads, kvh, hd)
        paged = lib.odsd_paged_attention_workspace_bytes(n, q, heads, kvh, hd, 1, k)
        assert packed == paged >= NOTHING, (n, q, k, heads, kvh, hd, packed, paged)


@pytest.mark.skipif(torch.cuda.is_available(), reason="passes addresses that are never read without a GPU")
def test_a_launch_takes_what_the_size_function_says_and_no_less():
    """Without a device every accepted call ends in ODSD_ERR_LAUNCH, after the workspace has been checked."""
    lib = _lib.load()
    at = 1 << 20                                    # an aligned address; nothing is launched, so nothing reads it

    def packed(shape, ws, nbytes):
        n, q, k, heads, kvh, hd = shape
        return lib.odsd_varlen_attention(at, at, at, at, at, n, q, k, heads, kvh, hd, 0.1, _lib.DT_BF16, at, ws, nbytes, None)

    def paged(shape, ws, nbytes):
        n, q, k, heads, kvh, hd = shape
        return lib.odsd_paged_attention(at, at, at, at, at, at, n, q, heads, kvh, hd, 1, k, k, 0.1, _lib.DT_BF16, at, ws, nbytes, None)

    split = whole = 0
    for shape in _shapes():
        n, q, k, heads, kvh, hd = shape
        if q * (heads // kvh) > 64:                 # the prefill kernel's: it takes no workspace
            continue
        need = lib.odsd_varlen_attention_workspace_bytes(n, q, k, heads, kvh, hd)
        for call in (packed, paged):
            assert call(shape, at, need) == ERR_LAUNCH, shape
            if need == NOTHING:
                assert call(shape, None, 0) == ERR_LAUNCH, shape
                whole += 1
            elif k > 480 and n * kvh < 512:         # (fewer keys or more units can do without)
                assert call(shape, None, 0) == ERR_NULL, shape
                assert call(shape, at, need - 1) == ERR_WORKSPACE, shape
                split += 1
    assert split > 100 and whole > 100


def test_a_list_of_shares_fits_32_bits():
    """A launch that would have to lay out more than 2^30 steps of 32 keys keeps its units whole."""
    size = _lib.load().odsd_paged_attention_workspace_bytes
    for n, q, blocks, split in ((256, 4096, 256, True), (256, 4096, 257, False), (256, 4096, 512, False), (1, 65535, 8193, False)):
        steps = n * 4 * ((q * 8 + 63) // 64) * (blocks * 256 // 32)
        assert (steps <= 1 << 30) == split
        assert (size(n, q, 32, 4, 128, 256, blocks) > NOTHING) == split, (n, q, blocks)


def test_the_workspace_holds_every_share_and_little_more():
    """Two slots of partial results for each workgroup that gets a share: the list restated for random lengths
    within the bounds (steps of 128 keys up to 32 query rows; above, of 32 keys when every workgroup gets 256
    that way, else of 256; 512 workgroups)."""
    size = _lib.load().odsd_paged_attention_workspace_bytes
    rng = random.Random(1)
    for n, q, heads, kvh, hd, keys in ((1, 8, 32, 4, 128, 4096), (1, 1, 32, 4, 128, 4000), (3, 5, 16, 2, 128, 1500),
                                       (32, 8, 32, 4, 128, 2048), (2, 30, 8, 1, 64, 3000), (7, 1, 8, 8, 64, 700)):
        group = heads // kvh
        rows = 16 if q * group <= 16 else 64
        slot = rows * (hd + 4) * 4
        slots = size(n, q, heads, kvh, hd, 1, keys) / slot
        fine, coarse = (128, 128) if rows == 16 else (32, 256)

        def shares(lens, qs):
            units = [kvh * -(-t * group // rows) for t in qs]
            steps = lambda g: sum(u * max(1, -(-L // g)) for u, L in zip(units, lens))
            total = steps(fine) if steps(fine) >= coarse // fine * 512 else steps(coarse)
            share = max(1, -(-total // 512))
            return -(-total // share)

        assert 2 * shares([keys] * n, [q] * n) <= slots <= 1025
        for _ in range(300):
            assert 2 * shares([rng.randint(0, keys) for _ in range(n)], [rng.randint(0, q) for _ in range(n)]) <= slots
    assert size(1, 8, 32, 4, 128, 256, 16) == 2 * 64 * 64 * 132 * 4          # one sequence of 4096 keys: 64 shares, 4.3 MB
    assert size(32, 8, 32, 4, 128, 256, 8) == 2 * 512 * 64 * 132 * 4
