"""The tile kernel, and the streaming kernel's 128-row passes that stand in for it where a call has few pieces of
weights, through the stage calls with row counts that the caller sets: the edges of 16- and 32-row blocks and
128-row passes, odd and single groups in the reduction, a weight matrix that ends inside a tile, a down
reduction split over workgroups and passes shared by workgroups."""
import numpy as np
import pytest
import torch

from tests.helpers import canon_to_oracle

pytestmark = pytest.mark.gpu

COUNTS = {
    "blocks": [1, 31, 32, 33, 64, 65, 96, 97, 128, 0, 129, 160, 257, 385],
    # up to 104 rows per expert on average (and "lone"): the streaming kernel's passes
    "stream_blocks": [1, 15, 16, 17, 31, 33, 64, 65, 96, 112, 113, 127, 128, 0, 129, 160, 257],
    "passes": [129, 255, 256, 300],
    "lone": [77],
    "hot": [700, 3, 1090, 0, 60, 1],       # up to nine passes of one expert, shared by four workgroups
}


@pytest.mark.parametrize("counts", list(COUNTS))
@pytest.mark.parametrize("H,I", [(256, 128), (384, 640), (640, 384), (512, 1024)])
def test_tile_kernel_rows(dev, counts, H, I):
    import on_device_sd_amd as odsd
    from on_device_sd_amd import ops
    print("tile kernel", counts, H, I, flush=True)
    n = COUNTS[counts]
    E, T = len(n), sum(n)
    g = torch.Generator().manual_seed(H + I + T)
    bank = odsd.W4ExpertBank(E, H, I, dev)
    mk = lambda r, c: torch.randn(r, c, generator=g) * 0.05 + 0.01  # noqa: E731
    experts = [canon_to_oracle(bank.load_expert(e, mk(I, H), mk(I, H), mk(H, I), keep_canonical=True)) for e in range(E)]
    ids = torch.repeat_interleave(torch.arange(E), torch.tensor(n))[torch.randperm(T, generator=g)]
    idx = ids.to(torch.int32).view(T, 1).to(dev)
    x = torch.randn(T, H, generator=g).to(torch.bfloat16)
    x16 = x.to(torch.float16).to(dev)
    disp = ops.dispatch(idx, E)
    assert disp.counts.cpu().tolist() == n
    st = ops.ExpertStages(T, H, E, 1, I, torch.bfloat16, dev)
    h = st.gate_up(x16, bank.table(), disp)
    y = st.down(bank.table(), disp).view(torch.float16).flatten()[: st.splits * T * H].view(st.splits, T, H)
    torch.cuda.synchronize()
    offs, slot_token = disp.offsets.cpu().numpy(), disp.slot_token.cpu().numpy()
    x32 = x.to(torch.float32)
    # weights are rounded to fp16 as they are expanded (relative 2^-11 at most, 2.4e-4 in the mean square) and
    # the results once more; sums are fp32: 5e-4 of the norm, and the bound has a factor of two over that
    for e in range(E):
        if n[e] == 0:
            continue
        rows = slice(int(offs[e]), int(offs[e + 1]))
        gw, uw, dw = experts[e].dequant()
        xe = x32[slot_token[rows]]
        ref = torch.nn.functional.silu(xe @ gw.T) * (xe @ uw.T)
        got = h[rows].cpu().to(torch.float32)
        assert torch.linalg.norm(got - ref) <= 1e-3 * torch.linalg.norm(ref), (e, n[e])
        assert (got - ref).norm(dim=1).max() <= 4e-3 * ref.norm(dim=1).mean(), (e, n[e])      # no single row off
        ref = got @ dw.T
        out = y[:, rows].cpu().to(torch.float32).sum(0)
        assert torch.linalg.norm(out - ref) <= 1e-3 * torch.linalg.norm(ref), (e, n[e])
        assert (out - ref).norm(dim=1).max() <= 4e-3 * ref.norm(dim=1).mean(), (e, n[e])
