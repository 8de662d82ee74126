"""Quantise-on-load in one launch against the quantise and pack calls (which the stage tests hold to the
oracle): the same bytes, for every mixture of weight dtypes and for weights at unaligned addresses."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,I", [(128, 128), (384, 128), (128, 640), (2048, 768)])
@pytest.mark.parametrize("dtypes", [(torch.bfloat16,) * 3, (torch.float32,) * 3, (torch.bfloat16, torch.float32, torch.bfloat16)])
def test_one_launch_load_equals_quantize_and_pack(dev, H, I, dtypes):
    import on_device_sd_amd as odsd
    print("load expert", H, I, dtypes, flush=True)
    g = torch.Generator().manual_seed(H + I)
    ws = [(torch.randn(*s, generator=g) * 0.02) for s in ((I, H), (I, H), (H, I))]
    ws[0][3, :128] = 0.25                              # constant group: scale guard
    ws[1][5, :128] = ws[1][5, :128].abs() + 0.5        # all-positive group: negative zero point
    ws[2][7, :128] *= 1e6                              # scale beyond fp16's finest codes
    ws[2][9, 5] = float("inf")                         # scale and codes saturate
    ws[0][11, :] = -0.0
    ws[1][2, 3] = float("nan")
    for i in range(16, 128):                           # every order of magnitude of scale and zero point
        ws[i % 3][i] = ws[i % 3][i] * 10.0 ** ((i % 23) - 14) + (i % 5) * 0.3
    ws = [w.to(dt).to(dev) for w, dt in zip(ws, dtypes)]
    ref = odsd.W4ExpertBank(3, H, I, dev)
    got = odsd.W4ExpertBank(3, H, I, dev)
    ref.load_expert(1, *ws, keep_canonical=True)
    assert got.load_expert(1, *ws) is None and got.loaded == [False, True, False] and got.generation[1] == 1
    for name in ("gu_q", "gu_sz", "dn_q", "dn_sz"):    # the neighbouring slots stay untouched as well
        assert torch.equal(getattr(ref, name), getattr(got, name)), name
    # rows of a larger, oddly offset buffer
    shifted = []
    for w in ws:
        buf = torch.empty(w.numel() + 3, dtype=w.dtype, device=dev)
        buf[3:].copy_(w.flatten())
        shifted.append(buf[3:].view(w.shape))
    got.load_expert(2, *shifted)
    assert torch.equal(got.gu_q[2], ref.gu_q[1]) and torch.equal(got.dn_q[2], ref.dn_q[1])
    assert torch.equal(got.gu_sz[2], ref.gu_sz[1]) and torch.equal(got.dn_sz[2], ref.dn_sz[1])
    with pytest.raises(ValueError):
        got.load_expert(0, ws[2].t().contiguous()[:, :-1], ws[1], ws[2])
