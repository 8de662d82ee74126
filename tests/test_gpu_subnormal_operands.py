"""Token rows, and rows of h = SiLU(gate) * up, that lie in fp16's subnormal range (below 2^-14).  The kernels that multiply
the codes as they are carry 1024 x and 64 x in their products and take them out again with sums of x formed by another
instruction: right only if both treat a subnormal alike.  One that takes it for zero would leave 1024 x where the true
term is at most 15 x."""
import pytest
import torch

from oracle import moe_oracle as orc
from tests.helpers import canon_to_oracle, check_output_relative

pytestmark = pytest.mark.gpu

SHAPES = [
    (24, 2048, 16, 2, 768),        # equal shares; down in two parts of three groups
    (5, 4096, 8, 2, 2048),         # equal shares with the top-k inside; down in eight parts of two groups
    (160, 2048, 128, 8, 768),      # the one-launch kernel
    (600, 4096, 40, 2, 256),       # the 48-row kernel (1200 pairs: more than the streaming kernel dispatches for itself)
]


def _run(dev, T, H, E, K, I, x, w_up, w_down, g):
    import on_device_sd_amd as odsd
    from on_device_sd_amd import ops
    bank = odsd.W4ExpertBank(E, H, I, dev)
    ws = [(torch.randn(I, H, generator=g) * w_up, torch.randn(I, H, generator=g) * w_up, torch.randn(H, I, generator=g) * w_down)
          for _ in range(3)]
    experts = {}
    for e in range(E):
        keep = e < 3
        canon = bank.load_expert(e, *ws[e % 3], keep_canonical=keep)
        experts[e] = canon_to_oracle(canon) if keep else experts[e % 3]
    wg = (torch.randn(E, H, generator=g) * 0.02).to(torch.bfloat16)
    out = ops.moe_forward(x.to(dev), wg.to(dev), bank.table(), K, I, renorm=True)
    ref, idx, w = orc.moe_block(x, wg, experts, K, True)
    assert (out.idx.cpu().numpy() == idx).all()
    return out.out_f32, ref, idx, w, experts


@pytest.mark.parametrize("T,H,E,K,I", SHAPES)
def test_subnormal_token_rows(dev, T, H, E, K, I):
    print("subnormal token rows", T, H, E, K, I, flush=True)
    g = torch.Generator().manual_seed(T + H + E)
    # multiples of fp16's smallest step with 7 bits: exact in bf16 and in fp16, and 2^-17.2 at most
    x = (torch.randint(-127, 128, (T, H), generator=g).float() * 2.0 ** -24).to(torch.bfloat16)
    assert x.float().abs().max() < 2.0 ** -14 and (x.float().to(torch.float16).float() == x.float()).all()
    got, ref, *_ = _run(dev, T, H, E, K, I, x, 2000.0, 0.02, g)
    check_output_relative(got, ref)        # x is exact: the helper's bounds for rows of ordinary size


@pytest.mark.parametrize("T,H,E,K,I", SHAPES)
def test_subnormal_intermediate(dev, T, H, E, K, I):
    print("subnormal intermediate", T, H, E, K, I, flush=True)
    g = torch.Generator().manual_seed(T + H + I)
    x = (torch.randn(T, H, generator=g) * 0.01).to(torch.bfloat16)
    w_up = 0.45 / H ** 0.5                 # gate and up of about 4.5e-3, h of about 1e-5
    got, ref, idx, w, experts = _run(dev, T, H, E, K, I, x, w_up, 0.02, g)
    deq = lambda c: torch.from_numpy(orc.dequantize_w4(*c))  # noqa: E731
    e = experts[int(idx[0, 0])]
    gate, up = x[:1].float() @ deq(e.gate).T, x[:1].float() @ deq(e.up).T
    h = torch.nn.functional.silu(gate) * up
    assert (h.abs() < 2.0 ** -14).float().mean() > 0.95
    # h lies on steps of 2^-24: an error of 2^-24 / sqrt(12) on an h of about 1e-5, 0.17 %, on top of the ordinary 2e-3
    check_output_relative(got, ref, mean_rel=6e-3)
