"""What the kernels that multiply the codes as they are lose against 64 bits: the roundings of h and of the expert outputs
to fp16 and nothing else of that size.

A value rounded to fp16 is off by up to 2^-11 of its mantissa's unit: 2^-10 / sqrt(12) in the mean square, divided by the
mantissa m.  With log m uniform over [1, 2) the mean of 1 / m^2 is 3 / (8 ln 2), so the relative error of a vector's 2-norm is
2^-10 / sqrt(12) * sqrt(3 / (8 ln 2)) = 2.07e-4.  h brings that once into the outputs, fp16 outputs once more: 2.07e-4 with
fp32 sums, 2.93e-4 with fp16 ones.  Weights rounded to fp16 one by one would add 2.07e-4 in each of the three products
(4.7e-4 in all); the bound of 1.15 times the expectation leaves no room for that.

Token rows of one sign add what fp32 loses of the offsets: with E x^2 = 1 the accumulator of a group of 128 columns starts at
(1024 + 64) / 2 * 128 * 0.8 = 5.6e4, where fp32's step is 2^-8, and takes four products: 2 * 2^-8 / sqrt(12) = 2.3e-3 in
the mean square, against 2.7 * sqrt(128) = 31 of the group's own sum (codes spread by 15 / 5.5 = 2.7 about the zero point):
7.3e-5 in gate and in up each."""
import pytest
import torch

from tests.helpers import canon_to_oracle

pytestmark = pytest.mark.gpu

OFFSETS = 2 * 2.0 ** -8 / 12 ** 0.5 / (2.7 * 128 ** 0.5)
ONE = 2.0 ** -10 / 12 ** 0.5 * (3 / (8 * 0.6931471805599453)) ** 0.5


@pytest.mark.parametrize("T,H,E,K,I,roundings", [
    (24, 2048, 16, 2, 768, 2),       # equal shares: 2 groups per part in gate_up, 3 in down
    (24, 3072, 16, 2, 1024, 2),      # 3 groups per part in gate_up, 2 in down
    (16, 4096, 16, 2, 2048, 1),      # one fp32 slice
    (5, 4096, 8, 2, 4096, 1),        # two fp32 slices, the top-k inside
    (40, 2048, 16, 2, 4608, 2),      # three fp16 slices: three roundings of a third of the sum's square each
    (160, 2048, 128, 8, 768, 2),     # the one-launch kernel
    (600, 4096, 40, 2, 256, 2),      # the 48-row kernel
])
@pytest.mark.parametrize("one_sign", [False, True])
def test_error_against_64_bits(dev, T, H, E, K, I, roundings, one_sign):
    import on_device_sd_amd as odsd
    from on_device_sd_amd import ops
    print("error against 64 bits", T, H, E, K, I, one_sign, flush=True)
    g = torch.Generator().manual_seed(T + H + I)
    bank = odsd.W4ExpertBank(E, H, I, dev)
    ws = [(torch.randn(I, H, generator=g) * 0.02, torch.randn(I, H, generator=g) * 0.02, torch.randn(H, I, generator=g) * 0.02)
          for _ in range(3)]
    deq = []
    for e in range(E):
        canon = bank.load_expert(e, *ws[e % 3], keep_canonical=e < 3)
        if e < 3:
            deq.append([w.to(dev).double() for w in canon_to_oracle(canon).dequant()])
    wg = (torch.randn(E, H, generator=g) * 0.02).to(torch.bfloat16)
    x = torch.randn(T, H, generator=g)
    x = (x.abs() if one_sign else x).to(torch.bfloat16).to(dev)      # (rows of one sign: the largest sums of offsets)
    out = ops.moe_forward(x, wg.to(dev), bank.table(), K, I, renorm=True)
    ref = torch.zeros(T, H, dtype=torch.float64, device=dev)
    for d in range(3):
        t, k = (out.idx % 3 == d).nonzero(as_tuple=True)
        gate, up, down = deq[d]
        xe = x[t].double()
        h = torch.nn.functional.silu(xe @ gate.T) * (xe @ up.T)
        ref.index_add_(0, t, (h @ down.T) * out.w[t, k].double()[:, None])
    rel = ((out.out_f32.double() - ref).norm() / ref.norm()).item()
    expected = (roundings * ONE ** 2 + (2 * OFFSETS ** 2 if one_sign else 0.0)) ** 0.5
    print(f"  {rel:.3e}, expected {expected:.3e}", flush=True)
    assert rel <= 1.15 * expected
