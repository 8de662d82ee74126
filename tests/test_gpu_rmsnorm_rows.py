"""RMSNorm with the row in registers (up to 4096 columns, aligned) against the kernel that walks the row in chunks, which an
odd address still gets: the same bits, and both within a unit in the last place of the oracle."""
import pytest
import torch

from oracle import moe_oracle as orc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H", [4, 128, 1020, 1024, 1028, 2048, 2052, 4092, 4096, 4100])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_row_in_registers_gives_the_same_bits(dev, H, dtype):
    from on_device_sd_amd import ops
    print("rmsnorm rows", H, dtype, flush=True)
    g = torch.Generator().manual_seed(H)
    T = 5
    x = (torch.randn(T, H, generator=g) * 3).to(dtype)
    x[1] = 0.0
    x[2] *= 1e-18                                          # squares below fp32: the statistics are fp64
    w = (1 + 0.2 * torch.randn(H, generator=g)).to(dtype)
    got = ops.rmsnorm(x.to(dev), w.to(dev), 1e-6)
    buf = torch.empty(T * H + 1, dtype=dtype, device=dev)
    buf[1:].copy_(x.flatten().to(dev))
    shifted = ops.rmsnorm(buf[1:].view(T, H), w.to(dev), 1e-6)
    assert torch.equal(got, shifted)
    want = orc.rmsnorm(x, w, 1e-6)
    if dtype == torch.bfloat16:
        ulp = (got.cpu().view(torch.int16).int() - want.view(torch.int16).int()).abs()
        assert ulp.max() <= 1 and (ulp > 0).float().mean() < 1e-2
    else:
        torch.testing.assert_close(got.cpu(), want, rtol=4e-7, atol=0)
