"""The combine of calls with many tokens (8 columns per thread) against the kernel of smaller calls, which an odd output address
and an fp32 output besides still get: the same bits, and the fp32 output within fp32 summation of the 64-bit sum."""
import pytest
import torch

pytestmark = pytest.mark.gpu


# rows of one chunk of 64 threads, of part of a chunk, of whole and of broken chunks of 256 threads; pairs fetched 1, 2, 4 and
# 8 together; the smallest T that takes the kernel.  fp32 activations: the kernel of smaller calls at any size
@pytest.mark.parametrize("H,K,dtype", [(128, 8, torch.bfloat16), (640, 3, torch.bfloat16), (1920, 6, torch.bfloat16),
                                       (2048, 8, torch.bfloat16), (2176, 4, torch.bfloat16), (4096, 16, torch.bfloat16),
                                       (640, 3, torch.float32), (2176, 4, torch.float32)])
@pytest.mark.parametrize("with_residual", [False, True])
def test_wide_combine_gives_the_same_bits(dev, H, K, dtype, with_residual):
    from on_device_sd_amd import ops
    print("combine", H, K, dtype, with_residual, flush=True)
    E, T = 16, max(-(-8000000 // (H * K)), -(-2000000 // H))
    P = T * K
    g = torch.Generator(device=dev).manual_seed(H + K)
    st = ops.ExpertStages(T, H, E, K, 128, dtype, dev)
    assert st.splits == 1
    y16 = st.y.view(torch.float16).view(-1)[: P * H].view(P, H)
    y16.normal_(generator=g)
    y16[: P // 7] *= 1e-6                                  # subnormal halves
    y16[5, 3], y16[6, 7] = float("inf"), float("nan")
    idx = torch.randint(0, E, (T, K), generator=g, device=dev, dtype=torch.int32)
    idx[0, 0], idx[1, K - 1] = -1, E                        # no expert: contributes nothing
    w = torch.rand(T, K, generator=g, device=dev)
    perm = torch.randperm(P, generator=g, device=dev).to(torch.int32)
    perm[9] = -1
    disp = ops.Dispatch(None, None, perm, None, None)
    table = torch.ones(E, 4, dtype=torch.int64, device=dev)
    table[3, 0] = 0                                        # not placed
    res = torch.randn(T, H, generator=g, device=dev).to(dtype) if with_residual else None

    def run(shift, f32=None):
        act = torch.zeros(T * H + 8, dtype=dtype, device=dev)[shift:shift + T * H].view(T, H)
        st.combine(idx, w, disp, table, residual=res, out_f32=f32, out_act=act)
        return act.contiguous().view(torch.int16 if dtype == torch.bfloat16 else torch.int32)

    f32 = torch.empty(T, H, device=dev)
    act = run(0)
    assert torch.equal(act, run(1)) and torch.equal(act, run(0, f32))
    # K multiply-adds and the residual's add, each rounded once
    ok = (idx >= 0) & (idx < E) & (perm.view(T, K) >= 0)
    ok &= table[:, 0][idx.clamp(0, E - 1).long()] != 0
    total, size = torch.zeros(T, H, dtype=torch.float64, device=dev), torch.zeros(T, H, dtype=torch.float64, device=dev)
    for k in range(K):
        v = y16[perm.view(T, K)[:, k].clamp(min=0).long()].double() * w[:, k:k + 1].double()
        v = torch.where(ok[:, k:k + 1], v, 0.0)
        total += v
        size += v.abs()
    if with_residual:
        total += res.double()
        size += res.double().abs()
    fin = total.isfinite()
    assert ((f32.double() - total).abs() <= (K + 1) * 2.0 ** -24 * size)[fin].all()
    assert not f32[~fin].isfinite().any() and f32[fin].isfinite().all()
