// Weighted combine of calls with many tokens: out[t] = sum_k w[t,k] * y[perm[t*K+k]] in k order, fp32, one rounding (the indexed
// "+=" of demo/src/model/qwen3_runner.py:363, with the residual add of :226).
#include "common.h"

// Many tokens, complete fp16 sums, bf16 output: 8 columns per thread, so that a row of a pair is a load of 16 bytes per lane, the
// rows of up to 8 pairs on their way together, read past the caches that a layer's sums would only sweep.  Bound by HBM
// (T = 4096, H = 4096, K = 8: 60 -> 50 us for 336 MB).  The sums are those of combine_kernel, bit for bit.  In a file of its own: the code of
// the expert kernels behind it in experts.hip moved and ran up to 5 % slower (w4_gemm_kernel at T = 600, H = 2048: 56.1 -> 58.9 us).
template <int KB>
__global__ __launch_bounds__(256) void combine_wide_kernel(const half_t *__restrict__ y, const int32_t *__restrict__ idx,
                                                           const float *__restrict__ w, const int32_t *__restrict__ perm,
                                                           const uint64_t *__restrict__ table,
                                                           const uint16_t *__restrict__ residual,
                                                           uint16_t *__restrict__ out_act, int H, int K, int E, int nchunk) {
    const int t = blockIdx.x / nchunk, chunk = blockIdx.x - t * nchunk;
    const int c = (chunk * (int)blockDim.x + (int)threadIdx.x) * 8;
    if (c >= H) return;
    const size_t o = (size_t)t * H + c;
    float acc[8] = {}, res[8] = {};
    typedef uint16_t act8 __attribute__((ext_vector_type(8)));
    if (residual) {
        const act8 rv = *(const act8 *)(residual + o);
#pragma unroll
        for (int i = 0; i < 8; ++i) { const uint16_t e = rv[i]; res[i] = ActIO<uint16_t>::load(&e, 0); }
    }
    for (int k0 = 0; k0 < K; k0 += KB) {
        int slot[KB];
        float wk[KB];
        uint64_t tq[KB];
        bool ok[KB];
#pragma unroll
        for (int u = 0; u < KB; ++u) {                   // (as in combine_gather)
            const int pr = t * K + k0 + u, sl = perm[pr], e = idx[pr];
            wk[u] = w[pr];
            ok[u] = sl >= 0 && e >= 0 && e < E;
            tq[u] = table[(size_t)(ok[u] ? e : 0) * ODSD_TABLE_COLS];
            slot[u] = ok[u] ? sl : 0;
        }
        half8_t v[KB];
#pragma unroll
        for (int u = 0; u < KB; ++u) v[u] = __builtin_nontemporal_load((const half8_t *)(y + (size_t)slot[u] * H + c));
#pragma unroll
        for (int u = 0; u < KB; ++u)
            if (ok[u] && tq[u] != 0) {
#pragma unroll
                for (int i = 0; i < 8; ++i) acc[i] = fmaf(wk[u], (float)v[u][i], acc[i]);
            }
    }
    act8 st;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const float m = ActIO<uint16_t>::round(acc[i]);
        uint16_t e;
        ActIO<uint16_t>::store(&e, 0, residual ? __fadd_rn(res[i], m) : m);
        st[i] = e;
    }
    *(act8 *)(out_act + o) = st;
}

void odsd_launch_combine_wide(const odsd_moe_shape *s, const half_t *y, const int32_t *idx, const float *w, const int32_t *perm,
                              const uint64_t *table, const void *residual, void *out_act, hipStream_t st) {
    const int threads = s->H >= 2048 ? 256 : (s->H / 8 + 63) / 64 * 64, nchunk = (s->H / 8 + threads - 1) / threads;
#define COMBINE_WIDE(KB)                                                                                                      \
    ODSD_LAUNCH(ODSD_KERNEL_COMBINE, combine_wide_kernel<KB>, dim3((unsigned)(nchunk * s->T)), threads, st, y, idx, w, perm,   \
                table, (const uint16_t *)residual, (uint16_t *)out_act, s->H, s->K, s->E, nchunk)
    if (s->K % 8 == 0) COMBINE_WIDE(8);
    else if (s->K % 4 == 0) COMBINE_WIDE(4);
    else if (s->K % 2 == 0) COMBINE_WIDE(2);
    else COMBINE_WIDE(1);
#undef COMBINE_WIDE
}
