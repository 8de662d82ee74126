// Router: logits = x . Wg^T accumulated in fp64, then softmax / top-k per token.
//
// Two kernels (for many bf16 tokens another pair with the same choices and weights: router_screen_kernel and
// router_topk_screened_kernel, below).
//  1. router_partial_kernel: a split-K [T,H]x[H,E] product on the fp64 matrix cores
//     (v_mfma_f64_16x16x4_f64).  One wavefront owns a tile of 16 tokens x (16*NE) experts
//     over one K slice and writes fp64 partial logits.  fp64 accumulation makes the logits
//     the exact dot product to ~1e-16, so the top-k choice does not depend on the
//     summation order -- which is what lets the expert indices be bit-exact against a CPU
//     restatement.  The tile with expert group 0 also writes the fp16 copy of x that the
//     expert kernels consume.
//  2. router_topk_kernel: one wavefront per token sums the partials in a fixed order,
//     selects the K largest logits (ties to the lower index) by K rounds of a wavefront
//     arg-max and computes the weights in fp32.
//
// Replaces: Qwen3MoEGate.forward (demo/src/layers/moe_layer.py:41-58), the stateless form
// (:210-216) and GPUOperators.router (demo/src/operators/gpu_operators.py:48-69).
#include "common.h"
#include "router_topk.h"
#include "w4_gemm.h"

#include <type_traits>

#define ROUTER_MAX_NE 4    // expert tiles (of 16) per wavefront
#define ROUTER_MAX_V 8     // most logits per lane in the top-k kernel -> E <= 512

// 8 consecutive activations of one row: the raw load and the conversion are separate so that
// the loads of the next chunk can be in flight while the current one is multiplied
template <typename XT> struct Row8;
template <> struct Row8<uint16_t> {  // 8 bf16 = 16 bytes
    typedef uint4_t Raw;
    __device__ static __forceinline__ Raw raw(const uint16_t *p) { return *(const uint4_t *)p; }
    __device__ static __forceinline__ void cvt(const Raw &u, float (&v)[8]) {
        const uint32_t w[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            v[2 * i] = __uint_as_float(w[i] << 16);
            v[2 * i + 1] = __uint_as_float(w[i] & 0xffff0000u);
        }
    }
};
template <> struct Row8<float> {
    struct Raw { float4_t a, b; };
    __device__ static __forceinline__ Raw raw(const float *p) {
        return Raw{*(const float4_t *)p, *(const float4_t *)(p + 4)};
    }
    __device__ static __forceinline__ void cvt(const Raw &u, float (&v)[8]) {
        v[0] = u.a.x; v[1] = u.a.y; v[2] = u.a.z; v[3] = u.a.w;
        v[4] = u.b.x; v[5] = u.b.y; v[6] = u.b.z; v[7] = u.b.w;
    }
};

// unit = (token tile, expert group, k split); 4 units (wavefronts) per workgroup.
// At thousands of tokens the fp64 matrix cores bound it (4.3 GFLOP at T = 4096, H = 4096, E = 128: 55 us at
// 78 TFLOP/s).  So the loop holds nothing but loads, conversions and products: no branch (NORMED is compiled, the
// fp16 copy has a loop of its own), no masking (rows past T or E are read from row 0 and their results not
// stored), and neighbouring products belong to two accumulators in turn (all four in turn need every row's
// load at the start of a chunk: 118 us where this takes 103).  With branches and masks in the loop, before / now,
// us: E = 128, H = 2048: T = 256 6.4 / 5.9, T = 512 10.7 / 9.4, T = 1000 17.6 / 16.3, T = 2200 41.8 / 37.7;
// H = 4096: T = 4096 113 / 103 (42 TFLOP/s, at the clock that the expert kernels in between leave).
template <typename XT, int NE, bool REDUCE4, bool NORMED>
__global__ __launch_bounds__(256) void router_partial_kernel(const XT *__restrict__ x,
                                                             const XT *__restrict__ wg,
                                                             double *__restrict__ partial,
                                                             half_t *__restrict__ x16, int T, int H,
                                                             int E, int S, int EG, int n_units,
                                                             const double *__restrict__ norm_ss,
                                                             const XT *__restrict__ norm_w, double eps) {
    const int unit = blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (unit >= n_units) return;
    const int lane = lane_id();
    const int r = lane & 15, kg = lane >> 4;
    const int s = unit % S;
    const int eg = (unit / S) % EG;
    const int tt = unit / (S * EG);
    const int Hs = H / S;
    const int k0 = s * Hs;
    const int t = tt * 16 + r;
    const bool t_ok = t < T;

    // Which (row, column) of the 16x16 result each of this lane's 4 accumulators holds is
    // read back from the matrix core itself: D = A.B with A[i][0]=i, B[0][j]=1 gives D=i,
    // and A[i][0]=1, B[0][j]=j gives D=j.
    int di[4], dj[4];
    {
        const double4_t z = {0.0, 0.0, 0.0, 0.0};
        const double a_i = kg == 0 ? (double)r : 0.0, one = kg == 0 ? 1.0 : 0.0;
        const double4_t pi = __builtin_amdgcn_mfma_f64_16x16x4f64(a_i, one, z, 0, 0, 0);
        const double4_t pj = __builtin_amdgcn_mfma_f64_16x16x4f64(one, a_i, z, 0, 0, 0);
        di[0] = (int)pi.x; di[1] = (int)pi.y; di[2] = (int)pi.z; di[3] = (int)pi.w;
        dj[0] = (int)pj.x; dj[1] = (int)pj.y; dj[2] = (int)pj.z; dj[3] = (int)pj.w;
    }

    double4_t acc[NE];
#pragma unroll
    for (int i = 0; i < NE; ++i) acc[i] = double4_t{0.0, 0.0, 0.0, 0.0};

    // fused RMSNorm (demo/src/layers/layernorm.py:21-27): the row statistic comes from the kernel
    // that produced x; the arithmetic per element is that of the stand-alone RMSNorm kernel
    double rstd = 1.0;
    if (NORMED) {
        const int nchunk = (H + 1023) / 1024;   // the statistic arrives as per-chunk sums
        double tot = 0.0;
        for (int c = 0; c < nchunk; ++c) tot += norm_ss[(size_t)(t_ok ? t : 0) * nchunk + c];
        rstd = 1.0 / sqrt(tot / (double)H + eps);
    }
    const XT *xrow = x + (size_t)(t_ok ? t : 0) * H;
    const XT *wrow[NE];
#pragma unroll
    for (int i = 0; i < NE; ++i) {
        const int e = (eg * NE + i) * 16 + r;
        wrow[i] = wg + (size_t)(e < E ? e : 0) * H;
    }

    // One chunk = 32 columns.  The raw loads of chunk c+1 are issued before chunk c is
    // converted and multiplied (two register sets used in turn), so that their latency hides
    // under the 8*NE fp64 MFMAs of the current chunk.
    typedef typename Row8<XT>::Raw Raw;
    struct Chunk {
        Raw x, n, w[NE];
    };
    auto fetch = [&](Chunk &ck, int c) {
        const int h = k0 + min(c, Hs - 32) + kg * 8;    // past the end: reload the last chunk
        ck.x = Row8<XT>::raw(xrow + h);
        if (NORMED) ck.n = Row8<XT>::raw(norm_w + h);
#pragma unroll
        for (int i = 0; i < NE; ++i) ck.w[i] = Row8<XT>::raw(wrow[i] + h);
    };
    auto consume = [&](auto copy_c, const Chunk &ck, int c) {
        float xa[8];
        Row8<XT>::cvt(ck.x, xa);
        if (NORMED) {
            float nw[8];
            Row8<XT>::cvt(ck.n, nw);
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const float xn = ActIO<XT>::round((float)((double)xa[j] * rstd));
                xa[j] = ActIO<XT>::round(__fmul_rn(xn, nw[j]));
            }
        }
        if (decltype(copy_c)::value) {
            half8_t o;
#pragma unroll
            for (int j = 0; j < 8; ++j) o[j] = f32_to_f16_sat(xa[j]);
            if (t_ok) *(half8_t *)(x16 + (size_t)t * H + k0 + c + kg * 8) = o;
        }
        // two accumulators in turn, so that the later rows' loads have until then to land
        constexpr int IB = NE > 1 ? 2 : 1;
#pragma unroll
        for (int i0 = 0; i0 < NE; i0 += IB) {
            float wa[IB][8];
#pragma unroll
            for (int i = 0; i < IB; ++i) Row8<XT>::cvt(ck.w[i0 + i], wa[i]);
#pragma unroll
            for (int j = 0; j < 8; ++j)
#pragma unroll
                for (int i = 0; i < IB; ++i)
                    acc[i0 + i] = __builtin_amdgcn_mfma_f64_16x16x4f64((double)xa[j], (double)wa[i][j], acc[i0 + i], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    auto reduce = [&](auto copy_c) {
        Chunk ca, cb;
        fetch(ca, 0);
        int c = 0;
        for (; c + 32 < Hs; c += 64) {
            fetch(cb, c + 32);
            consume(copy_c, ca, c);
            fetch(ca, c + 64);
            consume(copy_c, cb, c + 32);
        }
        if (c < Hs) consume(copy_c, ca, c);
    };
    if (x16 != nullptr && eg == 0) reduce(std::true_type{});
    else reduce(std::false_type{});

    // When the K slices come in fours, the 4 wavefronts of this workgroup hold 4 consecutive
    // slices of the same tile: add them through LDS in slice order and write one partial.
    int s_out = s, S_out = S;
    if (REDUCE4) {
        __shared__ double red[3][NE][4][64];
        const int wave = threadIdx.x >> 6;
        if (wave > 0) {
#pragma unroll
            for (int i = 0; i < NE; ++i) {
                red[wave - 1][i][0][lane] = acc[i].x;
                red[wave - 1][i][1][lane] = acc[i].y;
                red[wave - 1][i][2][lane] = acc[i].z;
                red[wave - 1][i][3][lane] = acc[i].w;
            }
        }
        __syncthreads();
        if (wave > 0) return;
#pragma unroll
        for (int w = 0; w < 3; ++w)
#pragma unroll
            for (int i = 0; i < NE; ++i) {
                acc[i].x += red[w][i][0][lane];
                acc[i].y += red[w][i][1][lane];
                acc[i].z += red[w][i][2][lane];
                acc[i].w += red[w][i][3][lane];
            }
        s_out = s >> 2;
        S_out = S >> 2;
    }
    (void)S_out;
#pragma unroll
    for (int i = 0; i < NE; ++i) {
        const double v[4] = {acc[i].x, acc[i].y, acc[i].z, acc[i].w};
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int tq = tt * 16 + di[q];
            const int eq = (eg * NE + i) * 16 + dj[q];
            if (tq < T && eq < E) partial[((size_t)s_out * T + tq) * E + eq] = v[q];
        }
    }
}

template <int V>
__global__ __launch_bounds__(256) void router_topk_kernel(const double *__restrict__ partial, int T, int E,
                                                          int K, int S, int renorm,
                                                          int32_t *__restrict__ idx,
                                                          float *__restrict__ w,
                                                          int64_t *__restrict__ idx64,
                                                          double *__restrict__ logits) {
    const int t = blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
    if (t >= T) return;
    topk_token<V>(partial, t, T, E, K, S, renorm, idx, w, idx64, logits);
}

// -----------------------------------------------------------------------------------------
// Many tokens, bf16: the logits on the bf16 matrix cores, and in fp64 only the winners' and those that the choice hangs on.
//
// v_mfma_f32_16x16x32_bf16 multiplies exactly and runs 30 times as fast as the fp64 product.  Two products of 32
// columns, each from zero, are added in fp32, and everything above them in fp64, so a logit is off by at most
//     SCREEN_ERR * |x| * |w|,  SCREEN_ERR = 35 * 2^-23
// (32 additions of a product and the one of two products, each off by no more than a unit in the last place of the
// sum of the magnitudes so far -- whatever order the matrix core adds in, and whether it rounds or truncates -- then
// Cauchy-Schwarz; the norms' own rounding and flushed subnormals are in the remaining 6 %).  The top-k kernel takes
// neighbours in the order that are further apart than twice this bound as they are, and computes the others anew in
// fp64: the indices are those of the exact logits.  On N(0, 1) tokens that is one token in thirty, two or three dot products
// each.  The winners' logits are computed anew in any case, for the weights; those of a softmax over all experts
// (renorm = 0) hang on all logits, and such calls take the fp64 kernels.
//
// A workgroup of 8 wavefronts owns 32 tokens x 128 experts over one K slice, 128 columns a step; a wavefront 64 of the
// experts and a quarter of the columns; the quarters meet in LDS.  Rows arrive by asynchronous copies two steps ahead,
// 256 bytes of a row together: fragments loaded straight into registers, 64 bytes of each of 16 rows 8 KB apart, took
// 32 us at T = 4096, H = 4096 where this takes 22.  The sums of two steps go to the fp64 accumulators together
// (conversion and addition are the larger part of the vector work).
// -----------------------------------------------------------------------------------------
#define SCREEN_NT 2
#define SCREEN_NE 4
#define SCREEN_EXPERTS (2 * 16 * SCREEN_NE)   // of a workgroup
#define SCREEN_ERR (35.0 / 8388608.0)
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));

// sum of squares of 8 bf16, and whether any of them is not zero
__device__ __forceinline__ float sumsq8(const uint4_t &u, float acc, uint32_t &bits) {
    float v[8];
    Row8<uint16_t>::cvt(u, v);
#pragma unroll
    for (int j = 0; j < 8; ++j) acc = __builtin_fmaf(v[j], v[j], acc);
    bits |= (u.x | u.y | u.z | u.w) & 0x7fff7fffu;
    return acc;
}
// what stands for a norm: 0 only for a row of zeros (squares may vanish where the row has not)
__device__ __forceinline__ float nonzero_sq(const float ss, const bool any) { return any ? fmaxf(ss, 1.17549435e-38f) : 0.0f; }

template <bool NORMED>
__global__ __launch_bounds__(512, 2) void router_screen_kernel(const uint16_t *__restrict__ x, const uint16_t *__restrict__ wg,
                                                            double *__restrict__ partial, float *__restrict__ xsq,
                                                            float *__restrict__ wsq, half_t *__restrict__ x16, int T,
                                                            int H, int E, int S, int EG,
                                                            const double *__restrict__ norm_ss,
                                                            const uint16_t *__restrict__ norm_w, double eps) {
    constexpr int XB = 16 * SCREEN_NT * 256, BUF = XB + SCREEN_EXPERTS * 256, N_DMA = BUF / 8192;
    constexpr int NTILE = SCREEN_NT * SCREEN_NE;
    __shared__ __attribute__((aligned(16))) char rows[3 * BUF];   // token rows, then expert rows, of 128 columns
    __shared__ float red_ss[4][16 * SCREEN_NT], red_w[8];
    static_assert(8 * N_DMA * 1024 == BUF && 4 * 2 * (NTILE - NTILE / 4) * 2048 <= 3 * BUF, "whole copies; partial sums take the rows' place");
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = lane_id();
    const int unit = blockIdx.x;
    const int s = unit % S, eg = (unit / S) % EG, tt = unit / (S * EG);
    const int Hs = H / S, k0 = s * Hs, ng = Hs / ODSD_GROUP;
    const int r = lane & 15, kg = lane >> 4;
    const int eh = wave & 1, q = wave >> 1;              // the wavefront's 64 experts and its 32 of the 128 columns
    // copies: 4 rows x 256 B each, 16-byte segments XORed with the row as in the expert kernels
    uint32_t off[N_DMA];
#pragma unroll
    for (int i = 0; i < N_DMA; ++i) {
        const int row = (wave * N_DMA + i) * 4 + kg;     // token rows first
        const int t = tt * 16 * SCREEN_NT + row, e = eg * SCREEN_EXPERTS + row - 16 * SCREEN_NT;
        const int src = row < 16 * SCREEN_NT ? (t < T ? t : 0) : (e < E ? e : 0);
        off[i] = ((uint32_t)src * (uint32_t)H + (uint32_t)(k0 + ((r ^ (row & 15)) * 8))) * 2u;
    }
    auto dma = [&](const int buf, const int g) {
        const global_char *xb = (const global_char *)x + (size_t)g * (2 * ODSD_GROUP), *wb = (const global_char *)wg + (size_t)g * (2 * ODSD_GROUP);
#pragma unroll
        for (int i = 0; i < N_DMA; ++i) {
            const int piece = wave * N_DMA + i;
            dma16_to_lds(piece < 4 * SCREEN_NT ? xb : wb, off[i], (lds_void *)(rows + buf * BUF + piece * 1024));
        }
    };
    int t_of[SCREEN_NT];
    double rstd[SCREEN_NT];
#pragma unroll
    for (int i = 0; i < SCREEN_NT; ++i) {
        const int t = (tt * SCREEN_NT + i) * 16 + r;
        t_of[i] = t < T ? t : -1;
        rstd[i] = 1.0;
        if (NORMED) {                                    // as in router_partial_kernel
            const int nchunk = (H + 1023) / 1024;
            double tot = 0.0;
            for (int c = 0; c < nchunk; ++c) tot += norm_ss[(size_t)(t < T ? t : 0) * nchunk + c];
            rstd[i] = 1.0 / sqrt(tot / (double)H + eps);
        }
    }
    double4_t acc[NTILE];
#pragma unroll
    for (int m = 0; m < NTILE; ++m) acc[m] = double4_t{0.0, 0.0, 0.0, 0.0};
    float ss[SCREEN_NT] = {};
    uint32_t bits[SCREEN_NT] = {};
    const uint32_t frag = (uint32_t)((r * 16 + ((4 * q + kg) ^ r)) * 16);

    dma(0, 0);
    dma(1, 1);                                           // (ng >= 2, screen_slices)
    // the experts' norms, one expert a workgroup while the rows travel
    for (int e = unit; e < E; e += gridDim.x) {
        float sw = 0.f;
        uint32_t bw = 0;
        for (int h = (int)threadIdx.x * 8; h < H; h += 4096) sw = sumsq8(*(const uint4_t *)(wg + (size_t)e * H + h), sw, bw);
        sw = nonzero_sq(wave_sum(sw), __any(bw != 0));
        if (lane == 0) red_w[wave] = sw;
        __syncthreads();
        if (threadIdx.x == 0) {
            float tot = 0.f;
            for (int i = 0; i < 8; ++i) tot += red_w[i];
            wsq[e] = tot;
        }
        __syncthreads();
    }
    int buf = 0;
    float4_t pend[NTILE];
    // one group; the sums of two groups go to the fp64 accumulators together
    auto step = [&](const int g, const bool second) {
        // This group's rows have landed: loads land in order, and no more than the next group's are left (the stores of the copy only
        // make this stricter).  And this wavefront has the last step's fragments in registers: behind the barrier their buffer is
        // written again.
        if (g + 1 < ng) ODSD_WAIT_VMCNT_LGKM0(N_DMA);
        else ODSD_WAIT_VMCNT_LGKM0(0);
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        if (g + 2 < ng) dma(buf == 0 ? 2 : buf - 1, g + 2);      // what the step before this one read
        const char *base = rows + buf * BUF + frag;
        uint4_t xf[SCREEN_NT], wf[SCREEN_NE];
#pragma unroll
        for (int i = 0; i < SCREEN_NT; ++i) xf[i] = *(const uint4_t *)(base + i * 4096);
#pragma unroll
        for (int j = 0; j < SCREEN_NE; ++j) wf[j] = *(const uint4_t *)(base + XB + (eh * SCREEN_NE + j) * 4096);
        if (NORMED) {
            float nw[8];
            Row8<uint16_t>::cvt(*(const uint4_t *)(norm_w + k0 + g * ODSD_GROUP + 32 * q + 8 * kg), nw);
#pragma unroll
            for (int i = 0; i < SCREEN_NT; ++i) {
                float v[8];
                Row8<uint16_t>::cvt(xf[i], v);
                uint32_t o[4];
#pragma unroll
                for (int k = 0; k < 8; ++k) {
                    const float xn = ActIO<uint16_t>::round((float)((double)v[k] * rstd[i]));
                    const uint32_t b = f32_to_bf16(__fmul_rn(xn, nw[k]));
                    o[k >> 1] = (k & 1) ? o[k >> 1] | (b << 16) : b;
                }
                xf[i] = uint4_t{o[0], o[1], o[2], o[3]};
            }
        }
        const float4_t z = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int j = 0; j < SCREEN_NE; ++j)
#pragma unroll
            for (int i = 0; i < SCREEN_NT; ++i) {
                const int m = i * SCREEN_NE + j;
                const float4_t v = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, xf[i]),
                                                                          __builtin_bit_cast(bf16x8_t, wf[j]), z, 0, 0, 0);
                if (second) {
                    acc[m].x += (double)(pend[m].x + v.x);
                    acc[m].y += (double)(pend[m].y + v.y);
                    acc[m].z += (double)(pend[m].z + v.z);
                    acc[m].w += (double)(pend[m].w + v.w);
                } else {
                    pend[m] = v;
                }
            }
        // expert group 0: norms and the fp16 copy of x, token block i by the wavefronts of expert half i
        if (eg == 0) {
#pragma unroll
            for (int i = 0; i < SCREEN_NT; ++i) {
                if (i != eh) continue;
                ss[i] = sumsq8(xf[i], ss[i], bits[i]);
                if (x16 != nullptr && t_of[i] >= 0) {
                    float v[8];
                    Row8<uint16_t>::cvt(xf[i], v);
                    half8_t o;
#pragma unroll
                    for (int k = 0; k < 8; ++k) o[k] = f32_to_f16_sat(v[k]);
                    *(half8_t *)(x16 + (size_t)t_of[i] * H + k0 + g * ODSD_GROUP + 32 * q + 8 * kg) = o;
                }
            }
        }
        buf = buf == 2 ? 0 : buf + 1;
    };
    for (int g = 0; g < ng; g += 2) {
        step(g, false);
        if (g + 1 < ng) {
            step(g + 1, true);
        } else {
#pragma unroll
            for (int m = 0; m < NTILE; ++m) {
                acc[m].x += (double)pend[m].x;
                acc[m].y += (double)pend[m].y;
                acc[m].z += (double)pend[m].z;
                acc[m].w += (double)pend[m].w;
            }
        }
    }
    // The four quarters of the columns meet in LDS, in the rows' place: each wavefront leaves the tiles that it does not
    // finish, and finishes two.
    __syncthreads();
    double *red = (double *)rows;
    constexpr int OWN = NTILE / 4;
    auto slot = [&](const int from, const int m) {       // tile m of wavefront (from, eh): m without the tiles that `from` owns
        const int k = m < from * OWN ? m : m - OWN;
        return red + ((size_t)((from * 2 + eh) * (NTILE - OWN) + k) * 4) * 64 + lane;
    };
#pragma unroll
    for (int m = 0; m < NTILE; ++m) {
        if (m / OWN == q) continue;
        double *o = slot(q, m);
        o[0] = acc[m].x; o[64] = acc[m].y; o[128] = acc[m].z; o[192] = acc[m].w;
    }
    if (eg == 0) {
#pragma unroll
        for (int i = 0; i < SCREEN_NT; ++i) {
            if (i != eh) continue;
            ss[i] += __shfl_xor(ss[i], 16, 64);
            ss[i] += __shfl_xor(ss[i], 32, 64);
            bits[i] |= (uint32_t)__shfl_xor((int)bits[i], 16, 64);
            bits[i] |= (uint32_t)__shfl_xor((int)bits[i], 32, 64);
            if (kg == 0) red_ss[q][i * 16 + r] = nonzero_sq(ss[i], bits[i] != 0);
        }
    }
    __syncthreads();
    if (eg == 0 && wave == 0 && lane < 16 * SCREEN_NT) {
        const int t = tt * 16 * SCREEN_NT + lane;
        if (t < T) xsq[(size_t)s * T + t] = (red_ss[0][lane] + red_ss[1][lane]) + (red_ss[2][lane] + red_ss[3][lane]);
    }
#pragma unroll
    for (int m = 0; m < NTILE; ++m) {
        if (m / OWN != q) continue;
        double v[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int from = 0; from < 4; ++from) {
            const double *o = slot(from, m);
            if (from == q) {
                v[0] += acc[m].x; v[1] += acc[m].y; v[2] += acc[m].z; v[3] += acc[m].w;
            } else {
#pragma unroll
                for (int k = 0; k < 4; ++k) v[k] += o[64 * k];
            }
        }
        // lane: tokens 4 kg .. of the block, expert r
        const int e = eg * SCREEN_EXPERTS + (eh * SCREEN_NE + m % SCREEN_NE) * 16 + r;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const int t = (tt * SCREEN_NT + m / SCREEN_NE) * 16 + kg * 4 + k;
            if (t < T && e < E) partial[((size_t)s * T + t) * E + e] = v[k];
        }
    }
}

// One wavefront per token, as router_topk_kernel, on the logits of router_screen_kernel.  K < E and K < 64.
// The weights come from the winners' logits, so these are computed anew in fp64 with those that the order hangs on: the weights are
// those of the fp64 kernels, whatever the tokens look like.  (From the screened logits they would be off by what 64 columns'
// fp32 sum is: with a column of 300 that all experts share 1.2e-5 in the 2-norm where this has 5.1e-8.)  What is to be computed
// goes on a list of the token, and the wavefronts of the workgroup share all its tokens' lists, four or eight experts of one token
// at a time.  That reads T K rows of gate_w from L2: T = 4096, H = 4096, E = 128, K = 8, both kernels 60 us, 43 of it
// without the winners (2 experts at a time 63, 8 61, 4 with 1024 columns on their way 61, with 2048 68).
#define SCREENED_WAVES 4
#define SCREENED_MAX_K 16
template <int V, bool NORMED>
__global__ __launch_bounds__(64 * SCREENED_WAVES) void router_topk_screened_kernel(
    const double *__restrict__ partial, const float *__restrict__ xsq, const float *__restrict__ wsq,
    const uint16_t *__restrict__ x, const uint16_t *__restrict__ wg, int T, int H, int E, int K, int S,
    int32_t *__restrict__ idx, float *__restrict__ w, int64_t *__restrict__ idx64, const double *__restrict__ norm_ss,
    const uint16_t *__restrict__ norm_w, double eps) {
    constexpr int ROWS = NORMED ? 8 : 4;                 // (a group repeats the normalisation of its token)
    __shared__ double anew[SCREENED_WAVES][64 * V];
    __shared__ uint16_t list[SCREENED_WAVES][64 * V];
    __shared__ int n_list[SCREENED_WAVES];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = lane_id();
    const int t = blockIdx.x * SCREENED_WAVES + wave;
    const bool mine = t < T;
    double lg[V];
    int my_e = 0, n_mine = 0, at[V];
    double my_l = 0.0, l_max = 0.0;
    uint32_t flag = 0;                                   // bit v: expert lane + 64 v is computed anew
    bool again = false;                                  // the order may change by it
    if (mine) {
        float nx = 0.f, nw = 0.f;
        for (int s = 0; s < S; ++s) nx += xsq[(size_t)s * T + t];
#pragma unroll
        for (int v = 0; v < V; ++v)
            if (lane + 64 * v < E) nw = fmaxf(nw, wsq[lane + 64 * v]);
        sum_logits<V>(partial, t, T, E, S, lg);
        nw = wave_max(nw);
        // what two logits may be apart and still change places.  Everything is computed anew where the norms have left the
        // range in which the argument for the bound holds (2^-80: below, flushed products could matter) and where a logit
        // is not finite.
        const double near = 2.0 * SCREEN_ERR * sqrt((double)nx) * sqrt((double)nw);
        bool odd = !(near < (double)INFINITY) || (nx > 0.f && nx < 8.2718061e-25f) || (nw > 0.f && nw < 8.2718061e-25f);
#pragma unroll
        for (int v = 0; v < V; ++v) odd |= lane + 64 * v < E && !(__builtin_fabs(lg[v]) < (double)INFINITY);
        // the winners and the best of the others, which lane K holds
        const uint32_t taken = select_top<V>(lg, K + 1, E, my_e, my_l, l_max);
        if (__any(odd)) {
            again = true;
#pragma unroll
            for (int v = 0; v < V; ++v) flag |= (lane + 64 * v < E ? 1u : 0u) << v;
        } else if (near > 0.0) {                         // (otherwise every logit is zero)
            const double below = __shfl_down(my_l, 1, 64);
            again = __any(lane < K && my_l - below <= near);
            if (again) {
                for (int k = 0; k <= K; ++k) {
                    const double wl = __shfl(my_l, k, 64);
                    const int we = __builtin_amdgcn_readlane(my_e, k);
#pragma unroll
                    for (int v = 0; v < V; ++v) {
                        const int e = lane + 64 * v;
                        // (against the runner-up only winners are compared, and it against them)
                        const bool counts = e < E && e != we && (k < K || ((taken >> v) & 1u));
                        if (counts && __builtin_fabs(lg[v] - wl) <= near) flag |= 1u << v;
                    }
                }
            }
            // the weights come from the winners' logits
            const int other = __builtin_amdgcn_readlane(my_e, K);
#pragma unroll
            for (int v = 0; v < V; ++v)
                if (lane + 64 * v < E && lane + 64 * v != other) flag |= taken & (1u << v);
        }
#pragma unroll
        for (int v = 0; v < V; ++v) {
            const uint64_t m = __ballot((flag >> v) & 1u);
            at[v] = n_mine + mask_rank(m);
            n_mine += __popcll(m);
            if ((flag >> v) & 1u) list[wave][at[v]] = (uint16_t)(lane + 64 * v);
        }
    }
    if (lane == 0) n_list[wave] = n_mine;
    __syncthreads();
    int n_of[SCREENED_WAVES];
#pragma unroll
    for (int i = 0; i < SCREENED_WAVES; ++i) n_of[i] = __builtin_amdgcn_readfirstlane(n_list[i]);
    for (int unit = wave;; unit += SCREENED_WAVES) {     // (at most as many as the lists have experts)
        int who = 0, first = unit;
        while (who < SCREENED_WAVES && first >= (n_of[who] + ROWS - 1) / ROWS)
            first -= (n_of[who++] + ROWS - 1) / ROWS;
        if (who == SCREENED_WAVES) break;
        first *= ROWS;
        const int tj = blockIdx.x * SCREENED_WAVES + who, n = min(ROWS, n_of[who] - first);
        const uint16_t *xr = x + (size_t)tj * H, *wr[ROWS];
#pragma unroll
        for (int j = 0; j < ROWS; ++j)          // (past the end: the last one again)
            wr[j] = wg + (size_t)__builtin_amdgcn_readfirstlane(list[who][first + min(j, n - 1)]) * H;
        double rstd = 1.0;
        if (NORMED) {
            const int nchunk = (H + 1023) / 1024;
            double tot = 0.0;
            for (int c = 0; c < nchunk; ++c) tot += norm_ss[(size_t)tj * nchunk + c];
            rstd = 1.0 / sqrt(tot / (double)H + eps);
        }
        double d[ROWS] = {};
        for (int h = lane * 8; h < H; h += 512) {
            uint4_t wa[ROWS];
            const uint4_t xa = *(const uint4_t *)(xr + h);
#pragma unroll
            for (int j = 0; j < ROWS; ++j) wa[j] = *(const uint4_t *)(wr[j] + h);
            float a[8];
            Row8<uint16_t>::cvt(xa, a);
            if (NORMED) {
                float g[8];
                Row8<uint16_t>::cvt(*(const uint4_t *)(norm_w + h), g);
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    const float xn = ActIO<uint16_t>::round((float)((double)a[i] * rstd));
                    a[i] = ActIO<uint16_t>::round(__fmul_rn(xn, g[i]));
                }
            }
#pragma unroll
            for (int j = 0; j < ROWS; ++j) {
                float b[8];
                Row8<uint16_t>::cvt(wa[j], b);
#pragma unroll
                for (int i = 0; i < 8; ++i) d[j] = __builtin_fma((double)a[i], (double)b[i], d[j]);
            }
        }
#pragma unroll
        for (int j = 0; j < ROWS; ++j) {
            double l = wave_sum(d[j]);
            if (__builtin_isnan(l)) l = __builtin_nan("");       // one key for every NaN
            if (lane == 0 && j < n) anew[who][first + j] = l;
        }
    }
    __syncthreads();
    if (!mine) return;
#pragma unroll
    for (int v = 0; v < V; ++v)
        if ((flag >> v) & 1u) lg[v] = anew[wave][at[v]];
    if (again) {
        select_top<V>(lg, K, E, my_e, my_l, l_max);
    } else {                                             // the same winners, with their logits as they are now
#pragma unroll
        for (int v = 0; v < V; ++v) {
            const double l = __shfl(lg[v], my_e & 63, 64);
            if (my_e >> 6 == v) my_l = l;
        }
        l_max = __shfl(my_l, 0, 64);
    }
    topk_weights<V>(lg, my_e, my_l, l_max, t, E, K, 1, idx, w, idx64);
}

// Few tokens (T <= 16, P = T * K <= ROUTER_SMALL_PAIRS): one workgroup, one wavefront per token, and
// behind a barrier the same workgroup sorts the pairs by expert -- the dispatch of dispatch.hip on a
// list that fits LDS, without its launch (decode and short verify steps: 4 us of a 107 us layer at
// T = 5).  A pair's slot is the number of pairs of lower experts plus the number of earlier pairs of
// its own expert, which is the stable order of the dispatch kernel.
#define ROUTER_SMALL_PAIRS 128
template <int V>
__global__ __launch_bounds__(1024) void router_topk_dispatch_small_kernel(
    const double *__restrict__ partial, int T, int E, int K, int S, int renorm, int32_t *__restrict__ idx,
    float *__restrict__ w, int64_t *__restrict__ idx64, double *__restrict__ logits,
    int32_t *__restrict__ counts, int32_t *__restrict__ offsets, int32_t *__restrict__ perm,
    int32_t *__restrict__ inv, int32_t *__restrict__ slot_token, int64_t *__restrict__ counts_mirror,
    uint32_t mirror_tag) {
    __shared__ int32_t ids[ROUTER_SMALL_PAIRS];
    const int t = threadIdx.x >> 6, lane = lane_id();
    if (t < T) {
        const int my_e = topk_token<V>(partial, t, T, E, K, S, renorm, idx, w, idx64, logits);
        if (lane < K) ids[t * K + lane] = my_e;
    }
    __syncthreads();
    // wavefront w sorts out experts w, w + nw, ...: the pair list sits in two registers per lane (pairs
    // lane and lane + 64), ballots count the pairs of the expert and of lower experts, and the lanes
    // that hold a pair of the expert take consecutive slots in pair order
    const int P = T * K, nw = blockDim.x >> 6;
    const int id0 = lane < P ? ids[lane] : -1, id1 = lane + 64 < P ? ids[lane + 64] : -1;
    for (int e = t; e < E; e += nw) {
        const uint64_t m0 = __ballot(id0 == e), m1 = __ballot(id1 == e);
        const int c0 = __popcll(m0), c = c0 + __popcll(m1);
        const int lt = __popcll(__ballot(id0 >= 0 && id0 < e)) + __popcll(__ballot(id1 >= 0 && id1 < e));
        if (lane == 0) {
            counts[e] = c;
            if (counts_mirror) counts_mirror[e] = (int64_t)(((uint64_t)mirror_tag << 32) | (uint32_t)c);
            offsets[e] = lt;
            if (e == E - 1) offsets[E] = lt + c;
        }
        if (id0 == e) {
            const int slot = lt + mask_rank(m0);
            perm[lane] = slot;
            inv[slot] = lane;
            slot_token[slot] = lane / K;
        }
        if (id1 == e) {
            const int slot = lt + c0 + mask_rank(m1);
            perm[lane + 64] = slot;
            inv[slot] = lane + 64;
            slot_token[slot] = (lane + 64) / K;
        }
    }
}

// ---- host side -----------------------------------------------------------------------------
struct RouterPlan {
    int NE, EG, TT, S;
    size_t partial_bytes;
};

static RouterPlan router_plan(const odsd_moe_shape *s, bool normed) {
    RouterPlan p;
    const int ET = (s->E + 15) / 16;
    p.TT = (s->T + 15) / 16;
    // Expert tiles per wavefront: more of them re-use a token chunk more often, fewer give more and
    // shorter wavefront units.  With few 16 x 16 output tiles the kernel is a latency chain and short
    // units win (E = 128: 4.6 against 6.9 us at T = 128, 6.5 against 7.1 at 256, 8.4 against 10.6 at
    // 320, with the kernel that the comment there calls "before"); from ~512 tiles on the re-use wins (T = 4096,
    // H = 4096: 94 against 117 us).  With the
    // RMSNorm folded in, every expert group also repeats the normalisation of its token chunk (two
    // fp64 conversions per element): two tiles per wavefront are then the least (T = 256 in the
    // 48-layer stack: 8.2 us against 9.3 with one, 8.3 with four).
    const long tiles = (long)p.TT * ET;
    const int ne = tiles <= 192 ? (normed ? 2 : 1) : (tiles <= 512 ? 2 : 4);
    p.NE = ET >= ne ? ne : (ET >= 2 ? 2 : 1);
    p.EG = (ET + p.NE - 1) / p.NE;
    // split K until there are ~2048 wavefront units or the slices get down to 64 columns
    int S = 1;
    const int maxS = s->H / 64;
    while (S * 2 <= maxS && (s->H / (S * 2)) % 32 == 0 && s->H % (S * 2) == 0 &&
           (long)p.TT * p.EG * S < 2048)
        S *= 2;
    p.S = S;
    p.partial_bytes = odsd_round_up((size_t)S * (size_t)(s->T > 0 ? s->T : 1) * s->E * sizeof(double), 256);
    return p;
}

// Slices of K for router_screen_kernel, or 0 where the fp64 kernels run.  Slices: as many as still give no CU a second workgroup (two
// steps of 128 columns and 8 MB of partial sums are the price at T = 1000).  The choice: from an estimate of either pair, us, because both
// go in steps, the fp64 kernel with the units of work per SIMD, the screen with the workgroups per CU and, where H / 128 is odd,
// with the whole row in one slice.  fp64: 12 + 9.4 for 1000 columns x 16 experts of a SIMD.  Screened: 10, 1 for a step, the winners' rows
// from L2 (10 for 1e8 columns, 32 for 1e5 columns one after the other, 4 experts at a time), the partial sums, the winners' selection.
// 3 us between them are left to the fp64 kernels, 17 with the RMSNorm folded in, which the dot products repeat.  Measured, fp64 /
// screened, K = 8: E = 128: H = 2048: T = 1600 32.5 / 29.4, T = 2000 33.1 / 30.7, T = 2600 41.4 / 34.7, T = 4096 49.8 / 38.8; H = 4096: T = 1000
// 31.0 / 35.8, T = 1300 41.4 / 39.4, T = 2000 51.3 / 41.0, T = 4096 89.1 / 59.8; H = 3968: T = 600 34.5 / 55.4, T = 2000 50.8 / 55.2, T = 4096
// 86.5 / 68.1; E = 66, H = 4096, T = 4096 88.7 / 58.6; E = 512, H = 4096, T = 1000 91.7 / 53.7.  K = 16: E = 128, H = 4096: T = 2000 52.9 / 57.9,
// T = 4096 91.2 / 85.3; E = 512, H = 2048, T = 1000 58.6 / 56.3.  More winners: E = 128, H = 4096, K = 30, T = 4096 96 / 130; K = 24, T = 8991 245 / 227; E = 256,
// K = 48, T = 7710 341 / 383.  Layers with the RMSNorm folded in, K = 8, I = 128: E = 128, H = 4096: T = 2000 214 / 217, T = 4096 412 / 374; E = 256, H = 4096: T = 600
// 145 / 158, T = 2000 284 / 256.  Of 200 shapes drawn where this says screened, 4 were slower, all short of 512 tokens (up to 15 %: too few wavefronts
// behind the winners' rows; hence the bound), the others took 71 % of the time on average.
#define SCREEN_WGS 256
static int screen_slices(const odsd_moe_shape *s, bool normed) {
    if (s->act_dtype != ODSD_DT_BF16 || !s->renorm || s->E <= 64 || s->K >= s->E || s->K > SCREENED_MAX_K || s->T < 512) return 0;
    if ((size_t)s->T * s->H * 2 > 0xffffffffull || (size_t)s->E * s->H * 2 > 0xffffffffull) return 0;
    const long tiles = (long)((s->T + 16 * SCREEN_NT - 1) / (16 * SCREEN_NT)) * ((s->E + SCREEN_EXPERTS - 1) / SCREEN_EXPERTS);
    int S = 1;
    while (s->H % (S * 2 * ODSD_GROUP) == 0 && tiles * S * 2 <= SCREEN_WGS) S *= 2;
    if (s->H / S < 2 * ODSD_GROUP) return 0;             // the kernel has two groups on their way
    const RouterPlan p = router_plan(s, false);
    const double mega = 1e-6 * s->T, steps = (double)((tiles * S + SCREEN_WGS - 1) / SCREEN_WGS) * (s->H / S / ODSD_GROUP);
    const double fp64 = 12 + 9.4e-3 * (((long)p.TT * p.EG * p.S + 1023) / 1024) * (s->H / p.S) * p.NE;
    const double screened = 10 + steps + mega * s->K * s->H / 10 + 3.2e-4 * s->H * ((s->K + 3) / 4) + 6.5 * mega * s->E * S + 1.3 * s->K;
    if (fp64 < screened + (normed ? 17 : 3)) return 0;
    // its logits and norms take no more room than the fp64 kernel's, with the RMSNorm folded in and without
    const size_t a = router_plan(s, false).partial_bytes, b = router_plan(s, true).partial_bytes;
    const size_t need = (size_t)S * s->T * ((size_t)s->E * sizeof(double) + sizeof(float)) + (size_t)s->E * sizeof(float);
    return need <= (a < b ? a : b) ? S : 0;
}

static int router_check(const odsd_moe_shape *s) {
    if (!s) return ODSD_ERR_NULL;
    if (s->T < 0 || s->H <= 0 || s->E <= 0 || s->K <= 0) return ODSD_ERR_SHAPE;
    if (s->H % 128) return ODSD_ERR_SHAPE;
    if (s->K > s->E) return ODSD_ERR_SHAPE;
    if (s->E > 64 * ROUTER_MAX_V || s->K > 64) return ODSD_ERR_UNSUPPORTED;
    if (s->act_dtype != ODSD_DT_F32 && s->act_dtype != ODSD_DT_BF16) return ODSD_ERR_DTYPE;
    return ODSD_OK;
}

extern "C" size_t odsd_router_workspace_bytes(const odsd_moe_shape *s) {
    if (router_check(s) != ODSD_OK) return 0;
    // (the split of K, and with it the partial sums, depends on whether the RMSNorm is folded in)
    const size_t a = router_plan(s, false).partial_bytes, b = router_plan(s, true).partial_bytes;
    return a > b ? a : b;
}

extern "C" int odsd_router_screened(const odsd_moe_shape *s, int32_t normed) {
    return router_check(s) == ODSD_OK && screen_slices(s, normed != 0) > 0;
}

template <typename XT, int NE>
static void launch_partial(const RouterPlan &p, const odsd_moe_shape *s, const void *x, const void *gw,
                           double *partial, void *x16, hipStream_t st, const double *norm_ss,
                           const void *norm_w, float eps) {
    const int n_units = p.TT * p.EG * p.S;
#define PARTIAL_GO(R4, NORMED)                                                                                       \
    ODSD_LAUNCH(ODSD_KERNEL_ROUTER_LOGITS, (router_partial_kernel<XT, NE, R4, NORMED>), (n_units + 3) / 4, 256, st, \
                (const XT *)x, (const XT *)gw, partial, (half_t *)x16, s->T, s->H, s->E, p.S, p.EG, n_units,         \
                norm_ss, (const XT *)norm_w, (double)eps)
    if (p.S % 4 == 0) {
        if (norm_ss) PARTIAL_GO(true, true); else PARTIAL_GO(true, false);
    } else {
        if (norm_ss) PARTIAL_GO(false, true); else PARTIAL_GO(false, false);
    }
#undef PARTIAL_GO
}

int odsd_launch_router(const odsd_moe_shape *s, const void *x, const void *gate_w, int32_t *idx, float *w,
                       int64_t *idx64, void *x16, void *ws, size_t ws_bytes, hipStream_t st,
                       const double *norm_ss, const void *norm_w, float eps, double *logits,
                       const OdsdDispatchOut *disp, int *logits_only) {
    const int rc = router_check(s);
    if (rc != ODSD_OK) return rc;
    if (disp && (!disp->counts || !disp->offsets || !disp->perm || !disp->inv || !disp->slot_token))
        return ODSD_ERR_NULL;
    if (s->T == 0) return ODSD_OK;
    if (!x || !gate_w || !idx || !w || !ws) return ODSD_ERR_NULL;
    if (norm_ss && (!norm_w || !odsd_aligned16(norm_w))) return norm_w ? ODSD_ERR_ALIGN : ODSD_ERR_NULL;
    if (!odsd_aligned16(x) || !odsd_aligned16(gate_w) || !odsd_aligned16(ws) ||
        (x16 && !odsd_aligned16(x16)))
        return ODSD_ERR_ALIGN;
    const RouterPlan p = router_plan(s, norm_ss != nullptr);
    if (ws_bytes < p.partial_bytes) return ODSD_ERR_WORKSPACE;
    double *partial = (double *)ws;
    const int screen_S = logits || logits_only ? 0 : screen_slices(s, norm_ss != nullptr);
    if (screen_S) {
        const int S = screen_S, EG = (s->E + SCREEN_EXPERTS - 1) / SCREEN_EXPERTS, TT = (s->T + 16 * SCREEN_NT - 1) / (16 * SCREEN_NT);
        float *xsq = (float *)(partial + (size_t)S * s->T * s->E), *wsq = xsq + (size_t)S * s->T;
#define SCREEN_GO(NORMED)                                                                                                   \
        ODSD_LAUNCH(ODSD_KERNEL_ROUTER_LOGITS, router_screen_kernel<NORMED>, TT * EG * S, 512, st,                          \
                    (const uint16_t *)x, (const uint16_t *)gate_w, partial, xsq, wsq, (half_t *)x16, s->T, s->H, s->E, S,   \
                    EG, norm_ss, (const uint16_t *)norm_w, (double)eps)
#define SCREENED_GO(VV, NORMED)                                                                                             \
        ODSD_LAUNCH(ODSD_KERNEL_ROUTER_TOPK, (router_topk_screened_kernel<VV, NORMED>),                               \
                    (s->T + SCREENED_WAVES - 1) / SCREENED_WAVES, 64 * SCREENED_WAVES, st, (const double *)partial, (const float *)xsq, (const float *)wsq, (const uint16_t *)x,   \
                    (const uint16_t *)gate_w, s->T, s->H, s->E, s->K, S, idx, w, idx64, norm_ss,             \
                    (const uint16_t *)norm_w, (double)eps)
#define SCREENED_BOTH(VV) do { if (norm_ss) SCREENED_GO(VV, true); else SCREENED_GO(VV, false); } while (0)
        if (norm_ss) SCREEN_GO(true); else SCREEN_GO(false);
        ODSD_CHECK_LAUNCH();
        if (s->E <= 128) SCREENED_BOTH(2);      // E > 64 here
        else if (s->E <= 256) SCREENED_BOTH(4);
        else SCREENED_BOTH(8);
#undef SCREENED_BOTH
#undef SCREENED_GO
#undef SCREEN_GO
        ODSD_CHECK_LAUNCH();
        if (disp)
            return odsd_launch_dispatch(s, idx, disp->counts, disp->offsets, disp->perm, disp->inv, disp->slot_token, st,
                                        disp->counts_mirror, disp->mirror_tag);
        return ODSD_OK;
    }
    const bool bf = s->act_dtype == ODSD_DT_BF16;
#define ROUTER_GO(NEV)                                                                   \
    do {                                                                                 \
        if (bf) launch_partial<uint16_t, NEV>(p, s, x, gate_w, partial, x16, st, norm_ss, norm_w, eps); \
        else launch_partial<float, NEV>(p, s, x, gate_w, partial, x16, st, norm_ss, norm_w, eps);       \
    } while (0)
    if (p.NE == 4) ROUTER_GO(4);
    else if (p.NE == 2) ROUTER_GO(2);
    else ROUTER_GO(1);
#undef ROUTER_GO
    ODSD_CHECK_LAUNCH();
    const int S_out = p.S % 4 == 0 ? p.S / 4 : p.S;
    if (logits_only) {
        *logits_only = S_out;
        return ODSD_OK;
    }
    // one wavefront per token; with few tokens each gets a workgroup of its own (a CU to itself:
    // 4.4 against 4.9 us at T = 256), with many, four share one (8.6 against 9.8 us at T = 4096)
    // (one CU then runs every token's selection: with 2 logits per lane 16 tokens take 10.2 us against
    // 8.6 for the two kernels, 5 tokens 7.2 against 8.4; with one logit per lane 16 tokens 5.4 against 8.1)
    const int topk_v = s->E <= 64 ? 1 : (s->E <= 128 ? 2 : (s->E <= 256 ? 4 : 8));
    if (disp && s->T * topk_v <= 16 && s->K <= 64 && s->T * s->K <= ROUTER_SMALL_PAIRS) {
        // a wavefront per token, and enough of them that the sort has at most 8 experts each
        const int small_waves = max(s->T, min(16, (s->E + 7) / 8));
#define TOPK_SMALL_GO(VV)                                                                                      \
    ODSD_LAUNCH(ODSD_KERNEL_ROUTER_TOPK, router_topk_dispatch_small_kernel<VV>, 1, 64 * small_waves, st,        \
                (const double *)partial, s->T, s->E, s->K, S_out, s->renorm, idx, w, idx64, logits, disp->counts, \
                disp->offsets, disp->perm, disp->inv, disp->slot_token, disp->counts_mirror, disp->mirror_tag)
        if (s->E <= 64) TOPK_SMALL_GO(1);
        else if (s->E <= 128) TOPK_SMALL_GO(2);
        else if (s->E <= 256) TOPK_SMALL_GO(4);
        else TOPK_SMALL_GO(8);
#undef TOPK_SMALL_GO
        ODSD_CHECK_LAUNCH();
        return ODSD_OK;
    }
    const int tk_waves = s->T <= 512 ? 1 : 4;
#define TOPK_GO(VV)                                                                                   \
    ODSD_LAUNCH(ODSD_KERNEL_ROUTER_TOPK, router_topk_kernel<VV>, (s->T + tk_waves - 1) / tk_waves, 64 * tk_waves, st, \
                (const double *)partial, s->T, s->E, s->K, S_out, s->renorm, idx, w, idx64, logits)
    if (s->E <= 64) TOPK_GO(1);
    else if (s->E <= 128) TOPK_GO(2);
    else if (s->E <= 256) TOPK_GO(4);
    else TOPK_GO(8);
#undef TOPK_GO
    ODSD_CHECK_LAUNCH();
    if (disp)
        return odsd_launch_dispatch(s, idx, disp->counts, disp->offsets, disp->perm, disp->inv, disp->slot_token, st,
                                    disp->counts_mirror, disp->mirror_tag);
    return ODSD_OK;
}

extern "C" int odsd_router_topk(const odsd_moe_shape *s, const void *x, const void *gate_w,
                                int32_t *out_idx, float *out_w, int64_t *out_idx64, void *x_f16,
                                void *workspace, size_t workspace_bytes, void *stream) {
    return odsd_launch_router(s, x, gate_w, out_idx, out_w, out_idx64, x_f16, workspace, workspace_bytes,
                              (hipStream_t)stream, nullptr, nullptr, 0.0f, nullptr, nullptr);
}

extern "C" int odsd_route_dispatch(const odsd_moe_shape *s, const void *x, const void *gate_w,
                                   int32_t *out_idx, float *out_w, int64_t *out_idx64, void *x_f16,
                                   int32_t *counts, int32_t *offsets, int32_t *perm, int32_t *inv,
                                   int32_t *slot_token, void *workspace, size_t workspace_bytes, void *stream) {
    const OdsdDispatchOut d{counts, offsets, perm, inv, slot_token};
    return odsd_launch_router(s, x, gate_w, out_idx, out_w, out_idx64, x_f16, workspace, workspace_bytes,
                              (hipStream_t)stream, nullptr, nullptr, 0.0f, nullptr, &d);
}

extern "C" int odsd_route_dispatch_host_counts(const odsd_moe_shape *s, const void *x, const void *gate_w,
                                               int32_t *out_idx, float *out_w, int64_t *out_idx64, void *x_f16,
                                               int32_t *counts, int32_t *offsets, int32_t *perm, int32_t *inv,
                                               int32_t *slot_token, int64_t *counts_host, uint32_t tag,
                                               void *workspace, size_t workspace_bytes, void *stream) {
    const OdsdDispatchOut d{counts, offsets, perm, inv, slot_token, counts_host, tag};
    return odsd_launch_router(s, x, gate_w, out_idx, out_w, out_idx64, x_f16, workspace, workspace_bytes,
                              (hipStream_t)stream, nullptr, nullptr, 0.0f, nullptr, &d);
}

extern "C" int odsd_router_topk_logits(const odsd_moe_shape *s, const void *x, const void *gate_w,
                                       int32_t *out_idx, float *out_w, int64_t *out_idx64, void *x_f16,
                                       double *out_logits, void *workspace, size_t workspace_bytes,
                                       void *stream) {
    if (!out_logits) return ODSD_ERR_NULL;
    return odsd_launch_router(s, x, gate_w, out_idx, out_w, out_idx64, x_f16, workspace, workspace_bytes,
                              (hipStream_t)stream, nullptr, nullptr, 0.0f, out_logits, nullptr);
}
