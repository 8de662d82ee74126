// W4 quantiser, streaming-layout packer, RMSNorm and activation conversion for gfx950.
// All of these are HBM-bound byte movers; none of them is shaped as a GEMM.
#include "common.h"

// -----------------------------------------------------------------------------------------
// Arithmetic of the quantiser, per (row, group of 128 columns).  It follows quantize_tensor (pre_exp/expert_skip_prediction/quant.py:99-106) per
// group with 4 bits: scale=(max-min)/15, zero=0-min/scale (a float, never rounded to an
// integer), q=clamp(round(w/scale+zero),0,15).  scale and zero are rounded to fp16 before
// the codes are computed.  Every fp32 step is a single correctly rounded operation
// (__f*_rn) so that a CPU restatement gets the same bits.
// -----------------------------------------------------------------------------------------
struct QuantParams {
    half_t s16, z16;     // as stored
    float sf, zf;        // the same values, what the codes are computed with
};
__device__ __forceinline__ QuantParams quant_params(const float mn, const float mx) {
    const float s32 = __fdiv_rn(__fsub_rn(mx, mn), 15.0f);
    half_t s16 = (half_t)s32;
    if (!(s16 > (half_t)0.0f)) s16 = (half_t)1.0f;
    if (__builtin_isinf((float)s16)) s16 = (half_t)ODSD_FP16_MAX;
    const float sf = (float)s16;
    float z32 = __fsub_rn(0.0f, __fdiv_rn(mn, sf));
    z32 = fminf(fmaxf(z32, -ODSD_FP16_MAX), ODSD_FP16_MAX);
    const half_t z16 = (half_t)z32;
    return QuantParams{s16, z16, sf, (float)z16};
}
__device__ __forceinline__ uint32_t quant_code(const float w, const QuantParams &p) {
    const float t = rintf(__fadd_rn(__fdiv_rn(w, p.sf), p.zf));
    return (uint32_t)fminf(fmaxf(t, 0.0f), 15.0f);
}

// Canonical form: one wavefront per (row, group); lane l owns columns 2l, 2l+1.
template <typename WT>
__global__ __launch_bounds__(256) void w4_quantize_kernel(const WT *__restrict__ w, int64_t n_units,
                                                          int64_t G, uint8_t *__restrict__ q,
                                                          uint16_t *__restrict__ scale,
                                                          uint16_t *__restrict__ zero) {
    const int lane = lane_id();
    const int64_t unit = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);  // row * G + g
    if (unit >= n_units) return;
    const size_t base = (size_t)unit * ODSD_GROUP + 2 * lane;
    const float w0 = ActIO<WT>::load(w, base);
    const float w1 = ActIO<WT>::load(w, base + 1);
    const float mn = wave_min(fminf(w0, w1));
    const float mx = wave_max(fmaxf(w0, w1));
    const QuantParams qp = quant_params(mn, mx);
    const uint32_t c0 = quant_code(w0, qp), c1 = quant_code(w1, qp);
    q[(size_t)unit * (ODSD_GROUP / 2) + lane] = (uint8_t)(c0 | (c1 << 4));
    if (lane == 0) {
        scale[unit] = __builtin_bit_cast(uint16_t, qp.s16);
        zero[unit] = __builtin_bit_cast(uint16_t, qp.z16);
    }
}

// -----------------------------------------------------------------------------------------
// Packer.  One thread per (destination block, group, lane): gathers its 4 words of 8 codes
// and writes them as one 16-byte store, so a wavefront later streams one [16 rows x 128
// columns] tile as a single contiguous 1 KiB read.
//   word j of lane l (r = l%16, kq = l/16): row 16*b+r, columns 128*g + 32*j + 8*kq + i,
//   code i in nibble {0,4,1,5,2,6,3,7}[i]  (pairs (0,1),(2,3),(4,5),(6,7) then fall out of
//   the masks 0x000F000F / 0x00F000F0 of the word and of the word >> 8).
// -----------------------------------------------------------------------------------------
__device__ __forceinline__ uint32_t permute_nibbles(uint32_t c) {
    // input nibble i (LSB first) = code i; output nibble pos(i)
    uint32_t o = 0;
    o |= ((c >> 0) & 0xFu) << 0;    // i=0 -> 0
    o |= ((c >> 4) & 0xFu) << 16;   // i=1 -> 4
    o |= ((c >> 8) & 0xFu) << 4;    // i=2 -> 1
    o |= ((c >> 12) & 0xFu) << 20;  // i=3 -> 5
    o |= ((c >> 16) & 0xFu) << 8;   // i=4 -> 2
    o |= ((c >> 20) & 0xFu) << 24;  // i=5 -> 6
    o |= ((c >> 24) & 0xFu) << 12;  // i=6 -> 3
    o |= ((c >> 28) & 0xFu) << 28;  // i=7 -> 7
    return o;
}

__global__ __launch_bounds__(256) void w4_pack_kernel(const uint8_t *__restrict__ q,
                                                      const uint16_t *__restrict__ scale,
                                                      const uint16_t *__restrict__ zero, int64_t nb_src,
                                                      int64_t G, int block_stride, int block_offset,
                                                      uint4_t *__restrict__ qp,
                                                      uint32_t *__restrict__ sz) {
    const int64_t gid = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int64_t total = nb_src * G * 64;
    if (gid >= total) return;
    const int lane = (int)(gid & 63);
    const int64_t bg = gid >> 6;
    const int64_t g = bg % G;
    const int64_t b = bg / G;
    const int r = lane & 15, kq = lane >> 4;
    const int64_t row = b * 16 + r;
    const int64_t kbytes = G * (ODSD_GROUP / 2);
    const uint32_t *src = (const uint32_t *)(q + row * kbytes + g * 64 + kq * 4);
    uint4_t out;
    out.x = permute_nibbles(src[0]);
    out.y = permute_nibbles(src[4]);   // +16 bytes
    out.z = permute_nibbles(src[8]);
    out.w = permute_nibbles(src[12]);
    const int64_t bd = b * block_stride + block_offset;
    qp[(bd * G + g) * 64 + lane] = out;
    if (kq == 0) {
        const uint32_t s = scale[row * G + g], z = zero[row * G + g];
        sz[(bd * G + g) * 16 + r] = s | (z << 16);
    }
}

// -----------------------------------------------------------------------------------------
// Quantise-on-load of one expert: gate, up and down weights -> streaming layout in ONE launch, with no
// canonical copy in between.  A wavefront takes one [16 rows x 128 columns] tile; its lane (r = l%16,
// kq = l/16) reads columns 32j + 8kq .. + 7 of row r (j = 0..3), which are exactly the codes of its
// four packed words, so the group's minimum and maximum need two exchanges between lanes and the tile
// leaves as one contiguous 1 KiB store.  Consecutive wavefronts take consecutive groups of a row
// block.  Bound by one launch with one round trip and the divisions behind it.  16 experts of [768, 2048] in bf16, 12 MB
// each, weights that no cache holds, the launches queued up: 88.0 us (92.7 with ordinary stores, whose lines the end of a launch
// writes back; nontemporal loads besides 90.7).  Rows read in runs of 1 KiB, the words turned through LDS: 96 (83 only where
// the same 12 MB come again and again).  As three quantise and three pack launches with a canonical copy in
// between, 96 calls in all, 715 us.
// -----------------------------------------------------------------------------------------
struct LoadMatrix {
    const void *w;
    uint4_t *qp;
    uint32_t *sz;
    int f32;                     // 1: fp32 weights, 0: bf16
    int G;                       // groups per row
    int first;                   // first tile of this matrix in the launch
    int bstride, boffset;        // destination block = b * bstride + boffset
};
struct LoadParams {
    LoadMatrix m[3];
    int n_tiles;
};
__global__ __launch_bounds__(256) void w4_load_expert_kernel(const LoadParams p) {
    const int tile = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (tile >= p.n_tiles) return;
    const int which = __builtin_amdgcn_readfirstlane((tile >= p.m[1].first) + (tile >= p.m[2].first));
    const LoadMatrix m = p.m[which];
    const int t = tile - m.first;
    const int b = t / m.G, g = t - b * m.G;
    const int lane = lane_id(), r = lane & 15, kq = lane >> 4;
    const size_t at = ((size_t)(b * 16 + r) * m.G + g) * ODSD_GROUP + kq * 8;
    float w[4][8];
    if (m.f32) {
        const float *src = (const float *)m.w + at;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const float4_t lo = *(const float4_t *)(src + 32 * j), hi = *(const float4_t *)(src + 32 * j + 4);
            w[j][0] = lo.x; w[j][1] = lo.y; w[j][2] = lo.z; w[j][3] = lo.w;
            w[j][4] = hi.x; w[j][5] = hi.y; w[j][6] = hi.z; w[j][7] = hi.w;
        }
    } else {
        const uint16_t *src = (const uint16_t *)m.w + at;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const uint4_t v = *(const uint4_t *)(src + 32 * j);
            const uint32_t u[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                w[j][2 * i] = __uint_as_float(u[i] << 16);
                w[j][2 * i + 1] = __uint_as_float(u[i] & 0xffff0000u);
            }
        }
    }
    float mn = w[0][0], mx = w[0][0];
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            mn = fminf(mn, w[j][i]);
            mx = fmaxf(mx, w[j][i]);
        }
#pragma unroll
    for (int d = 16; d <= 32; d <<= 1) {
        mn = fminf(mn, __shfl_xor(mn, d, ODSD_WAVE));
        mx = fmaxf(mx, __shfl_xor(mx, d, ODSD_WAVE));
    }
    const QuantParams qp = quant_params(mn, mx);
    // w / scale, correctly rounded, in three instructions: q0 = w y with y = 1 / scale correctly rounded is
    // within 1.5 units of the quotient, its residual w - q0 scale is exact, and one correction leaves an
    // error below 2^-23 units before the last rounding.  scale has 11 significant bits (it is an fp16
    // value), so a quotient that is not itself halfway between two floats is at least 2^-12 units away
    // from that point, and no 24-bit w has a quotient exactly there: the last rounding is the right one.
    // (Quotients too small for that argument vanish when the zero point is added.)  Groups with
    // infinities take the division.
    const bool finite = mx - mn < INFINITY;
    const float y = __fdiv_rn(1.0f, qp.sf);
    uint32_t out[4];
    constexpr int pos[8] = {0, 16, 4, 20, 8, 24, 12, 28};      // permute_nibbles: code i -> bit position
#pragma unroll
    for (int j = 0; j < 4; ++j) out[j] = 0;
    if (__all(finite)) {
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const float q0 = __fmul_rn(w[j][i], y);
                const float q = fmaf(fmaf(-q0, qp.sf, w[j][i]), y, q0);
                const float t = rintf(__fadd_rn(q, qp.zf));
                out[j] |= (uint32_t)__builtin_amdgcn_fmed3f(t, 0.0f, 15.0f) << pos[i];
            }
    } else {
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int i = 0; i < 8; ++i) out[j] |= quant_code(w[j][i], qp) << pos[i];
    }
    const size_t dst = (size_t)(b * m.bstride + m.boffset) * m.G + g;
    __builtin_nontemporal_store(uint4_t{out[0], out[1], out[2], out[3]}, &m.qp[dst * 64 + lane]);
    if (kq == 0)
        m.sz[dst * 16 + r] = (uint32_t)__builtin_bit_cast(uint16_t, qp.s16) | ((uint32_t)__builtin_bit_cast(uint16_t, qp.z16) << 16);
}

// -----------------------------------------------------------------------------------------
// RMSNorm (demo/src/layers/layernorm.py:21-27): statistics in fp64, the normalised value is
// rounded to the activation dtype BEFORE the weight multiply, the product is rounded again.
// One workgroup per token.
// -----------------------------------------------------------------------------------------
template <typename XT>
__global__ __launch_bounds__(256) void rmsnorm_kernel(const XT *__restrict__ x, const XT *__restrict__ wt,
                                                      int H, double eps, XT *__restrict__ out) {
    __shared__ double red[2][4];
    const size_t row = (size_t)blockIdx.x * H;
    // The sum of squares is built exactly as the combine kernel builds the row statistic it
    // leaves for the next block (per 1024-column chunk: 4 consecutive columns per thread, a
    // wavefront sum, the 4 wavefront sums pairwise; chunks added in ascending order), so that
    // the stand-alone and the folded RMSNorm give the same bits.
    double tot = 0.0;
    for (int c0 = 0, n = 0; c0 < H; c0 += 1024, ++n) {
        const int c = c0 + (int)threadIdx.x * 4;
        double ss = 0.0;
        if (c < H) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const double v = (double)ActIO<XT>::load(x, row + c + i);
                ss += v * v;
            }
        }
        ss = wave_sum(ss);
        if (lane_id() == 0) red[n & 1][threadIdx.x >> 6] = ss;
        __syncthreads();
        tot += (red[n & 1][0] + red[n & 1][1]) + (red[n & 1][2] + red[n & 1][3]);
    }
    const double r = 1.0 / sqrt(tot / (double)H + eps);
    for (int h = threadIdx.x; h < H; h += 256) {
        const float xn = ActIO<XT>::round((float)((double)ActIO<XT>::load(x, row + h) * r));
        ActIO<XT>::store(out, row + h, __fmul_rn(xn, ActIO<XT>::load(wt, h)));
    }
}

// The same for rows of up to 1024 NC columns at aligned addresses: the row and the weights are requested once, together, and stay in
// registers (one round trip to memory and one barrier where the kernel above has a round trip and a barrier per 1024 columns
// and then reads the row again).  Same additions in the same order.  T = 24, H = 2048, four layers of
// an engine loop: 260.3 -> 254.2 us.
template <typename XT, int NC>
__global__ __launch_bounds__(256) void rmsnorm_row_kernel(const XT *__restrict__ x, const XT *__restrict__ wt, int H, double eps,
                                                          XT *__restrict__ out) {
    typedef XT xt4 __attribute__((ext_vector_type(4)));
    __shared__ double red[NC][4];
    const size_t row = (size_t)blockIdx.x * H;
    xt4 xv[NC], wv[NC];
#pragma unroll
    for (int n = 0; n < NC; ++n) {
        const int c = 1024 * n + (int)threadIdx.x * 4;
        xv[n] = xt4{};
        wv[n] = xt4{};
        if (c < H) {
            xv[n] = *(const xt4 *)(x + row + c);
            wv[n] = *(const xt4 *)(wt + c);
        }
    }
    double ss[NC];
#pragma unroll
    for (int n = 0; n < NC; ++n) {
        ss[n] = 0.0;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const XT e = xv[n][i];
            const double v = (double)ActIO<XT>::load(&e, 0);
            ss[n] += v * v;
        }
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1)
#pragma unroll
        for (int n = 0; n < NC; ++n) ss[n] += __shfl_xor(ss[n], o, ODSD_WAVE);
    if (lane_id() == 0) {
#pragma unroll
        for (int n = 0; n < NC; ++n) red[n][threadIdx.x >> 6] = ss[n];
    }
    __syncthreads();
    double tot = 0.0;
#pragma unroll
    for (int n = 0; n < NC; ++n)
        if (1024 * n < H) tot += (red[n][0] + red[n][1]) + (red[n][2] + red[n][3]);
    const double r = 1.0 / sqrt(tot / (double)H + eps);
#pragma unroll
    for (int n = 0; n < NC; ++n) {
        const int c = 1024 * n + (int)threadIdx.x * 4;
        if (c >= H) break;
        xt4 o;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const XT xe = xv[n][i], we = wv[n][i];
            const float xn = ActIO<XT>::round((float)((double)ActIO<XT>::load(&xe, 0) * r));
            XT e;
            ActIO<XT>::store(&e, 0, __fmul_rn(xn, ActIO<XT>::load(&we, 0)));
            o[i] = e;
        }
        *(xt4 *)(out + row + c) = o;
    }
}

// Fused residual add + RMSNorm (RMSNorm.add_rms_forward, demo/src/layers/layernorm.py:29-36):
//   s = float(x) + float(residual); residual_out = cast(s);
//   normed = cast(s * rsqrt(mean(s^2) + eps)) * weight   -- statistics over the UNROUNDED sum s.
// One workgroup per token; the sum is recomputed in the second sweep instead of being kept.
template <typename XT>
__global__ __launch_bounds__(256) void add_rmsnorm_kernel(const XT *__restrict__ x, const XT *__restrict__ res,
                                                          const XT *__restrict__ wt, int H, double eps,
                                                          XT *__restrict__ out, XT *__restrict__ res_out) {
    __shared__ double red[4];
    const size_t row = (size_t)blockIdx.x * H;
    double ss = 0.0;
    for (int h = threadIdx.x; h < H; h += 256) {
        const float s = __fadd_rn(ActIO<XT>::load(x, row + h), ActIO<XT>::load(res, row + h));
        ss += (double)s * (double)s;
    }
    ss = wave_sum(ss);
    if (lane_id() == 0) red[threadIdx.x >> 6] = ss;
    __syncthreads();
    const double tot = (red[0] + red[1]) + (red[2] + red[3]);
    const double r = 1.0 / sqrt(tot / (double)H + eps);
    for (int h = threadIdx.x; h < H; h += 256) {
        const float s = __fadd_rn(ActIO<XT>::load(x, row + h), ActIO<XT>::load(res, row + h));
        ActIO<XT>::store(res_out, row + h, s);
        const float xn = ActIO<XT>::round((float)((double)s * r));
        ActIO<XT>::store(out, row + h, __fmul_rn(xn, ActIO<XT>::load(wt, h)));
    }
}

template <typename XT>
__global__ __launch_bounds__(256) void convert_f16_kernel(const XT *__restrict__ x, int64_t n,
                                                          half_t *__restrict__ o) {
    int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int64_t step = (int64_t)gridDim.x * 256;
    for (; i < n; i += step) o[i] = f32_to_f16_sat(ActIO<XT>::load(x, i));
}

// -----------------------------------------------------------------------------------------
// entry points
// -----------------------------------------------------------------------------------------
extern "C" int odsd_w4_quantize(const void *w, int32_t w_dtype, int64_t N, int64_t Kd, uint8_t *q,
                                uint16_t *scale, uint16_t *zero, void *stream) {
    if (!w || !q || !scale || !zero) return ODSD_ERR_NULL;
    if (N <= 0 || Kd <= 0 || Kd % ODSD_GROUP) return ODSD_ERR_SHAPE;
    const int64_t G = Kd / ODSD_GROUP, units = N * G;
    if ((units + 3) / 4 > 0x7fffffffLL) return ODSD_ERR_SHAPE;
    const dim3 grid((unsigned)((units + 3) / 4));
    hipStream_t st = (hipStream_t)stream;
    if (w_dtype == ODSD_DT_F32)
        w4_quantize_kernel<float><<<grid, 256, 0, st>>>((const float *)w, units, G, q, scale, zero);
    else if (w_dtype == ODSD_DT_BF16)
        w4_quantize_kernel<uint16_t><<<grid, 256, 0, st>>>((const uint16_t *)w, units, G, q, scale, zero);
    else
        return ODSD_ERR_DTYPE;
    ODSD_CHECK_LAUNCH();
    return ODSD_OK;
}

extern "C" size_t odsd_w4_packed_q_bytes(int64_t N, int64_t Kd) {
    if (N <= 0 || Kd <= 0 || N % 16 || Kd % ODSD_GROUP) return 0;
    return (size_t)N * (size_t)Kd / 2;
}
extern "C" size_t odsd_w4_packed_sz_bytes(int64_t N, int64_t Kd) {
    if (N <= 0 || Kd <= 0 || N % 16 || Kd % ODSD_GROUP) return 0;
    return (size_t)N * (size_t)(Kd / ODSD_GROUP) * 4;
}

extern "C" int odsd_w4_pack(const uint8_t *q, const uint16_t *scale, const uint16_t *zero, int64_t N,
                            int64_t Kd, int32_t block_stride, int32_t block_offset, uint32_t *qp,
                            uint16_t *sz, void *stream) {
    if (!q || !scale || !zero || !qp || !sz) return ODSD_ERR_NULL;
    if (N <= 0 || Kd <= 0 || N % 16 || Kd % ODSD_GROUP) return ODSD_ERR_SHAPE;
    if (block_stride < 1 || block_offset < 0 || block_offset >= block_stride) return ODSD_ERR_SHAPE;
    if (!odsd_aligned16(qp) || (((uintptr_t)q) & 3u) || (((uintptr_t)sz) & 3u)) return ODSD_ERR_ALIGN;
    const int64_t G = Kd / ODSD_GROUP, nb = N / 16, total = nb * G * 64;
    if ((total + 255) / 256 > 0x7fffffffLL) return ODSD_ERR_SHAPE;
    w4_pack_kernel<<<dim3((unsigned)((total + 255) / 256)), 256, 0, (hipStream_t)stream>>>(
        q, scale, zero, nb, G, block_stride, block_offset, (uint4_t *)qp, (uint32_t *)sz);
    ODSD_CHECK_LAUNCH();
    return ODSD_OK;
}

extern "C" int odsd_w4_load_expert(const void *gate, int32_t gate_dtype, const void *up, int32_t up_dtype,
                                   const void *down, int32_t down_dtype, int64_t H, int64_t I, uint32_t *gu_q,
                                   uint16_t *gu_sz, uint32_t *dn_q, uint16_t *dn_sz, void *stream) {
    if (!gate || !up || !down || !gu_q || !gu_sz || !dn_q || !dn_sz) return ODSD_ERR_NULL;
    if (H <= 0 || I <= 0 || H % ODSD_GROUP || I % ODSD_GROUP || H * I > (1LL << 40)) return ODSD_ERR_SHAPE;
    for (const int32_t d : {gate_dtype, up_dtype, down_dtype})
        if (d != ODSD_DT_F32 && d != ODSD_DT_BF16) return ODSD_ERR_DTYPE;
    for (const void *q : {gate, up, down, (const void *)gu_q, (const void *)dn_q})
        if (!odsd_aligned16(q)) return ODSD_ERR_ALIGN;
    if ((((uintptr_t)gu_sz) | ((uintptr_t)dn_sz)) & 3u) return ODSD_ERR_ALIGN;
    const int64_t tiles = I / 16 * (H / ODSD_GROUP), tiles_dn = H / 16 * (I / ODSD_GROUP);   // the same number
    if (2 * tiles + tiles_dn > 0x7fffffffLL / 4) return ODSD_ERR_SHAPE;
    const int Gu = (int)(H / ODSD_GROUP), Gd = (int)(I / ODSD_GROUP);
    const LoadParams p{{{gate, (uint4_t *)gu_q, (uint32_t *)gu_sz, gate_dtype == ODSD_DT_F32, Gu, 0, 2, 0},
                        {up, (uint4_t *)gu_q, (uint32_t *)gu_sz, up_dtype == ODSD_DT_F32, Gu, (int)tiles, 2, 1},
                        {down, (uint4_t *)dn_q, (uint32_t *)dn_sz, down_dtype == ODSD_DT_F32, Gd, (int)(2 * tiles), 1, 0}},
                       (int)(2 * tiles + tiles_dn)};
    w4_load_expert_kernel<<<dim3((unsigned)((p.n_tiles + 3) / 4)), 256, 0, (hipStream_t)stream>>>(p);
    ODSD_CHECK_LAUNCH();
    return ODSD_OK;
}

extern "C" int odsd_rmsnorm(const void *x, const void *weight, int32_t dtype, int32_t T, int32_t H,
                            float eps, void *out, void *stream) {
    if (!x || !weight || !out) return ODSD_ERR_NULL;
    if (T < 0 || H <= 0) return ODSD_ERR_SHAPE;
    if (T == 0) return ODSD_OK;
    hipStream_t st = (hipStream_t)stream;
    if (dtype != ODSD_DT_F32 && dtype != ODSD_DT_BF16) return ODSD_ERR_DTYPE;
    // rows that the registers hold, four columns at a time
    const uintptr_t all = (uintptr_t)x | (uintptr_t)weight | (uintptr_t)out;
    if (H <= 4096 && H % 4 == 0 && (all & (dtype == ODSD_DT_F32 ? 15u : 7u)) == 0) {
#define NORM_ROW(XT, NC)                                                                                             \
        ODSD_LAUNCH(ODSD_KERNEL_NORM, (rmsnorm_row_kernel<XT, NC>), T, 256, st, (const XT *)x, (const XT *)weight, H, \
                    (double)eps, (XT *)out)
#define NORM_ROW_XT(XT)                        \
        do {                                   \
            if (H <= 1024) NORM_ROW(XT, 1);    \
            else if (H <= 2048) NORM_ROW(XT, 2); \
            else NORM_ROW(XT, 4);              \
        } while (0)
        if (dtype == ODSD_DT_F32) NORM_ROW_XT(float);
        else NORM_ROW_XT(uint16_t);
#undef NORM_ROW_XT
#undef NORM_ROW
        ODSD_CHECK_LAUNCH();
        return ODSD_OK;
    }
    if (dtype == ODSD_DT_F32)
        ODSD_LAUNCH(ODSD_KERNEL_NORM, rmsnorm_kernel<float>, T, 256, st, (const float *)x, (const float *)weight,
                    H, (double)eps, (float *)out);
    else
        ODSD_LAUNCH(ODSD_KERNEL_NORM, rmsnorm_kernel<uint16_t>, T, 256, st, (const uint16_t *)x,
                    (const uint16_t *)weight, H, (double)eps, (uint16_t *)out);
    ODSD_CHECK_LAUNCH();
    return ODSD_OK;
}

extern "C" int odsd_add_rmsnorm(const void *x, const void *residual, const void *weight, int32_t dtype,
                                int32_t T, int32_t H, float eps, void *out, void *residual_out, void *stream) {
    if (!x || !residual || !weight || !out || !residual_out) return ODSD_ERR_NULL;
    if (T < 0 || H <= 0) return ODSD_ERR_SHAPE;
    if (T == 0) return ODSD_OK;
    hipStream_t st = (hipStream_t)stream;
    if (dtype == ODSD_DT_F32)
        add_rmsnorm_kernel<float><<<T, 256, 0, st>>>((const float *)x, (const float *)residual,
                                                     (const float *)weight, H, (double)eps, (float *)out,
                                                     (float *)residual_out);
    else if (dtype == ODSD_DT_BF16)
        add_rmsnorm_kernel<uint16_t><<<T, 256, 0, st>>>((const uint16_t *)x, (const uint16_t *)residual,
                                                        (const uint16_t *)weight, H, (double)eps,
                                                        (uint16_t *)out, (uint16_t *)residual_out);
    else
        return ODSD_ERR_DTYPE;
    ODSD_CHECK_LAUNCH();
    return ODSD_OK;
}

extern "C" int odsd_convert_act_f16(const void *x, int32_t dtype, int64_t n, void *x_f16, void *stream) {
    if (!x || !x_f16) return ODSD_ERR_NULL;
    if (n < 0) return ODSD_ERR_SHAPE;
    if (n == 0) return ODSD_OK;
    int64_t blocks = (n + 255) / 256;
    if (blocks > 65536) blocks = 65536;
    hipStream_t st = (hipStream_t)stream;
    if (dtype == ODSD_DT_F32)
        convert_f16_kernel<float><<<(unsigned)blocks, 256, 0, st>>>((const float *)x, n, (half_t *)x_f16);
    else if (dtype == ODSD_DT_BF16)
        convert_f16_kernel<uint16_t><<<(unsigned)blocks, 256, 0, st>>>((const uint16_t *)x, n,
                                                                      (half_t *)x_f16);
    else
        return ODSD_ERR_DTYPE;
    ODSD_CHECK_LAUNCH();
    return ODSD_OK;
}
