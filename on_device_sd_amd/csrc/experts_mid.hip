// Streaming W4 GEMM for experts with some 13 to 48 rows and long token rows (32 groups of 128 columns or more).
//
// One workgroup of 4 wavefronts owns 16 blocks of 16 weight rows of one expert, two workgroups per CU; a wavefront owns
// 4 blocks and all token rows of a pass (up to 3 blocks of 16; compiled per number of blocks).
//   * Codes go to the matrix cores as they are, scale and zero point are applied to each group's sum, as in the
//     equal-share kernel (a layer's error against 64 bits, weights rounded to fp16 / this: 4.7e-4 / 2.9e-4); the sums of the token columns that this takes come from a product with a constant operand.
//   * Token rows arrive by asynchronous global -> LDS copies two groups ahead (three buffers, one barrier per group), a
//     group's fragments are read once and serve all four tiles.
//   * Each product is followed by its share of the next tile's expansion and of the previous tile's scales, so that
//     matrix and vector instructions of one wavefront overlap.
//   * Workgroups start on different groups.  Row blocks lie 32 KiB apart at H = 4096, and workgroups that all walk
//     the groups in step ask the same few memory channels at a time: from the same group / from different ones, whole
//     layer, us: H = 4096, I = 14336, E = 8, T = 56 165 / 142, T = 100 177 / 164; I = 1536, E = 128, T = 256 296 / 257.
//     Neighbours on one XCD (every eighth workgroup) are 5 groups apart, XCDs one.  Apart by one in launch order,
//     i.e. an XCD's all at the same L2 channels: 266 for the last.
//   * Up to four workgroups share the passes over a tile: a popular expert's passes run side by side instead of in turn, the
//     workgroups without one come last and only look at the row count.  Zipf-distributed routing, E = 128, one / four,
//     layer, us: T = 256 352 / 302, T = 400 464 / 357; uniform routing does not notice (256 / 256, 291 / 293).
//
// Bound by issue from some 25 rows on: H = 4096, I = 14336, E = 8, T = 136 (34 rows) matrix cores busy 37 % of the cycles, other
// vector instructions issuing 35 %, 1.75 rounds of workgroups; T = 100 32 % and 34 %.  At up to 16 rows by HBM.  Measured and
// not kept: no interleaving of vector and matrix instructions (before the workgroups started on different groups, E = 128,
// T = 400: 318 / 309 with it; E = 8, T = 160 208 / 211).  Passes of 64 rows take 254 registers without the interleaving and leave none for it.
//
//   MODE 0  gate_up: h = SiLU(gate) * up -> fp16
//   MODE 1  down: KS splits of the reduction across workgroups, fp16 sums
#include "w4_gemm.h"
#include "w4_raw.h"

#include <type_traits>

#define MID_WAVES 4
#define MID_MB 3               // token blocks of a pass: 48 rows
#define MID_XB 3               // token-row buffers

template <int MODE, int NB>
__global__ __launch_bounds__(64 * MID_WAVES, 2) void w4_mid_kernel(const GemmParams p) {
    constexpr int XS = 16 * MID_MB * 256;                // bytes of a token-row buffer: 48 rows of one group
    __shared__ __attribute__((aligned(16))) char xs_raw[MID_XB * XS];
    // everyone's first passes come before anyone's second
    const int b = (int)blockIdx.x % p.n_wg, ps = (int)blockIdx.x / p.n_wg;
    static_assert(NB % 2 == 0, "a wavefront has gate and up of its features");
    const int ks = b % p.KS, chunk = (b / p.KS) % p.nchunks, e = b / (p.KS * p.nchunks);
    const uint64_t *trow = p.table + (size_t)e * ODSD_TABLE_COLS;
    const uint64_t t_present = trow[0];
    const uint64_t t_q = MODE == 0 ? trow[0] : trow[2], t_sz = MODE == 0 ? trow[1] : trow[3];
    const int M_e = p.counts[e], base = p.offsets[e];
    if (M_e <= ps * 16 * MID_MB || t_present == 0) return;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r = lane & 15, kq = lane >> 4;
    const int g_begin = ks * p.gper, g_end = min(p.G, g_begin + p.gper);
    const int blk0 = (chunk * MID_WAVES + wave) * NB;
    // the group that step n of the reduction works on
    const int ng = g_end - g_begin, rot = ((b >> 3) * 5 + (b & 7)) % ng;
    auto grp = [&](const int n) { const int k = n + rot; return g_begin + (k >= ng ? k - ng : k); };
    const RawConsts rc = raw_consts();
    const global_char *src_c = (const global_char *)p.src;
    const __amdgpu_buffer_rsrc_t rq = __builtin_amdgcn_make_buffer_rsrc((void *)(uintptr_t)t_q, 0, p.NBLK * p.G * 1024, 0x00020000);
    const __amdgpu_buffer_rsrc_t rsz = __builtin_amdgcn_make_buffer_rsrc((void *)(uintptr_t)t_sz, 0, p.NBLK * p.G * 64, 0x00020000);
    // blocks past the last repeat it; their sums are not stored
    int tile0[NB];
#pragma unroll
    for (int i = 0; i < NB; ++i) tile0[i] = min(blk0 + i, p.NBLK - 1) * p.G;
    const int st_seg = tid & 15, st_row0 = tid >> 4;
    uint32_t lds_frag[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) lds_frag[j] = (uint32_t)((r * 16 + ((4 * j + kq) ^ r)) * 16);
    // A operand whose product with a token block gives, in every lane, minus the offsets' share of its token's sum (row 0
    // of 4) and the sum of the token's columns (row 1 of 4)
    half8_t asum;
    {
        const half_t lo = (half_t)((r & 3) == 0 ? -ODSD_RAW_OFFSET_LO : (r & 3) == 1 ? 1.0f : 0.0f);
        const half_t hi = (half_t)((r & 3) == 0 ? -ODSD_RAW_OFFSET_HI : (r & 3) == 1 ? 1.0f : 0.0f);
        asum = half8_t{lo, lo, hi, hi, lo, lo, hi, hi};
    }

    auto pass = [&](auto nm_c, const int m0, const int mcnt) {
        constexpr int NM = decltype(nm_c)::value;
        uint32_t st_off[NM];
#pragma unroll
        for (int i = 0; i < NM; ++i) {
            const int row = st_row0 + 16 * i;
            const int slot = base + m0 + (row < mcnt ? row : 0);
            const int srow = MODE == 0 ? p.rowmap[slot] : slot;
            st_off[i] = ((uint32_t)srow * (uint32_t)p.src_ld + (uint32_t)((st_seg ^ (row & 15)) * 8)) * 2u;
        }
        uint4_t wq[NB], wsz[NB];
        uint32_t q_voff = (uint32_t)lane * 16u, sz_voff = (uint32_t)kq * 16u;
        auto load_q = [&](const int i, const int g) {
            wq[i] = __builtin_amdgcn_raw_buffer_load_b128(rq, (int)q_voff, (tile0[i] + grp(g)) * 1024, 2 /* nt */);
        };
        auto load_sz = [&](const int i, const int g) {
            wsz[i] = __builtin_amdgcn_raw_buffer_load_b128(rsz, (int)sz_voff, (tile0[i] + grp(g)) * 64, 0);
        };
        auto dma_x = [&](const int buf, const int g) {
            const global_char *xg = src_c + (size_t)grp(min(g, ng - 1)) * (ODSD_GROUP * 2u);
#pragma unroll
            for (int i = 0; i < NM; ++i)
                dma16_to_lds(xg, st_off[i], (lds_void *)(xs_raw + buf * XS + (i * 64 * MID_WAVES + wave * 64) * 16));
        };
        __builtin_amdgcn_s_barrier();        // the previous pass is done with the buffers
        dma_x(0, 0);
        dma_x(1, 1);
#pragma unroll
        for (int i = 0; i < NB; ++i) {
            load_q(i, 0);
            load_sz(i, 0);
        }
        float4_t acc[NB][NM];
#pragma unroll
        for (int i = 0; i < NB; ++i)
#pragma unroll
            for (int m = 0; m < NM; ++m) acc[i][m] = float4_t{0.f, 0.f, 0.f, 0.f};
        ODSD_WAIT_VMCNT(NM + 2 * NB);        // the first group's rows
        __builtin_amdgcn_s_barrier();
        int xb = 0;
        for (int g = 0; g < ng; ++g) {
            ODSD_FENCE();
            // rows two groups ahead, into the buffer that the previous step read
            dma_x(xb == 0 ? 2 : xb - 1, g + 2);
            if (g + 1 == ng) q_voff = sz_voff = 0x80000000u;       // nothing left to fetch
            half8_t bx[NM][4];
            const char *xf = xs_raw + xb * XS;
#pragma unroll
            for (int m = 0; m < NM; ++m)
#pragma unroll
                for (int j = 0; j < 4; ++j) bx[m][j] = *(const half8_t *)(xf + m * 4096 + lds_frag[j]);
            float4_t off[NM];
            float xs[NM];
            half8_t a[2][4];
            float4_t t[2][NM];
            auto expand = [&](const int i) {
                a[i & 1][0] = raw_word(rc, wq[i].x);
                a[i & 1][1] = raw_word(rc, wq[i].y);
                a[i & 1][2] = raw_word(rc, wq[i].z);
                a[i & 1][3] = raw_word(rc, wq[i].w);
            };
            auto pin_a = [&](const int i) {
                asm volatile("" : "+v"(a[i & 1][0]), "+v"(a[i & 1][1]), "+v"(a[i & 1][2]), "+v"(a[i & 1][3]));
            };
            auto scale = [&](const int i) {
                const uint4_t z = wsz[i];
                const half2_t p0 = as_half2(z.x), p1 = as_half2(z.y), p2 = as_half2(z.z), p3 = as_half2(z.w);
#pragma unroll
                for (int m = 0; m < NM; ++m) {
                    float4_t &o = acc[i][m];
                    const float4_t v = t[i & 1][m];
                    const float4_t u = {__builtin_fmaf(-(float)p0.y, xs[m], v.x), __builtin_fmaf(-(float)p1.y, xs[m], v.y),
                                        __builtin_fmaf(-(float)p2.y, xs[m], v.z), __builtin_fmaf(-(float)p3.y, xs[m], v.w)};
                    o.x = __builtin_fmaf((float)p0.x, u.x, o.x);
                    o.y = __builtin_fmaf((float)p1.x, u.y, o.y);
                    o.z = __builtin_fmaf((float)p2.x, u.z, o.z);
                    o.w = __builtin_fmaf((float)p3.x, u.w, o.w);
                }
            };
            auto pin_acc = [&](const int i) {
#pragma unroll
                for (int m = 0; m < NM; ++m) asm volatile("" : "+v"(acc[i][m].x), "+v"(acc[i][m].y), "+v"(acc[i][m].z), "+v"(acc[i][m].w));
            };
            expand(0);
#pragma unroll
            for (int m = 0; m < NM; ++m) off[m] = float4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int m = 0; m < NM; ++m) off[m] = __builtin_amdgcn_mfma_f32_16x16x32_f16(asum, bx[m][j], off[m], 0, 0, 0);
#pragma unroll
            for (int m = 0; m < NM; ++m) {
                xs[m] = off[m].y;
                off[m] = float4_t{off[m].x, off[m].x, off[m].x, off[m].x};
            }
            pin_a(0);
            ODSD_FENCE();
            load_q(0, g + 1);
#pragma unroll
            for (int i = 0; i < NB; ++i) {
                ODSD_FENCE();
                if (i + 1 < NB) expand(i + 1);
#pragma unroll
                for (int j = 0; j < 4; ++j)
#pragma unroll
                    for (int m = 0; m < NM; ++m)
                        t[i & 1][m] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[i & 1][j], bx[m][j], j == 0 ? off[m] : t[i & 1][m], 0, 0, 0);
                if (i > 0) scale(i - 1);
                // every product is followed by its share of the vector instructions: the next tile's expansion, the previous one's scales
#pragma unroll
                for (int k = 0; k < 4 * NM; ++k) {
                    __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
                    __builtin_amdgcn_sched_group_barrier(0x2, (20 + 8 * NM + 4 * NM - 1) / (4 * NM), 0);
                }
                if (i + 1 < NB) pin_a(i + 1);
                if (i > 0) pin_acc(i - 1);
                ODSD_FENCE();
                if (i + 1 < NB) load_q(i + 1, g + 1);
                if (i > 0) load_sz(i - 1, g + 1);
            }
            ODSD_FENCE();
            scale(NB - 1);
            pin_acc(NB - 1);
            ODSD_FENCE();
            load_sz(NB - 1, g + 1);
            ODSD_FENCE();
            // the next group's rows, requested in the step before this one, have landed once no more than that step's
            // weights, this step's rows and this step's weights are outstanding
            ODSD_WAIT_VMCNT(4 * NB + NM);
            __builtin_amdgcn_s_barrier();
            xb = xb == 2 ? 0 : xb + 1;
        }
        ODSD_WAIT_VMCNT(0);                  // no copy outlives the pass
        // lane: rows 4 kq .. of each block, token r
#pragma unroll
        for (int m = 0; m < NM; ++m) {
            const int row = m * 16 + r;
            if (row >= mcnt) continue;
            const size_t slot = (size_t)(base + m0 + row);
            if constexpr (MODE == 0) {
#pragma unroll
                for (int i = 0; i < NB; i += 2) {
                    if (blk0 + i >= p.NBLK) break;
                    const float4_t gt = acc[i][m], up = acc[i + 1][m];
                    const half4_t h = {f32_to_f16_sat(silu_f32(gt.x) * up.x), f32_to_f16_sat(silu_f32(gt.y) * up.y),
                                       f32_to_f16_sat(silu_f32(gt.z) * up.z), f32_to_f16_sat(silu_f32(gt.w) * up.w)};
                    *(half4_t *)(p.h16 + slot * p.ldo + ((blk0 + i) >> 1) * 16 + kq * 4) = h;
                }
            } else {
#pragma unroll
                for (int i = 0; i < NB; ++i) {
                    if (blk0 + i >= p.NBLK) break;
                    const float4_t v = acc[i][m];
                    const size_t at = ((size_t)ks * p.P + slot) * p.ldo + (blk0 + i) * 16 + kq * 4;
                    *(half4_t *)((half_t *)p.y + at) = half4_t{f32_to_f16_sat(v.x), f32_to_f16_sat(v.y), f32_to_f16_sat(v.z), f32_to_f16_sat(v.w)};
                }
            }
        }
    };
    for (int m0 = ps * 16 * MID_MB; m0 < M_e; m0 += p.PS * 16 * MID_MB) {
        const int mcnt = min(M_e - m0, 16 * MID_MB);
        if (mcnt <= 16) pass(std::integral_constant<int, 1>{}, m0, mcnt);
        else if (mcnt <= 32) pass(std::integral_constant<int, 2>{}, m0, mcnt);
        else pass(std::integral_constant<int, 3>{}, m0, mcnt);
    }
}

void odsd_launch_mid(int mode, GemmParams &gp, hipStream_t st) {
    constexpr int NB = 4;
    gp.nchunks = (gp.NBLK + MID_WAVES * NB - 1) / (MID_WAVES * NB);
    gp.n_wg = gp.E * gp.nchunks * gp.KS;
    if (mode == 0) ODSD_LAUNCH(ODSD_KERNEL_GATE_UP, (w4_mid_kernel<0, NB>), gp.n_wg * gp.PS, 64 * MID_WAVES, st, gp);
    else ODSD_LAUNCH(ODSD_KERNEL_DOWN, (w4_mid_kernel<1, NB>), gp.n_wg * gp.PS, 64 * MID_WAVES, st, gp);
}
