// Grouped W4A16 expert product for calls with more than 52 token rows per expert on average.
//
// One workgroup of 4 wavefronts owns 256 weight rows x up to 128 token rows, two workgroups per CU;
// a wavefront owns 64 of the weight rows and ALL of the token rows (2 x NM blocks of 32 x 32 on
// v_mfma_f32_32x32x16_f16, NM = 1 .. 4 compiled separately, chosen per pass by the rows there are).
//   * The weights never pass through LDS: a wavefront expands its own rows (int4 -> fp16 in
//     registers, once per pass), straight from the packed tiles.  Two 16-row tiles make a 32-row A
//     operand: lane l takes row l % 16 of tile (l >> 4) & 1, columns 32 j + 16 (l >> 5) + 8 i + 0..7
//     for step (i, j), which is one word of the packed layout.  In gate_up the two tiles are a gate
//     and an up block, so accumulator registers q and q + 8 of a lane are gate and up of one feature.
//   * The token rows of a 128-column group arrive by asynchronous global -> LDS copies, 256 bytes a
//     row, 16-byte segments XORed with the row (mod 16): no bank conflicts in the loop.  Double
//     buffered, one barrier per group.
//   * A group is 8 steps of 16 columns.  Each step's MFMAs run with the fragment reads and the
//     expansion of the next step between them; the last step crosses the barrier and takes the first
//     fragments of the next group.
//   * fp16 results leave through LDS in whole rows of the tile.
// Passes: an expert with more rows than a pass holds shares its 32-row blocks evenly between passes.
//
// What bounds it: before, weights went expanded through LDS (192 KB read + 64 KB written per 64-column
// stage of 2048 matrix cycles, the 128 bytes per cycle that LDS has).  Now LDS reads are half of that,
// and the matrix unit is busy 71 % of the cycles (down: 63 %) at the 1.4 GHz that the load takes the clock down to
// (Qwen3-235B experts, T = 4096: gate_up 987 -> 830 us, 990 TFLOP/s, down 578 -> 425 us, 970 TFLOP/s;
// the library's fp16 product of 8192^3 reaches 1160 on the same card).  At 62 rows per expert vector
// and matrix instructions share the time (53 % each of the cycles with workgroups).
// Variants: one wavefront per SIMD with 256 token rows per pass, i.e. half the expansion: 1.50 against
// 1.45 ms for that layer (nothing runs under its barriers, prologue and epilogue).
//
// Replaces the same reference code as the streaming kernel: the three F.linear calls of
// expert_forward_with_weights (demo/src/layers/mlp.py:227-230) inside the per-expert loop of
// demo/src/model/qwen3_runner.py:303-380.
#include "w4_gemm.h"

#include <type_traits>

typedef float float16_t __attribute__((ext_vector_type(16)));

template <int MODE>
__global__ __launch_bounds__(256, 2) void w4_gemm_prefill_kernel(const GemmParams p) {
    constexpr int MAXNM = 4;                   // 32-row token blocks per pass
    constexpr int XS_BUF = MAXNM * 32 * 256;   // one group of the token rows
    __shared__ __attribute__((aligned(16))) char xs[2 * XS_BUF];

    // consecutive logical ids stay on one XCD: the row tiles of one expert share its token rows.  Everyone's
    // first passes come before anyone's second: a workgroup without a pass then costs the end of the launch
    // a look at the row count, and not the others a place.
    const int b = blockIdx.x;
    const int ps = (b >> 3) / p.wg_per_xcd;
    const int L = (b & 7) * p.wg_per_xcd + (b >> 3) - ps * p.wg_per_xcd;
    if (L >= p.n_wg) return;
    // row chunks innermost: neighbours share the token rows of one (expert, pass, K slice)
    const int chunk = L % p.nchunks;
    const int ks = (L / p.nchunks) % p.KS;
    const int e = L / (p.nchunks * p.KS);

    // requested together: one round trip to memory instead of three dependent ones
    const uint64_t *trow = p.table + (size_t)e * ODSD_TABLE_COLS;
    const int M_e = p.counts[e];
    const int base = p.offsets[e];
    const uint64_t t_present = trow[0];
    const uint64_t t_q = MODE == 0 ? trow[0] : trow[2], t_sz = MODE == 0 ? trow[1] : trow[3];
    if (M_e == 0 || t_present == 0) return;
    const global_char *src_c = (const global_char *)p.src;
    const __amdgpu_buffer_rsrc_t rsrc_q = __builtin_amdgcn_make_buffer_rsrc((void *)(uintptr_t)t_q, 0, p.NBLK * p.G * 1024, 0x00020000);
    const __amdgpu_buffer_rsrc_t rsrc_sz = __builtin_amdgcn_make_buffer_rsrc((void *)(uintptr_t)t_sz, 0, p.NBLK * p.G * 64, 0x00020000);

    const DequantConsts dc = dequant_consts();
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n = lane & 31, kh = lane >> 5;
    const int G = p.G;
    const int g_begin = ks * p.gper, g_end = min(G, g_begin + p.gper);   // this K slice (never empty)

    // this wavefront's tiles 4 wave .. 4 wave + 3 of the chunk: all inside the matrix or none
    // (its row blocks are a multiple of 8); a wavefront without tiles works on tile 0 and stores nothing
    const int cblk0 = chunk * 16 + 4 * wave;
    const bool blk_ok = cblk0 < p.NBLK;
    uint32_t wq_off[2], sz_off[2];
#pragma unroll
    for (int rb = 0; rb < 2; ++rb) {
        const uint32_t blk = (blk_ok ? cblk0 : 0) + 2 * rb + ((lane >> 4) & 1);
        wq_off[rb] = (blk * G * 64 + (lane & 15) + 32 * kh) * 16u;
        sz_off[rb] = (blk * G * 16 + (lane & 15)) * 4u;
    }
    // this lane's B fragment of step s = (i, j) = (s & 1, s >> 1): token row n, segment 4 j + 2 kh + i
    const uint32_t frag0 = (uint32_t)(n * 256 + (((2 * kh) ^ (n & 15)) << 4));
    auto frag = [&](const int s) { return frag0 ^ (uint32_t)((4 * (s >> 1) + (s & 1)) << 4); };

    const int nblk = (M_e + 31) >> 5;                   // 32-row token blocks of this expert
    const int npass = (nblk + MAXNM - 1) / MAXNM;

    auto run_pass = [&](auto nm_c, const int m0, const int mcnt) {
        constexpr int NM = decltype(nm_c)::value;
        // copies of this wavefront: token rows 16 i + 4 wave + lane / 16, source segment (lane % 16) ^ (row % 16);
        // rows past the expert's last one copy its first: what they feed is never stored
        uint32_t st_off[2 * NM];
#pragma unroll
        for (int i = 0; i < 2 * NM; ++i) {
            const int row = 16 * i + 4 * wave + (lane >> 4);
            const int slot = base + m0 + (row < mcnt ? row : 0);
            const int srow = p.rowmap ? p.rowmap[slot] : slot;
            st_off[i] = ((uint32_t)srow * (uint32_t)p.src_ld + ((lane & 15) ^ (row & 15)) * 8) * 2u;
        }
        float16_t acc[2][NM];
#pragma unroll
        for (int rb = 0; rb < 2; ++rb)
#pragma unroll
            for (int m = 0; m < NM; ++m)
#pragma unroll
                for (int i = 0; i < 16; ++i) acc[rb][m][i] = 0.0f;

        // Packed weights in registers: those of the group at hand (wq) and F groups on their way, fetched
        // behind the copies of the token rows that have to land before them, so that the wait for those
        // copies leaves the youngest in flight.  (F == 2 with four blocks of rows spills.)
        constexpr int F = NM <= 3 ? 2 : 1;
        uint4_t wq[2][2], wq_f[F][2][2];       // [slot = group % F][row block][i], words j = 0..3
        uint32_t wsz_f[F][2];
        auto load_w = [&](auto slot_c, const int g) {
            constexpr int slot = decltype(slot_c)::value % F;
            const int gc = min(g, g_end - 1);
#pragma unroll
            for (int rb = 0; rb < 2; ++rb) {
                wq_f[slot][rb][0] = __builtin_amdgcn_raw_buffer_load_b128(rsrc_q, (int)wq_off[rb], gc * 1024, 2 /* nt */);
                wq_f[slot][rb][1] = __builtin_amdgcn_raw_buffer_load_b128(rsrc_q, (int)wq_off[rb] + 256, gc * 1024, 2 /* nt */);
                wsz_f[slot][rb] = __builtin_amdgcn_raw_buffer_load_b32(rsrc_sz, (int)sz_off[rb], gc * 64, 0);
            }
        };
        auto dma_piece = [&](const uint32_t buf, const int g, const int i) {
            lds_void *dst = (lds_void *)(xs + buf + (16 * i + 4 * wave) * 256);
            dma16_to_lds(src_c + (size_t)g * (ODSD_GROUP * 2u), st_off[i], dst);
        };
        half8_t a[2][2], bx[2][NM];  // [step parity]
        DequantPrep pr[2];
        auto expand = [&](const int par, const int s) {
#pragma unroll
            for (int rb = 0; rb < 2; ++rb) a[par][rb] = dequant_word(dc, pr[rb], wq[rb][s & 1][s >> 1]);
        };
        // group g's weights have landed and become those at hand; past the slice's end their scale is zero
        auto take_w = [&](auto slot_c, const int g) {
            constexpr int slot = decltype(slot_c)::value % F;
#pragma unroll
            for (int rb = 0; rb < 2; ++rb) {
                wq[rb][0] = wq_f[slot][rb][0];
                wq[rb][1] = wq_f[slot][rb][1];
                pr[rb] = dequant_prep(F == 1 || g < g_end ? wsz_f[slot][rb] : 0u);
            }
        };
        using Slot0 = std::integral_constant<int, 0>;
        using Slot1 = std::integral_constant<int, 1>;

        __builtin_amdgcn_s_barrier();          // the previous pass is done with the token rows
#pragma unroll
        for (int i = 0; i < 2 * NM; ++i) dma_piece(0, g_begin, i);
        load_w(Slot0{}, g_begin);
        if (F == 2) load_w(Slot1{}, g_begin + 1);
        __builtin_amdgcn_sched_barrier(0);
        ODSD_WAIT_VMCNT_LGKM0((F - 1) * 6);
        __builtin_amdgcn_s_barrier();
        uint32_t cur = 0;                      // byte offset of the buffer of the group at hand
#pragma unroll
        for (int m = 0; m < NM; ++m) bx[0][m] = *(const half8_t *)(xs + frag(0) + m * 8192);
        take_w(Slot0{}, g_begin);
        expand(0, 0);

        // One group.  Every load is issued whatever follows (past the slice's end: its last group again).
        auto group = [&](auto slot_c, const int g) {
            constexpr int slot = decltype(slot_c)::value;
            const char *xb = xs + cur;
            const int gx = min(g + 1, g_end - 1);
#pragma unroll
            for (int s = 0; s < 8; ++s) {
                const int par = s & 1;
                __builtin_amdgcn_sched_barrier(0);
                if (s == 7) {
                    // into the next group: this wavefront's copies and its next weights have landed, its
                    // reads of this group's rows are complete; then the same of every wavefront
                    ODSD_WAIT_VMCNT_LGKM0((F - 1) * 6);
                    __builtin_amdgcn_s_barrier();
                    xb = xs + (cur ^ XS_BUF);
                }
#pragma unroll
                for (int m = 0; m < NM; ++m) bx[par ^ 1][m] = *(const half8_t *)(xb + frag((s + 1) & 7) + m * 8192);
                if (s == 7) take_w(std::integral_constant<int, slot ^ 1>{}, g + 1);
                expand(par ^ 1, (s + 1) & 7);
#pragma unroll
                for (int m = 0; m < NM; ++m)
#pragma unroll
                    for (int rb = 0; rb < 2; ++rb)
                        acc[rb][m] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[par][rb], bx[par][m], acc[rb][m], 0, 0, 0);
                constexpr int NV = (27 + 2 * NM - 1) / (2 * NM);
#pragma unroll
                for (int m = 0; m < NM; ++m) {
                    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);     // MFMA
                    __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);     // LDS read
                    __builtin_amdgcn_sched_group_barrier(0x002, NV, 0);    // vector
                    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                    __builtin_amdgcn_sched_group_barrier(0x002, NV, 0);
                }
                // the next group's copies, two a step (into the buffer of the group before this one); the
                // weights of the next group in front of them (F == 1), or those of the group after it behind them
                if (s <= NM) __builtin_amdgcn_sched_barrier(0);
                if (F == 1 && s == 0) load_w(Slot0{}, g + 1);
                if (s < NM) {
                    dma_piece(cur ^ XS_BUF, gx, 2 * s);
                    dma_piece(cur ^ XS_BUF, gx, 2 * s + 1);
                }
                if (F == 2 && s == NM) load_w(slot_c, g + 2);
            }
            __builtin_amdgcn_sched_barrier(0);
            cur ^= XS_BUF;
        };
        for (int g = g_begin; g < g_end; g += F) {
            group(Slot0{}, g);
            if (F == 2) group(Slot1{}, g + 1);
        }
        ODSD_WAIT_VMCNT_LGKM0(0);              // the copies that nobody waited for must not land in the results

        // epilogue: register 4 q + u of a lane is row 8 q + 4 kh + u of the 32-row block, token n
        // The results (fp16 in both modes: this plan keeps fp16 sums) go through LDS (16-byte pieces of a token's row XORed with the token), so that
        // they leave in whole rows of the tile
        constexpr int OUTB = MODE == 0 ? 256 : 512;    // bytes of one token's results in this tile
        constexpr int PIECES = OUTB / 16;
        __builtin_amdgcn_s_barrier();                  // every wavefront has read its last fragments
#pragma unroll
        for (int m = 0; m < NM; ++m) {
            const int row = m * 32 + n;
#pragma unroll
            for (int rb = 0; rb < 2; ++rb)
#pragma unroll
                for (int q = 0; q < (MODE == 0 ? 2 : 4); ++q) {
                    half4_t h;
#pragma unroll
                    for (int u = 0; u < 4; ++u)
                        h[u] = f32_to_f16_sat(MODE == 0 ? silu_f32(acc[rb][m][4 * q + u]) * acc[rb][m][(8 + 4 * q + u) & 15] : acc[rb][m][4 * q + u]);
                    const int piece = MODE == 0 ? 4 * wave + 2 * rb + q : 8 * wave + 4 * rb + q;
                    *(half4_t *)(xs + row * OUTB + ((piece ^ (n & (PIECES - 1))) << 4) + 8 * kh) = h;
                }
        }
        __syncthreads();
        char *out = MODE == 0 ? (char *)p.h16 : (char *)p.y + (size_t)ks * p.P * p.ldo * 2;
        const int width = min(OUTB, (int)(p.ldo * 2 - chunk * OUTB));     // the matrix may end inside the tile
        const int piece = lane & (PIECES - 1), sub = lane / PIECES;
        for (int row = wave * (64 / PIECES) + sub; row < mcnt; row += 256 / PIECES) {
            const uint4_t v = *(const uint4_t *)(xs + row * OUTB + ((piece ^ (row & (PIECES - 1))) << 4));
            if (piece * 16 < width)
                *(uint4_t *)(out + (size_t)(base + m0 + row) * p.ldo * 2 + (size_t)chunk * OUTB + piece * 16) = v;
        }
        __syncthreads();                               // the next pass copies into the same memory
    };

    for (int q = ps; q < npass; q += p.PS) {
        const int per = nblk / npass, rest = nblk % npass;       // the first `rest` passes take one block more
        const int b0 = q * per + min(q, rest), nm = per + (q < rest);
        const int m0 = b0 * 32, mcnt = min(M_e - m0, nm * 32);
        switch (nm) {
#define PASS(N) case N: run_pass(std::integral_constant<int, N>{}, m0, mcnt); break;
            PASS(1) PASS(2) PASS(3) PASS(4)
#undef PASS
        }
    }
}

template <int MODE>
void odsd_launch_gemm_prefill(GemmParams &gp, hipStream_t st) {
    gp.nchunks = (gp.NBLK + 15) / 16;
    if (gp.PS < 1) gp.PS = 1;
    gp.n_wg = gp.E * gp.nchunks * gp.KS;
    gp.wg_per_xcd = (gp.n_wg + 7) / 8;
    ODSD_LAUNCH(MODE == 0 ? ODSD_KERNEL_GATE_UP : ODSD_KERNEL_DOWN, (w4_gemm_prefill_kernel<MODE>), gp.wg_per_xcd * 8 * gp.PS, 256, st, gp);
}

template void odsd_launch_gemm_prefill<0>(GemmParams &, hipStream_t);
template void odsd_launch_gemm_prefill<1>(GemmParams &, hipStream_t);
