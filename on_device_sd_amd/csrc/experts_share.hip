// Streaming W4 GEMM in equal shares: experts with few rows on average.
//
// The weights of the experts with rows are one long list of units -- (expert, pass of 16 rows, blocks of 16 weight rows) --
// and every workgroup takes the same number of consecutive units, one more or less, whichever experts they belong to: one
// workgroup per CU, no second round of workgroups, no CU left over because its expert has no rows, and an expert with more
// rows than a pass holds is just more units of the list.  Where a unit is large and a share short that one unit shows: down
// at I = 768 has units of 51 KB, 6.3 to 7.1 per CU at T = 24 to 64, so the slowest, with 7 or 8, takes 11 to 13 % longer
// than the mean.
//
// The wavefronts of a workgroup split the reduction: a wavefront owns GW groups of 128 columns of every unit, so
// the token rows it needs -- its columns of the expert's rows -- stay in registers as MFMA B operands for as long
// as the expert lasts; nothing is staged through LDS and nothing waits for a copy inside the stream.  The
// accumulators of the parts meet in LDS once per unit (fixed order, two buffers, one barrier that no load waits
// at), and the wavefronts share the sums and stores, 4 rows x 16 outputs at a time.
//
// Codes go to the matrix cores as they are, scale and zero point are applied to each group's sum (as in
// w4_expert_fused_kernel: 5 vector instructions per 8 weights instead of 13).
//
// Bound by HBM once it streams: 3.5 GB of gate_up (H = 4096, I = 14336, 56 experts) take 496 us, 7.0 TB/s.  Short streams are
// mostly start-up: 2.8 us until the list is there, 1 to 2 until the first rows and weights are.  H = 2048, I = 768, E = 128,
// T = 24, the kernel whose workgroups own (expert, 128 rows) / this: gate_up 39.3 / 29.8 us (169 MB, 5.7 TB/s), down
// 20.1 / 18.2 (84 MB, 4.6 TB/s); H = 4096, I = 14336, T = 5: 59.4 / 48.6 and 30.7 / 27.7.  Measured and not kept: reading a
// unit's sums behind the next unit's steps (no change), one wavefront per whole reduction without a barrier (down there 20.2:
// its rows are then read eight times), 6 wavefronts with one group each (21.9: two SIMDs have twice the work of the others),
// 16 wavefronts per CU with 3 steps in flight each (23.5), two token blocks per pass (T = 256: 47 + 34).
//
//   MODE 0  gate_up: unit = a gate block and its up block, h = SiLU(gate) * up -> fp16
//   MODE 1  down: unit = RSUB * NB blocks of output rows, KS splits of the reduction across workgroups, fp32 or fp16 sums
#include "w4_gemm.h"
#include "w4_raw.h"
#include "router_topk.h"

#include <type_traits>

#define SHARE_WAVES 8
#define SHARE_MAX_P 4096       // slot -> token list in LDS
#define SHARE_MAX_ITEMS 1024   // (expert, pass) pairs

// inclusive prefix sum over the wavefront
__device__ __forceinline__ int wave_prefix(int x) {
#define ODSD_SCAN_STEP(CTRL, ROWMASK) x += __builtin_amdgcn_update_dpp(0, x, CTRL, ROWMASK, 0xF, false)
    ODSD_SCAN_STEP(0x111, 0xF);   // row_shr:1
    ODSD_SCAN_STEP(0x112, 0xF);
    ODSD_SCAN_STEP(0x114, 0xF);
    ODSD_SCAN_STEP(0x118, 0xF);   // within rows of 16
    ODSD_SCAN_STEP(0x142, 0xA);   // row_bcast:15 into rows 1 and 3
    ODSD_SCAN_STEP(0x143, 0xC);   // row_bcast:31 into rows 2 and 3
#undef ODSD_SCAN_STEP
    return x;
}

// NI    0: dispatch arrays are given; otherwise the kernel dispatches for itself, up to 512 NI pairs
// ROUTE 1, 2: it does the top-k as well, E <= 64 / 128
template <int MODE, int GW, int WK, int NB, int DEPTH, int NI, int ROUTE>
__global__ __launch_bounds__(64 * SHARE_WAVES, 2) void w4_share_kernel(const GemmParams p) {
    constexpr int WAVES = SHARE_WAVES, RSUB = WAVES / WK, UBLK = RSUB * NB;   // 16-row blocks of a unit
    constexpr bool DISP = NI > 0;
    constexpr int ROWS = 16, MAX_E = 64 * WAVES;     // one thread per expert in the prologue
    constexpr int SPU = GW * NB / 2;                      // steps (one group of two blocks) per unit
    static_assert(SPU % DEPTH == 0, "every unit begins on ring slot 0");
    static_assert(MODE == 1 || UBLK == 2, "gate_up: a gate block and its up block");
    static_assert(!DISP || MODE == 0, "gate_up dispatches");
    __shared__ __attribute__((aligned(16))) float red[2][WK][UBLK][256];
    __shared__ int32_t cnt_lds[MAX_E], off_lds[MAX_E];
    __shared__ uint64_t tq_lds[MAX_E], tsz_lds[MAX_E];
    __shared__ uint16_t list_lds[MODE == 0 ? SHARE_MAX_P : 1];   // token of a slot
    __shared__ uint32_t item_lds[SHARE_MAX_ITEMS];               // expert | pass << 16
    __shared__ int32_t tot_lds[WAVES];
    __shared__ __attribute__((aligned(16))) uint16_t cntw_lds[DISP ? WAVES : 1][DISP ? MAX_E : 1];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r = lane & 15, kq = lane >> 4;
    const int kpart = wave / RSUB, rsub = wave % RSUB;
    const int ks = blockIdx.x % p.KS, share = blockIdx.x / p.KS, n_share = p.n_wg / p.KS;

    // ---- which experts have rows, and where: everything is requested at once ---------------------------
    // DISP: the pair list is sorted by expert here, by every workgroup for itself.  Wavefront w takes pairs
    // w * 64 NI .., 64 at a time; a pair's rank among the earlier pairs of its expert is what lies before it in the
    // wavefront's batch (a match by ballots over the bits of the id), plus the wavefront's earlier batches, plus the
    // wavefronts before it.
    int id[DISP ? NI : 1], rank[DISP ? NI : 1];
    if (DISP && ROUTE == 0) {
#pragma unroll
        for (int n = 0; n < NI; ++n) {
            const int i = (wave * NI + n) * 64 + lane;
            id[n] = i < p.P ? p.idx[i] : -1;
        }
    }
    uint64_t q = 0, sz = 0;
    int c = 0, o = 0;
    if (tid < p.E) {
        const uint64_t *trow = p.table + (size_t)tid * ODSD_TABLE_COLS;
        q = trow[MODE == 0 ? 0 : 2];
        sz = trow[MODE == 0 ? 1 : 3];
        if (MODE == 1 && trow[0] == 0) q = 0;
        if (!DISP) {
            c = p.counts[tid];
            o = p.offsets[tid];
        }
    }
    if (MODE == 0 && !DISP)
        for (int i = tid; i < p.P; i += 64 * WAVES) list_lds[i] = (uint16_t)p.rowmap[i];
    if (ROUTE > 0) {
        // every workgroup selects for every token; workgroup t leaves token t's experts and weights behind
        for (int t = wave; t < p.T; t += WAVES) {
            const bool mine = t == (int)blockIdx.x;
            const int e = topk_token<(ROUTE > 0 ? ROUTE : 1)>(p.partial, t, p.T, p.E, p.K, p.route_S, p.renorm, mine ? p.route_idx : nullptr,
                                                                 mine ? p.route_w : nullptr, nullptr, nullptr);
            if (lane < p.K) list_lds[t * p.K + lane] = (uint16_t)e;
        }
        __syncthreads();
#pragma unroll
        for (int n = 0; n < NI; ++n) {
            const int i = (wave * NI + n) * 64 + lane;
            id[n] = i < p.P ? (int)list_lds[i] : -1;
        }
    }
    if (DISP) {
        *(uint4_t *)&cntw_lds[wave][8 * lane] = uint4_t{0, 0, 0, 0};
#pragma unroll
        for (int n = 0; n < NI; ++n) {
            {
                const int x = (uint32_t)id[n] < (uint32_t)p.E ? id[n] : -1;   // others belong to nobody
                id[n] = x;
                uint64_t same = __ballot(x >= 0);
                for (int bit = 0; (1 << bit) < p.E; ++bit) {
                    const uint64_t m = __ballot(x >> bit & 1);
                    same &= x >> bit & 1 ? m : ~m;
                }
                if (x >= 0) {
                    rank[n] = cntw_lds[wave][x] + mask_rank(same);
                    if (lane == 63 - __builtin_clzll(same)) cntw_lds[wave][x] = (uint16_t)(rank[n] + 1);
                }
            }
        }
        __syncthreads();
        // counts over the wavefronts -> first rank of each wavefront, and the expert's rows
        int k[WAVES];
#pragma unroll
        for (int w = 0; w < WAVES; ++w) k[w] = cntw_lds[w][tid];
#pragma unroll
        for (int w = 0; w < WAVES; ++w) {
            cntw_lds[w][tid] = (uint16_t)c;
            c += k[w];
        }
    }
    tq_lds[tid] = q;
    tsz_lds[tid] = sz;
    cnt_lds[tid] = c;
    // (expert, pass) items in expert order and, DISP, the experts' first slots: prefix sums of both in one word
    const int np = q != 0 ? (c + ROWS - 1) / ROWS : 0;
    const int incl = wave_prefix((np << 16) | c);
    if (lane == 63) tot_lds[wave] = incl;
    __syncthreads();
    int before = incl - ((np << 16) | c), n_items = 0;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) {
        const int t = tot_lds[w];
        if (w < wave) before += t;
        n_items += t >> 16;
    }
    if (DISP) o = before & 0xffff;
    off_lds[tid] = o;
    for (int k = 0; k < np; ++k) {
        const int at = (before >> 16) + k;
        if (at < SHARE_MAX_ITEMS) item_lds[at] = (uint32_t)tid | ((uint32_t)k << 16);
    }
    __syncthreads();
    if (DISP) {
#pragma unroll
        for (int n = 0; n < NI; ++n) {
            if (id[n] >= 0) {
                const int i = (wave * NI + n) * 64 + lane;
                const int slot = off_lds[id[n]] + cntw_lds[wave][id[n]] + rank[n];
                list_lds[slot] = (uint16_t)((uint32_t)i / (uint32_t)p.K);
                // the slots for the kernels behind this one: batch b (of at most 64) by workgroup b
                if (wave * NI + n == (int)blockIdx.x) p.out_perm[i] = slot;
            }
        }
        if (blockIdx.x == 0 && tid < p.E) {
            p.out_counts[tid] = c;
            p.out_offsets[tid] = o;
            if (tid == p.E - 1) p.out_offsets[p.E] = o + c;
        }
        __syncthreads();
    }
    const int U = p.nchunks;                              // units per item
    const int total = __builtin_amdgcn_readfirstlane(min(n_items, SHARE_MAX_ITEMS)) * U;
    const int u0 = (int)((uint32_t)(total * share) / (uint32_t)n_share), u1 = (int)((uint32_t)(total * (share + 1)) / (uint32_t)n_share);
    if (u0 >= u1) return;

    const RawConsts rc = raw_consts();
    const global_char *src_c = (const global_char *)p.src;
    const int g0 = (ks * WK + kpart) * GW;              // first group of this wavefront
    const int last_item = (u1 - 1) / U;
    int item = u0 / U, in = u0 - item * U;

    // token rows of an item: B fragments, and per group the sums that take the codes' offsets and the zero point out.
    // The next item's rows are fetched one unit ahead where there are registers for it (GW <= 3).
    constexpr bool AHEAD = GW <= 3;
    half8_t bx[GW][4], bn[GW][4];
    float cxo[GW], cxs[GW];
    int mcnt = 0, base = 0;
    auto item_rows = [&](const int it_, int &base_, int &mcnt_) {
        const uint32_t it = __builtin_amdgcn_readfirstlane(item_lds[it_]);
        const int e = (int)(it & 0xffffu), m0 = (int)(it >> 16) * ROWS;
        base_ = __builtin_amdgcn_readfirstlane(off_lds[e]) + m0;
        mcnt_ = min(__builtin_amdgcn_readfirstlane(cnt_lds[e]) - m0, ROWS);
    };
    auto fetch_rows = [&](const int base_, const int mcnt_, half8_t (&dst)[GW][4]) {
        const int slot = base_ + (r < mcnt_ ? r : 0);         // rows past the last: their columns are never stored
        const int srow = MODE == 1 ? slot : (int)list_lds[slot];
        const uint32_t off = ((uint32_t)srow * (uint32_t)p.src_ld + (uint32_t)(g0 * ODSD_GROUP + kq * 8)) * 2u;
#pragma unroll
        for (int g = 0; g < GW; ++g)
#pragma unroll
            for (int j = 0; j < 4; ++j)
                dst[g][j] = __builtin_bit_cast(half8_t, *(const global_u4 *)(src_c + (off + g * (ODSD_GROUP * 2u) + j * 64u)));
    };
    auto group_sums = [&]() {
#pragma unroll
        for (int g = 0; g < GW; ++g) {
            float lo = 0.f, hi = 0.f;
            const half2_t one = {(half_t)1.0f, (half_t)1.0f};
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const half8_t f = bx[g][j];
                lo = __builtin_amdgcn_fdot2(half2_t{f[0], f[1]}, one, lo, false);
                hi = __builtin_amdgcn_fdot2(half2_t{f[2], f[3]}, one, hi, false);
                lo = __builtin_amdgcn_fdot2(half2_t{f[4], f[5]}, one, lo, false);
                hi = __builtin_amdgcn_fdot2(half2_t{f[6], f[7]}, one, hi, false);
            }
            lo += __shfl_xor(lo, 16, 64);
            hi += __shfl_xor(hi, 16, 64);
            lo += __shfl_xor(lo, 32, 64);
            hi += __shfl_xor(hi, 32, 64);
            cxo[g] = -(ODSD_RAW_OFFSET_LO * lo + ODSD_RAW_OFFSET_HI * hi);
            cxs[g] = lo + hi;
        }
    };
    auto rows_now = [&](const int it_) {
        item_rows(it_, base, mcnt);
        fetch_rows(base, mcnt, bx);
    };
    rows_now(item);

    // ---- weights: a ring of DEPTH steps, each a group's tiles of two blocks --------------------------------
    uint4_t wq[DEPTH][2], wsz[DEPTH][2];
    uint32_t q_voff = (uint32_t)lane * 16u, sz_voff = (uint32_t)kq * 16u;   // (scale, zero) in accumulator order: rows 4 kq ..
    const int n_q = p.NBLK * p.G * 1024, n_sz = p.NBLK * p.G * 64;
    int au = u0, a_in = in, a_item = item, a_tile = 0;    // the unit that the ring fetches
    __amdgpu_buffer_rsrc_t rq, rsz;
    auto ring_item = [&]() {
        const int e = (int)(__builtin_amdgcn_readfirstlane(item_lds[a_item]) & 0xffffu);
        const uint64_t eq = uniform_u64(tq_lds[e]), esz = uniform_u64(tsz_lds[e]);
        rq = __builtin_amdgcn_make_buffer_rsrc((void *)(uintptr_t)eq, 0, n_q, 0x00020000);
        rsz = __builtin_amdgcn_make_buffer_rsrc((void *)(uintptr_t)esz, 0, n_sz, 0x00020000);
    };
    // step s of the ring's unit: the codes first, (scale, zero) -- until then in use -- at the end of the step that
    // empties the slot
    auto load_codes = [&](const int slot, const int s) {
        a_tile = (a_in * UBLK + rsub * NB + s / GW * 2) * p.G + g0 + s % GW;
#pragma unroll
        for (int i = 0; i < 2; ++i)
            wq[slot][i] = __builtin_amdgcn_raw_buffer_load_b128(rq, (int)q_voff, (a_tile + i * p.G) * 1024, 2 /* nt */);
    };
    auto load_scales = [&](const int slot, const int s) {
#pragma unroll
        for (int i = 0; i < 2; ++i)
            wsz[slot][i] = __builtin_amdgcn_raw_buffer_load_b128(rsz, (int)sz_voff, (a_tile + i * p.G) * 64, 0);
        if (s == SPU - 1) {
            ++au;
            ++a_in;
            if (au >= u1) {
                // past the share's end: offsets beyond the resource, loads return zero without a fetch
                a_in = 0;
                q_voff = sz_voff = 0x80000000u;
            } else if (a_in == U) {
                a_in = 0;
                ++a_item;
                ring_item();
            }
        }
    };
    ring_item();
#pragma unroll
    for (int d = 0; d < DEPTH; ++d) {
        load_codes(d, d % SPU);
        load_scales(d, d % SPU);
    }
    group_sums();

    float4_t acc[NB];
    auto step = [&](const int slot, const int s) {
        const int g = s % GW, i0 = s / GW * 2;
        ODSD_FENCE();
        half8_t a[2][4];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            a[i][0] = raw_word(rc, wq[slot][i].x);
            a[i][1] = raw_word(rc, wq[slot][i].y);
            a[i][2] = raw_word(rc, wq[slot][i].z);
            a[i][3] = raw_word(rc, wq[slot][i].w);
        }
        // expanded here and not behind the refill (or the slot's registers would have to be copied)
#pragma unroll
        for (int i = 0; i < 2; ++i)
            asm volatile("" : "+v"(a[i][0]), "+v"(a[i][1]), "+v"(a[i][2]), "+v"(a[i][3]));
        ODSD_FENCE();
        load_codes(slot, (s + DEPTH) % SPU);
        ODSD_FENCE();
        __builtin_amdgcn_s_setprio(2);
        // the group's sum of q_k x_k: the accumulator starts at minus the offsets' share
        float4_t t[2];
        t[0] = t[1] = float4_t{cxo[g], cxo[g], cxo[g], cxo[g]};
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int i = 0; i < 2; ++i)
                t[i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[i][j], bx[g][j], t[i], 0, 0, 0);
        // w = (q - zero) * scale per output row: acc += scale * (sum q x - zero * sum x)
        const float xs = cxs[g];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const uint4_t z = wsz[slot][i];
            const half2_t p0 = as_half2(z.x), p1 = as_half2(z.y), p2 = as_half2(z.z), p3 = as_half2(z.w);
            const float4_t b = g == 0 ? float4_t{0.f, 0.f, 0.f, 0.f} : acc[i0 + i];
            acc[i0 + i].x = __builtin_fmaf((float)p0.x, __builtin_fmaf(-(float)p0.y, xs, t[i].x), b.x);
            acc[i0 + i].y = __builtin_fmaf((float)p1.x, __builtin_fmaf(-(float)p1.y, xs, t[i].y), b.y);
            acc[i0 + i].z = __builtin_fmaf((float)p2.x, __builtin_fmaf(-(float)p2.y, xs, t[i].z), b.z);
            acc[i0 + i].w = __builtin_fmaf((float)p3.x, __builtin_fmaf(-(float)p3.y, xs, t[i].w), b.w);
        }
        // (arithmetic has no memory side: its results are tied to the fence)
#pragma unroll
        for (int i = 0; i < 2; ++i)
            asm volatile("" : "+v"(acc[i0 + i].x), "+v"(acc[i0 + i].y), "+v"(acc[i0 + i].z), "+v"(acc[i0 + i].w));
        __builtin_amdgcn_s_setprio(0);
        ODSD_FENCE();
        load_scales(slot, (s + DEPTH) % SPU);
        ODSD_FENCE();
    };

    // ---- sums over the parts -------------------------------------------------------------------------------
    // position of a lane's 4 sums in an accumulator tile: rows rotated by 4 per kq, so that the readers' 4 rows x
    // 16 outputs fall on 64 different banks
    const int red_w = (kq * 16 + ((r + 4 * kq) & 15)) * 4;
    const int rd_comp = lane & 3, rd_kq = (lane >> 2) & 3, rd_r = lane >> 4;
    constexpr int QUADS = (MODE == 0 ? 1 : UBLK) * 4;   // 4 rows x 16 outputs each
    int turn = 0;                                         // which wavefronts sum up: moves on with the unit
    auto finish = [&]() {
        const int buf = turn & 1;
#pragma unroll
        for (int i = 0; i < NB; ++i) *(float4_t *)&red[buf][kpart][rsub * NB + i][red_w] = acc[i];
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        turn = (turn + WAVES - 1) % WAVES;
        // quads by rows, then blocks: with few rows the first ones are all there are
#pragma unroll
        for (int t = 0; t < (QUADS + WAVES - 1) / WAVES; ++t) {
            const int q = (wave + turn) % WAVES + t * WAVES;
            const int blk = MODE == 0 ? 0 : q % UBLK, row4 = (MODE == 0 ? q : q / UBLK) * 4;
            if (q >= QUADS || row4 >= mcnt) break;
            const int row = row4 + rd_r;
            const int at = (rd_kq * 16 + ((row + 4 * rd_kq) & 15)) * 4 + rd_comp;
            float v = 0.f, up = 0.f;
#pragma unroll
            for (int k = 0; k < WK; ++k) {
                v += red[buf][k][blk][at];
                if (MODE == 0) up += red[buf][k][1][at];
            }
            if (row < mcnt) {
                const int o = ((MODE == 0 ? 0 : ks * p.P) + base + row) * p.ldo + (MODE == 0 ? in : in * UBLK + blk) * 16 + rd_kq * 4 + rd_comp;
                if (MODE == 0) p.h16[o] = f32_to_f16_sat(silu_f32(v) * up);
                else if (p.y_f16) ((half_t *)p.y)[o] = f32_to_f16_sat(v);
                else p.y[o] = v;
            }
        }
    };

    // ---- the stream ------------------------------------------------------------------------------------------
    // One loop with one exit and one copy of a unit (unrolled trips and what is left behind them cost a first pass 7 us in
    // instruction fetches, and a break between two units would count as a way back to the loop's top: the wait counts
    // there would allow for the ring as that way leaves it).
    int base_n = 0, mcnt_n = 0;
    for (int left = u1 - u0; left > 0; --left) {
        if (in == U) {
            in = 0;
            ++item;
            if constexpr (AHEAD) {
                base = base_n;
                mcnt = mcnt_n;
#pragma unroll
                for (int g = 0; g < GW; ++g)
#pragma unroll
                    for (int j = 0; j < 4; ++j) bx[g][j] = bn[g][j];
                group_sums();
            } else {
                rows_now(item);
                group_sums();
                // nothing of the rows is outstanding from here on, whichever way was taken (or the wait counts
                // of the stream would have to allow for it, at the cost of half the ring)
                ODSD_WAIT_VMCNT(0);
            }
        }
        if constexpr (AHEAD)
            if (in == U - 1 && item < last_item) {
                item_rows(item + 1, base_n, mcnt_n);
                fetch_rows(base_n, mcnt_n, bn);
            }
#pragma unroll
        for (int s = 0; s < SPU; ++s) step(s % DEPTH, s);
        finish();
        ++in;
    }
}

// ---- host side -----------------------------------------------------------------------------------
// How the wavefronts of a workgroup split a reduction of G groups: WK parts of GW groups, KS splits across workgroups.
// The token rows of a part live in registers, 16 GW of them (207 in all at GW = 3, where the next item's rows are fetched
// ahead, 194 at GW = 4): 2 to 4 groups.  One group per part would make a unit of gate_up a single step, with a barrier
// every 2 KiB of a wavefront's stream.  gate_up (8 parts, both blocks of a unit): 16, 24 or 32 groups.  down: the most
// parts that divide the reduction, two groups before three, and what is left over across workgroups.
// Layer, us, the plan without equal shares / this: H = 3072, E = 128, I = 768, K = 8: T = 1 34.1 / 25.3, T = 64 102.5 / 93.4,
// T = 176 114.6 / 111.4; H = 2048, I = 512, E = 512, K = 10, T = 64 166 / 119; I = 1024, E = 64, K = 8: T = 8 53.3 / 42.6,
// T = 88 63.1 / 58.6; I = 2560 (5 splits), E = 16, K = 2: T = 8 37.8 / 30.1, T = 88 47.9 / 43.4; H = 4096, I = 3072, E = 32,
// K = 2: T = 24 116 / 93; I = 5632 (11 splits), E = 16: T = 24 125 / 104, T = 88 130 / 126.
struct ShareSplit { int WK, GW, KS; };
static bool share_split(int mode, int G, ShareSplit *s) {
    if (mode == 0) {
        if (G % 8 || G < 16 || G > 32) return false;
        *s = {8, G / 8, 1};
        return true;
    }
    static const int parts[][2] = {{8, 2}, {8, 3}, {4, 3}, {4, 2}, {2, 3}, {2, 2}};
    for (const auto &w : parts)
        if (G % (w[0] * w[1]) == 0 && G / (w[0] * w[1]) <= 16) {
            *s = {w[0], w[1], G / (w[0] * w[1])};
            return true;
        }
    return false;
}

int odsd_share_supported(int H, int I, int E, int P) {
    ShareSplit u, d;
    return share_split(0, H / ODSD_GROUP, &u) && share_split(1, I / ODSD_GROUP, &d) && E <= 64 * SHARE_WAVES &&
           P <= SHARE_MAX_P && E + P / 16 <= SHARE_MAX_ITEMS;
}
// The top-k in gate_up's prologue, a token per wavefront: every workgroup repeats it, which costs less than the launch
// it saves up to 8 tokens (layer, us, separate / inside: E = 128, H = 2048: T = 1 24.5 / 22.8, T = 8 42.5 / 41.7, T = 9
// 44.1 / 44.7, T = 16 51.9 / 53.6; E = 8, H = 4096: T = 1 49.9 / 48.4, T = 5 99.4 / 97.2, T = 8 116.3 / 114.8).
int odsd_share_route_supported(int T, int E) { return T <= SHARE_WAVES && E <= 128; }
int odsd_share_down_splits(int I) {
    ShareSplit s;
    return share_split(1, I / ODSD_GROUP, &s) ? s.KS : 0;
}

#define SHARE_CUS 256
template <int MODE, int GW, int WK, int DEPTH>
static void share_go(GemmParams &gp, int KS, hipStream_t st) {
    constexpr int NB = 2;
    gp.nchunks = gp.NBLK / (SHARE_WAVES / WK * NB);        // units per item
    gp.n_wg = SHARE_CUS / KS * KS;
#define SHARE_GO(NI, ROUTE)                                                                                        \
    ODSD_LAUNCH(MODE == 0 ? ODSD_KERNEL_GATE_UP : ODSD_KERNEL_DOWN, (w4_share_kernel<MODE, GW, WK, NB, DEPTH, NI, ROUTE>), \
                gp.n_wg, 64 * SHARE_WAVES, st, gp)
    if constexpr (MODE == 0) {
        if (gp.idx) {
            if (gp.route_S > 0 && gp.E <= 64) SHARE_GO(1, 1);          // (at most 8 tokens of 64 choices)
            else if (gp.route_S > 0) SHARE_GO(1, 2);
            else if (gp.P <= 512) SHARE_GO(1, 0);
            else if (gp.P <= 1024) SHARE_GO(2, 0);
            else SHARE_GO(SHARE_MAX_P / 512, 0);
            return;
        }
    }
    SHARE_GO(0, 0);
#undef SHARE_GO
}

// Steps in flight per wavefront (2 KiB each): 2 to 4, as many as a unit has, so that every unit begins on ring slot 0.  More
// did not stream faster in an earlier form whose ring ran on over several units (H = 2048, I = 768, T = 24: gate_up
// 2 / 3 / 4 / 6 steps 27.5 / 27.8 / 27.8 / 28.7 us; down 3 / 4 / 6 17.7 / 17.9 / 18.8).
void odsd_launch_share(int mode, GemmParams &gp, hipStream_t st) {
    ShareSplit s;
    if (!share_split(mode, gp.G, &s)) return;
    if (mode == 0) {
        if (s.GW == 2) share_go<0, 2, 8, 2>(gp, s.KS, st);
        else if (s.GW == 3) share_go<0, 3, 8, 3>(gp, s.KS, st);
        else share_go<0, 4, 8, 4>(gp, s.KS, st);
    } else if (s.GW == 2) {
        if (s.WK == 2) share_go<1, 2, 2, 2>(gp, s.KS, st);
        else if (s.WK == 4) share_go<1, 2, 4, 2>(gp, s.KS, st);
        else share_go<1, 2, 8, 2>(gp, s.KS, st);
    } else {
        if (s.WK == 2) share_go<1, 3, 2, 3>(gp, s.KS, st);
        else if (s.WK == 4) share_go<1, 3, 4, 3>(gp, s.KS, st);
        else share_go<1, 3, 8, 3>(gp, s.KS, st);
    }
}
