// Causal attention over cached or packed keys with few query rows per sequence: the decode / verify
// step over the paged KV cache, and packed calls that the prefill kernel does not take.
//
// A query row is one (token, query head) pair of a KV head's group; up to 16, 32 or 64 rows of one
// (sequence, KV head) -- a unit -- are worked on together, so one pass over the keys serves a whole group
// of query heads and all draft tokens.  What the kernels have to do is stream K and V from HBM.  The keys
// of all units are laid end to end and dealt out in equal contiguous shares to 512 workgroups, two per
// CU.  A share may begin and end in the middle of a unit: such pieces leave partial results
// that a second kernel merges, whole units are finished in place.  Sequences of mixed lengths then cost
// what their bytes cost; with a fixed number of slices per sequence, as before, the longest sequence set
// the time.  Two forms:
//   * up to 16 rows (decode; 32 with a lot of keys), attn_stream_kernel: each of the 4 wavefronts takes
//     its own 32 keys of every 128, for all rows of the unit, with no barrier in the loop.  K goes from
//     memory straight into the registers that S^T = K Q^T wants as its A operand (v_mfma_f32_16x16x32); V
//     goes through a piece of LDS that belongs to the wavefront, because O^T = V^T P^T needs its transpose
//     (ds_read_b64_tr_b16).  A tile's registers are refilled as soon as it has been multiplied (K) or put
//     into LDS (V); what is left of the latency is hidden by two wavefronts per SIMD, three (what registers and
//     LDS allow) where nothing is split;
//   * more rows, attn_tile_kernel: a wavefront cannot hold the rows next to its keys, so the workgroup
//     shares the keys through LDS.
// In both the scores of one query row stay in the 4 lanes that share lane % 16, in the order in which P^T
// is wanted as the B operand, and O^T keeps the row there too: maximum, sum and rescaling factor are lane
// values.  Softmax in fp32 in the exp2 domain; a row's reference point follows its running maximum lazily.
// Measured (32 query / 4 KV heads of 128, bf16, kernel + merge, before -> now): 64 sequences of 750 to 3000
// keys, one query each, 263 MB: 64.1 -> 47.5 us (the kernel alone 6.1 TB/s: bound by HBM); 64 of 2048
// keys 53.3 -> 45.9; one of 4000 13.9 -> 13.0; 16 of 300 13.3 -> 7.7 (no merge).  32 sequences of 512 to 2048
// keys x 8 queries, 85 MB: 31.8 -> 30.8: start-up, pieces and merge are as long as the stream there.  Block sizes that
// are no multiple of 32 (ALIGNED false) spill 28 bytes per lane at head size 128 and still gain: block size 16, 64
// sequences of 750 to 3000 keys 68.5 -> 61.6, of 125 to 500 18.1 -> 13.6, with 32 / 8 heads 115 -> 106.5.
//
// Paged form: the cache is addressed through the sequence's block table exactly as the reference
// gathers it: position p lives in slot block_table[p / block_size] * block_size + p % block_size.
// Packed form: the keys of sequence s are rows cu_seqlens_k[s] .. of k / v.
//
// Replaces Qwen3Attention._fallback_decode_attention (demo/src/layers/attention.py:290-352: gather
// of the cached K/V by slot, repeat_interleave for GQA, causal mask with offset k_len - q_len,
// scaled_dot_product_attention), the flash_attn_with_kvcache call it stands in for (:252-272) and
// the flash_attn_varlen_func call of the prefill branch (:229-240).
#include "attn.h"
#include "w4_gemm.h"
#include <type_traits>

#define ATTN_WG 512          // workgroups that share the work: two per CU
// Granularities of the list in keys: it is cut at multiples of FINE when that gives every workgroup at least
// COARSE keys, otherwise at multiples of COARSE; with no sequence longer than WHOLE nothing is split and
// there is nothing to merge.  (A merge costs 4 to 6 us, what a workgroup needs for WHOLE keys: 16 sequences
// of 300 keys, decode, 7.7 us whole against 10.2 split.)  With more units nothing is split up to more
// keys, and with MANY never: they fill the chip and level mixed lengths out by themselves.  (attn_keep_whole;
// 32 / 4 heads of 128, split / whole, us.  Stream form: 40 sequences of up to 700 keys 15.2 / 12.6, 64 of 1000
// 21.1 / 18.8, 384 of 700 67.9 / 58.2, but 128 of 2000 59.7 / 62.2.  Tile form, 8 queries each: 16 of 300 15.0 /
// 11.3, of 700 17.5 / 19.3; 32 of 700 20.4 / 19.5, of 1000 21.4 / 25.6; 48 of 1000 29.4 / 25.8, of 1500 34.1 / 40.3; 64 of
// 1500 42.4 / 42.3; 96 of 2000 80 / 72; 128 of 700 48.3 / 28.9, of 2000 101 / 83; 256 of 1500 158 / 121.)
#define ATTN_STREAM_FINE 128
#define ATTN_STREAM_COARSE 128
#define ATTN_STREAM_WHOLE 512
#define ATTN_TILE_FINE 32
#define ATTN_TILE_COARSE 256
#define ATTN_TILE_WHOLE 256
#define ATTN_MANY (4 * ATTN_WG)
#define ATTN_XCD_GROUP 8     // row groups of a (sequence, KV head) that go to one XCD together, at most

// ---- how the work is dealt out -----------------------------------------------------------------------
// A sequence is KVH * rg units, each of `steps` list steps of g keys (a sequence without keys still owns
// output rows, which are written as zeros: one step).  A sequence takes no more of the list than the host sized
// the launch for: a context longer than its table is walked by the last step of its units, and row groups
// past the bound on the query lengths are left out, so that the others' shares stay where they are.
struct SeqCost {
    int L, ql, rg, steps, cost;
};
__device__ __forceinline__ void seq_steps(const AttnParams &p, SeqCost &c, const int g) {
    c.steps = max(1, (min(c.L, p.max_keys) + g - 1) / g);
    c.cost = c.rg * p.KVH * c.steps;
}
__device__ __forceinline__ SeqCost seq_cost(const AttnParams &p, const int s, const int rows_per_unit, const int g) {
    SeqCost c{0, 0, 0, 0, 0};
    if (s < p.n_seqs) {
        if (p.cu_k) {
            c.L = p.cu_k[s + 1] - p.cu_k[s];
            c.ql = p.cu_q[s + 1] - p.cu_q[s];
        } else {
            c.L = p.context_lens[s];
            c.ql = p.q_lens ? p.q_lens[s] : 1;
        }
        c.ql = max(c.ql, 0);
        c.rg = min((c.ql * p.Gq + rows_per_unit - 1) / rows_per_unit, p.max_rg);
        seq_steps(p, c, g);
    }
    return c;
}
// inclusive prefix sum over the wavefront
__device__ __forceinline__ int wave_scan(int v) {
#define ATTN_SCAN(CTRL, ROWMASK) v += __builtin_amdgcn_update_dpp(0, v, CTRL, ROWMASK, 0xF, false)
    ATTN_SCAN(0x111, 0xF);   // row_shr:1, 2, 4, 8
    ATTN_SCAN(0x112, 0xF);
    ATTN_SCAN(0x114, 0xF);
    ATTN_SCAN(0x118, 0xF);
    ATTN_SCAN(0x142, 0xA);   // row_bcast:15 into rows 1 and 3
    ATTN_SCAN(0x143, 0xC);   // row_bcast:31 into rows 2 and 3
#undef ATTN_SCAN
    return v;
}
__device__ __forceinline__ int lane_value(int v, int lane) { return __builtin_amdgcn_readlane(v, lane); }

// Where a sequence stands in the list: found either by a position in the list or by its number.
struct SeqAt {
    int seq, L, ql, rg, steps;
    int first;       // list position of its first step
    int q0;          // its first query token (packed form: cu_q[seq], wherever the offsets begin)
};
struct ListPlan {
    int g;                   // keys per list step
    int total, share;        // steps in all, steps per workgroup
    SeqAt at;
    int me;                  // the share (unit) that is this workgroup's
    bool found;
};
// Workgroups go round the 8 XCDs, each with an L2 of its own, and the row groups of a (sequence, KV head) read the same
// keys.  Unsplit units: `group` neighbours of the list go to workgroups that are 8 apart, in whole periods of 8 groups
// (what is left at the end stays as it is), so that the groups still go round.  (32 / 4 heads of 128, 8 queries a row group, us,
// workgroup = unit or share / so: unsplit, 64 sequences of 1024 keys x 16 queries 40.2 / 35.9, 100 of 900 x 12 55.7 / 45.0; split, 8
// of 3000 x 16 29.3 / 27.9, x 40 43.9 / 40.8, 30 of 1777 x 9 39.2 / 38.4; one row group each: no difference.)
__device__ __forceinline__ int unit_of_workgroup(const int wg, const int n, const int group) {
    if (group <= 1) return wg;
    const int period = 8 * group, o = wg % period;
    return wg - o + period > n ? wg : wg - o + (o & 7) * group + (o >> 3);
}
// Shares, which cost the same: a contiguous eighth of the `used` ones to each XCD, so that the pieces of a unit and the units of
// a sequence are neighbours there.  Not below `used`: a workgroup without a share.  Shares of one step stay as they are (9 sequences
// of 1225 keys x 24 24.3 / 25.0; others no difference).  With more, as above; two of 15 such lose (2 of 1939 x 160, 16 / 2 heads, 26.2 / 27.0,
// 7 of 1294 x 24, 64 / 4 heads of 64, 22.9 / 23.7).
__device__ __forceinline__ int share_of_workgroup(const int wg, const int used) {
    if (wg >= used) return wg;
    const int q = used >> 3, r = used & 7, x = wg & 7;
    return x * q + min(x, r) + (wg >> 3);
}
// fine, coarse: the two granularities.  The list is cut at multiples of `fine` keys when every workgroup gets at
// least `coarse` keys that way; otherwise at multiples of `coarse`, so that short units stay whole.
// SPLIT, UNSPLIT: the launches that the caller is compiled for (p.whole: its direct way to the unit).  BY_XCD: `who` is a
// workgroup, and its share or unit is chosen by the two functions above.
template <bool BY_SEQ, bool SPLIT, bool UNSPLIT, bool BY_XCD = false>
__device__ __forceinline__ ListPlan list_plan(const AttnParams &p, const int rows_per_unit, const int fine,
                                              const int coarse, int who) {
    const int lane = lane_id();
    ListPlan pl;
    if (BY_XCD && !SPLIT) who = unit_of_workgroup(who, p.n_wg, min(p.max_rg, ATTN_XCD_GROUP));
    pl.me = who;
    if (UNSPLIT && p.whole) {
        // A workgroup per (sequence, KV head, row group that a sequence can have), found without the list: with
        // 512 sequences its scan cost every workgroup two rounds of 8 dependent loads (MANY, below).
        pl.g = 1 << 30;                       // (longer than any sequence: one step per unit, whatever its length)
        pl.total = 0x7fffffff;
        pl.share = 1;
        const int per_seq = p.KVH * p.whole, s = who / per_seq, l = who - s * per_seq;
        // (the query lengths before s in front of everything that waits for the sequence's own)
        int tok = 0;
        if (!p.cu_k && p.q_lens)
            for (int i = lane; i < s; i += 64) tok += max(p.q_lens[i], 0);
        const SeqCost c = seq_cost(p, s, rows_per_unit, pl.g);
        pl.found = l < __builtin_amdgcn_readfirstlane(c.cost);
        if (p.cu_k) tok = p.cu_q[s];
        else tok = p.q_lens ? lane_value(wave_scan(tok), 63) : s;
        pl.at = SeqAt{s, __builtin_amdgcn_readfirstlane(c.L), __builtin_amdgcn_readfirstlane(c.ql),
                      __builtin_amdgcn_readfirstlane(c.rg), 1, who - l, __builtin_amdgcn_readfirstlane(tok)};
        return pl;
    }
    pl.g = SPLIT ? fine : 1 << 30;                        // (unsplit: each unit is one step)
    SeqCost c0 = seq_cost(p, lane, rows_per_unit, pl.g);
    int s0, total;
    for (;;) {
        s0 = wave_scan(c0.cost);
        total = lane_value(s0, 63);
        for (int b = 64; b < p.n_seqs; b += 64)
            total += lane_value(wave_scan(seq_cost(p, b + lane, rows_per_unit, pl.g).cost), 63);
        if (!SPLIT || pl.g == coarse || total >= (coarse / fine) * p.n_wg) break;
        pl.g = coarse;
        seq_steps(p, c0, coarse);
    }
    pl.total = total;
    pl.share = max(1, (total + p.n_wg - 1) / p.n_wg);
    pl.found = false;
    if (BY_XCD && SPLIT && pl.share > 1) pl.me = who = share_of_workgroup(who, (total + pl.share - 1) / pl.share);
    const int target = BY_SEQ ? 0 : who * pl.share;
    if (!BY_SEQ && target >= total) return pl;
    int before = 0, tok = 0;
    SeqCost c = c0;
    int sc = s0;
    for (int b = 0; b < p.n_seqs; b += 64) {
        if (b > 0) {
            c = seq_cost(p, b + lane, rows_per_unit, pl.g);
            sc = wave_scan(c.cost);
        }
        const int tc = wave_scan(c.ql);
        const int sum = lane_value(sc, 63);
        if (BY_SEQ ? who < b + 64 : target < before + sum) {
            const int l = BY_SEQ ? who - b : __builtin_ctzll(__ballot(before + sc > target));
            pl.at = SeqAt{b + l, lane_value(c.L, l), lane_value(c.ql, l), lane_value(c.rg, l), lane_value(c.steps, l),
                          before + lane_value(sc, l) - lane_value(c.cost, l),
                          p.cu_k ? __builtin_amdgcn_readfirstlane(p.cu_q[b + l]) : tok + lane_value(tc, l) - lane_value(c.ql, l)};
            pl.found = true;
            return pl;
        }
        before += sum;
        tok += lane_value(tc, 63);
    }
    return pl;
}

// the unit after this one: of the same sequence, or of the next one that has any
__device__ __forceinline__ void next_unit(const AttnParams &p, SeqAt &sq, int &unit, int &step, const int rows_per_unit,
                                          const int g) {
    step = 0;
    if (++unit < p.KVH * sq.rg) return;
    unit = 0;
    sq.first += p.KVH * sq.rg * sq.steps;
    do {                                                   // (a sequence without queries has no units)
        ++sq.seq;
        sq.q0 = p.cu_k ? __builtin_amdgcn_readfirstlane(p.cu_q[sq.seq]) : sq.q0 + sq.ql;
        const SeqCost nx = seq_cost(p, sq.seq, rows_per_unit, g);
        sq.L = __builtin_amdgcn_readfirstlane(nx.L);
        sq.ql = __builtin_amdgcn_readfirstlane(nx.ql);
        sq.rg = __builtin_amdgcn_readfirstlane(nx.rg);
        sq.steps = __builtin_amdgcn_readfirstlane(nx.steps);
    } while (sq.rg == 0);
}

// ---- one 32-key tile of 16 query rows -----------------------------------------------------------------
// Lane (c, kq) holds the scores of keys 16 t + 4 kq + i of query row c (a[4 t + i], before the softmax
// scale, masked ones -inf); returns the probabilities as the B operand of O^T = V^T P^T and keeps the row's
// reference point, this lane's part of its sum, and O^T.  The reference point moves only when some score of
// the wavefront exceeds it by more than 2^8 (probabilities up to 256 are as exact in fp16 / bf16 as those
// below 1, and the sums are fp32): most tiles then need no exchange between lanes at all.
template <typename T, int NDB>
__device__ __forceinline__ typename AttnT<T>::V8 softmax_tile(const float (&a)[8], const float sc, float &m_run,
                                                              float &l_run, float4_t (&o)[NDB]) {
    float mx = fmaxf(fmaxf(fmaxf(a[0], a[1]), fmaxf(a[2], a[3])), fmaxf(fmaxf(a[4], a[5]), fmaxf(a[6], a[7])));
    if (__any(mx * sc > m_run + 8.0f)) {
        mx = fmaxf(mx, __shfl_xor(mx, 16, ODSD_WAVE));
        mx = fmaxf(mx, __shfl_xor(mx, 32, ODSD_WAVE));
        const float m_new = fmaxf(m_run, mx * sc);
        // a row with nothing to attend yet keeps m = -inf: use 0 as the reference point then
        const float alpha = __builtin_amdgcn_exp2f(m_run - (m_new == -INFINITY ? 0.0f : m_new));   // m_run = -inf -> 0
        l_run *= alpha;
        m_run = m_new;
#pragma unroll
        for (int db = 0; db < NDB; ++db) { o[db].x *= alpha; o[db].y *= alpha; o[db].z *= alpha; o[db].w *= alpha; }
    }
    const float neg_ref = m_run == -INFINITY ? 0.0f : -m_run;
    float pe[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) pe[e] = __builtin_amdgcn_exp2f(fmaf(a[e], sc, neg_ref));   // masked -> 0
    l_run += ((pe[0] + pe[1]) + (pe[2] + pe[3])) + ((pe[4] + pe[5]) + (pe[6] + pe[7]));
    return __builtin_bit_cast(typename AttnT<T>::V8,
                              uint4_t{AttnT<T>::pack2(pe[0], pe[1]), AttnT<T>::pack2(pe[2], pe[3]),
                                      AttnT<T>::pack2(pe[4], pe[5]), AttnT<T>::pack2(pe[6], pe[7])});
}
// A operand of O^T = V^T P^T: this lane's dimension of keys 4 kq .. + 3 (at `at`) and 16 + 4 kq .. + 3
// (`further` bytes on), the keys of the lane's 8 probabilities
template <typename V8>
__device__ __forceinline__ V8 read_vt(const char *at, const int further) {
    typedef short s4_t __attribute__((ext_vector_type(4)));
    typedef short s8_t __attribute__((ext_vector_type(8)));
    typedef __attribute__((address_space(3))) s4_t lds_s4;
    const s4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4 *)at);
    const s4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4 *)(at + further));
    return __builtin_bit_cast(V8, s8_t{lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w});
}

template <typename T, int HD, int RB, bool ALIGNED>
__global__ __launch_bounds__(256, RB == 1 ? 3 : 2) void attn_stream_kernel(const AttnParams p) {
    typedef typename AttnT<T>::V8 V8;
    constexpr int NJ = HD / 32;          // 32-dim steps of the score product
    constexpr int NDB = HD / 16;         // 16-dim blocks of the output
    constexpr int NP = HD / 8;           // 16-byte pieces of a row
    constexpr int NV = 32 * NP / 64;     // 16-byte pieces of a 32-key V tile per lane
    constexpr int RPI = 64 / NP;         // rows per V load
    constexpr int ROWS = 16 * RB;        // rows of a unit
    constexpr int STEP = 128;            // keys of a turn, 32 per wavefront
    constexpr int VT = 32 * HD * 2;      // bytes of a V tile
    constexpr int XROW = HD + 4;         // floats per row of the exchange area (and of partial results)
    constexpr int LDS_BYTES = 4 * ROWS * XROW * 4 > 4 * VT ? 4 * ROWS * XROW * 4 : 4 * VT;
    __shared__ __attribute__((aligned(16))) char lds[LDS_BYTES];   // V tiles, one per wavefront; then the exchange
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int c = lane & 15, kq = lane >> 4;
    char *vt = lds + wave * VT;
    float *xch = (float *)lds;
    auto vswz = [](int key) { return HD == 128 ? (key & 7) : ((key >> 1) & 3); };

    const ListPlan pl = list_plan<false, true, true>(p, ROWS, ATTN_STREAM_FINE, ATTN_STREAM_COARSE, blockIdx.x);
    if (!pl.found) return;
    int pos = blockIdx.x * pl.share;                       // list position of the next step
    const int end = min(pl.total, pos + pl.share);
    SeqAt sq = pl.at;
    int unit = (pos - sq.first) / sq.steps;                // unit of the sequence, step inside the unit
    int step = (pos - sq.first) - unit * sq.steps;

    const int D = p.KVH * HD;
    const float sc = p.scale_log2e;
    const uint32_t rowb = (uint32_t)(D * 2);
    const char *kc = (const char *)p.k_cache, *vc = (const char *)p.v_cache;
    // V tile in LDS as stored, 32-byte segments of a row XORed with vswz(key): where this lane's pieces go ...
    const int vrow0 = lane / NP, vpc = lane % NP;
    // (vswz(RPI u + vrow0): with 4 rows per load the odd ones differ by 4, with 8 all are alike)
    const uint32_t vw_at[2] = {(uint32_t)(vrow0 * HD * 2 + ((vpc >> 1) ^ vswz(vrow0)) * 32 + (vpc & 1) * 16),
                               (uint32_t)(vrow0 * HD * 2 + ((vpc >> 1) ^ vswz(vrow0 + RPI)) * 32 + (vpc & 1) * 16)};
    // ... and where it reads: dims 16 db + c of keys 4 kq .. + 3 (lane c of a group of 16 addresses key c / 4, 4 dims)
    const int rkey = 4 * kq + (c >> 2);
    uint32_t vr_at[NDB];
#pragma unroll
    for (int db = 0; db < NDB; ++db) vr_at[db] = (uint32_t)(rkey * HD * 2 + (db ^ vswz(rkey)) * 32 + (c & 3) * 8);

    while (pos < end) {
        // ---- one piece: steps step .. step + n - 1 of one unit ----------------------------------------
        const int n = min(end - pos, sq.steps - step);
        const int kvh = unit / sq.rg, rg = unit - kvh * sq.rg;
        const int L = sq.L, ql = sq.ql, k_last = L - 1;
        const int rows_total = ql * p.Gq, row0 = rg * ROWS;
        const int rows_here = min(ROWS, rows_total - row0);
        const int k_start = p.cu_k ? __builtin_amdgcn_readfirstlane(p.cu_k[sq.seq]) : 0;
        const int32_t *bt = p.block_tables + (size_t)sq.seq * p.max_blocks;

        V8 qf[RB][NJ];
        int kmax[RB];                                      // last position that row attends
#pragma unroll
        for (int rb = 0; rb < RB; ++rb) {
            const int row = row0 + 16 * rb + c;
            const bool ok = row < rows_total;
            const int tok = ok ? row / p.Gq : 0, hq = ok ? row - tok * p.Gq : 0;
            kmax[rb] = ok ? L - ql + tok : -1;
            const uint16_t *qp = (const uint16_t *)p.q + ((size_t)(sq.q0 + tok) * p.H + kvh * p.Gq + hq) * HD + 8 * kq;
#pragma unroll
            for (int j = 0; j < NJ; ++j) {
                uint4_t raw = {0u, 0u, 0u, 0u};
                if (ok) raw = *(const uint4_t *)(qp + 32 * j);
                qf[rb][j] = __builtin_bit_cast(V8, raw);
            }
        }
        const int kmin = L - ql + row0 / p.Gq;            // the unit's first row: tiles that end at or before it need no mask

        float m_run[RB], l_run[RB];
        float4_t o[RB][NDB];
#pragma unroll
        for (int rb = 0; rb < RB; ++rb) {
            m_run[rb] = -INFINITY;
            l_run[rb] = 0.0f;
#pragma unroll
            for (int db = 0; db < NDB; ++db) o[rb][db] = float4_t{0.f, 0.f, 0.f, 0.f};
        }

        // this wavefront's tiles: 32 keys from 32 * wave on, every STEP; 64 of them at a time (their
        // table entries sit one per lane)
        const char *kh = kc + kvh * (HD * 2), *vh = vc + kvh * (HD * 2);
        const int key_end = step + n == sq.steps ? L : pl.g * (step + n);
        for (int key0 = pl.g * step + 32 * wave; key0 < key_end; key0 += 64 * STEP) {
            const int nt = min(64, (key_end - key0 + STEP - 1) / STEP);
            // ALIGNED: the slot of each tile's first key and the last row of the tile that may be read, one
            // tile per lane (an entry that is negative or beyond the cache reads slot 0)
            int slot_l = 0, lim_l = 0;
            if constexpr (ALIGNED) {
                const int kp = min(key0 + STEP * lane, k_last & ~31);
                if (p.cu_k) {
                    slot_l = k_start + kp;
                    lim_l = k_last - kp;
                } else {
                    const int blk = kp / p.block_size;
                    const int32_t b = bt[min(blk, p.max_blocks - 1)];
                    const bool ok = b >= 0 && blk < p.max_blocks && ((int64_t)b + 1) * p.block_size <= p.num_slots;
                    slot_l = ok ? b * p.block_size + (kp - blk * p.block_size) : 0;
                    lim_l = ok ? k_last - kp : 0;
                }
            }
            // !ALIGNED: lane l (and l + 32) looks up the slot of key l of a tile, one tile ahead of its fetch
            auto entry = [&](const int i) -> int {
                const int pc = min(key0 + STEP * i + (lane & 31), k_last);
                return bt[min(pc / p.block_size, p.max_blocks - 1)];
            };
            auto slot_of = [&](const int i, const int b) -> int {
                const int pc = min(key0 + STEP * i + (lane & 31), k_last);
                const int blk = pc / p.block_size;
                const int64_t sl = (int64_t)b * p.block_size + (pc - blk * p.block_size);
                return (b >= 0 && blk < p.max_blocks && sl < p.num_slots) ? (int)sl : 0;
            };
            uint4_t kreg[2][NJ], vreg[NV];
            int pend = 0, slot_v = 0;
            auto fetch_k = [&](const int i) {
                if constexpr (ALIGNED) {
                    const uint32_t lim = (uint32_t)lane_value(lim_l, i);
                    const char *kb = kh + (uint64_t)(uint32_t)lane_value(slot_l, i) * rowb;
#pragma unroll
                    for (int t = 0; t < 2; ++t) {
                        const uint32_t off = min((uint32_t)(16 * t + c), lim) * rowb + kq * 16u;
#pragma unroll
                        for (int j = 0; j < NJ; ++j) kreg[t][j] = *(const uint4_t *)(kb + off + 64 * j);
                    }
                } else {
                    slot_v = slot_of(i, pend);
                    pend = entry(i + 1);
#pragma unroll
                    for (int t = 0; t < 2; ++t) {
                        const uint32_t s = (uint32_t)__shfl(slot_v, 16 * t + c, ODSD_WAVE);
                        const char *kb = kh + (uint64_t)s * rowb + kq * 16;
#pragma unroll
                        for (int j = 0; j < NJ; ++j) kreg[t][j] = *(const uint4_t *)(kb + 64 * j);
                    }
                }
            };
            auto fetch_v = [&](const int i) {      // (after fetch_k of the same tile)
                if constexpr (ALIGNED) {
                    const uint32_t lim = (uint32_t)lane_value(lim_l, i);
                    const char *vb = vh + (uint64_t)(uint32_t)lane_value(slot_l, i) * rowb;
#pragma unroll
                    for (int u = 0; u < NV; ++u)
                        vreg[u] = __builtin_nontemporal_load((const uint4_t *)(vb + (min((uint32_t)(RPI * u + vrow0), lim) * rowb + vpc * 16u)));
                } else {
#pragma unroll
                    for (int u = 0; u < NV; ++u) {
                        const uint32_t s = (uint32_t)__shfl(slot_v, RPI * u + vrow0, ODSD_WAVE);
                        vreg[u] = __builtin_nontemporal_load((const uint4_t *)(vh + (uint64_t)s * rowb + vpc * 16));
                    }
                }
            };
            // one tile.  FETCH: there is a next one; it is requested into the registers this one has just left
            auto tile = [&](auto fetch_c, const int i) {
                const int k0 = key0 + STEP * i;
                float4_t st[RB][2];
#pragma unroll
                for (int t = 0; t < 2; ++t)
#pragma unroll
                    for (int rb = 0; rb < RB; ++rb) {
                        st[rb][t] = float4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                        for (int j = 0; j < NJ; ++j)
                            st[rb][t] = AttnT<T>::mfma(__builtin_bit_cast(V8, kreg[t][j]), qf[rb][j], st[rb][t]);
                    }
                if constexpr (decltype(fetch_c)::value) fetch_k(i + 1);
#pragma unroll
                for (int u = 0; u < NV; ++u) *(uint4_t *)(vt + vw_at[u & 1] + RPI * u * HD * 2) = vreg[u];
                if constexpr (decltype(fetch_c)::value) fetch_v(i + 1);
                V8 pf[RB];
#pragma unroll
                for (int rb = 0; rb < RB; ++rb) {
                    // lane (c, kq) holds keys k0 + 16 t + 4 kq + i of query row c (raw scores)
                    float a[8] = {st[rb][0].x, st[rb][0].y, st[rb][0].z, st[rb][0].w, st[rb][1].x, st[rb][1].y, st[rb][1].z, st[rb][1].w};
                    if (k0 + 31 > kmin) {
#pragma unroll
                        for (int e = 0; e < 8; ++e)
                            a[e] = k0 + 16 * (e >> 2) + 4 * kq + (e & 3) <= kmax[rb] ? a[e] : -INFINITY;
                    }
                    pf[rb] = softmax_tile<T, NDB>(a, sc, m_run[rb], l_run[rb], o[rb]);
                }
#pragma unroll
                for (int db = 0; db < NDB; ++db) {
                    const V8 vf = read_vt<V8>(vt + vr_at[db], 16 * HD * 2);
#pragma unroll
                    for (int rb = 0; rb < RB; ++rb) o[rb][db] = AttnT<T>::mfma(vf, pf[rb], o[rb][db]);
                }
            };
            if constexpr (!ALIGNED) pend = entry(0);
            fetch_k(0);
            fetch_v(0);
            int i = 0;
            for (; i + 1 < nt; ++i) tile(std::true_type{}, i);
            tile(std::false_type{}, i);
        }

        // ---- the four wavefronts' sums, through LDS -----------------------------------------------------
        const bool whole = n == sq.steps;
        __syncthreads();                                   // every wavefront is done with its V tile
#pragma unroll
        for (int rb = 0; rb < RB; ++rb) {
            float *xr = xch + (wave * ROWS + 16 * rb + c) * XROW;
            float l = l_run[rb];
            l += __shfl_xor(l, 16, ODSD_WAVE);
            l += __shfl_xor(l, 32, ODSD_WAVE);
#pragma unroll
            for (int db = 0; db < NDB; ++db) *(float4_t *)(xr + 16 * db + 4 * kq) = o[rb][db];
            if (kq == 0) {
                xr[HD] = m_run[rb];
                xr[HD + 1] = l;
            }
        }
        __syncthreads();
        // (a piece that begins where its workgroup's share begins goes to the workgroup's first slot)
        float *part = p.part + (size_t)(2 * blockIdx.x + (pos > (int)blockIdx.x * pl.share ? 1 : 0)) * (ROWS * XROW);
        for (int it = tid; it < rows_here * (HD / 4); it += 256) {
            const int row = it / (HD / 4), d = 4 * (it % (HD / 4));
            const float *xr = xch + row * XROW;
            float m = -INFINITY;
#pragma unroll
            for (int w = 0; w < 4; ++w) m = fmaxf(m, xr[w * ROWS * XROW + HD]);
            const float ref = m == -INFINITY ? 0.0f : m;
            float l = 0.0f;
            float4_t acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int w = 0; w < 4; ++w) {
                const float f = __builtin_amdgcn_exp2f(xr[w * ROWS * XROW + HD] - ref);      // -inf -> 0
                const float4_t v = *(const float4_t *)(xr + w * ROWS * XROW + d);
                l += f * xr[w * ROWS * XROW + HD + 1];
                acc.x += f * v.x; acc.y += f * v.y; acc.z += f * v.z; acc.w += f * v.w;
            }
            if (whole) {
                const float inv = l > 0.0f ? 1.0f / l : 0.0f;
                const int r = row0 + row, tok = r / p.Gq, hq = r - tok * p.Gq;
                typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
                *(u32x2 *)((uint16_t *)p.out + ((size_t)(sq.q0 + tok) * p.H + kvh * p.Gq + hq) * HD + d) =
                    u32x2{AttnT<T>::pack2(acc.x * inv, acc.y * inv), AttnT<T>::pack2(acc.z * inv, acc.w * inv)};
            } else {
                *(float4_t *)(part + row * XROW + d) = acc;
                if (d == 0) {
                    part[row * XROW + HD] = m;
                    part[row * XROW + HD + 1] = l;
                }
            }
        }
        pos += n;
        if (pos < end) {
            __syncthreads();                               // the exchange area becomes V tiles again
            next_unit(p, sq, unit, step, ROWS, pl.g);
        }
    }
}

// The form for more rows per sequence than the stream form takes (a verify step of a model with many query heads per
// KV head, a prompt chunk over the cache): a wavefront cannot hold 64 rows next to its keys, so here the four
// wavefronts own 16 rows each and share the keys through LDS, 32 at a time.  K and V rows are copied there
// asynchronously (a ring of tiles, one barrier per tile, waits that leave the younger copies in flight) and on across
// the end of a piece; the rows of the keys are looked up for many tiles at a time and kept in LDS.
// SPLIT: two workgroups per CU share all keys, with a ring of four.  Unsplit launches have workgroups to
// spare: a ring of two, 36 KB, lets a CU hold four of them, whose copies overlap (ring of four / three / two, us, 32
// / 4 heads: 256 sequences of 1500 keys x 8 144 / 138 / 121, 64 of 700 x 12, 32 / 8 heads, 33.4 / 32.6 / 27.0).
template <typename T, int HD, bool SPLIT>
__global__ __launch_bounds__(256, 2) void attn_tile_kernel(const AttnParams p) {
    typedef typename AttnT<T>::V8 V8;
    constexpr int NJ = HD / 32, NDB = HD / 16;
    constexpr int NP = HD / 8;           // 16-byte pieces of a row
    constexpr int RPC = 64 / NP;         // rows of one copy
    constexpr int COPIES = 32 / RPC / 4; // copies per wavefront, tile and matrix
    constexpr int ROWS = 64, XROW = HD + 4;
    constexpr int TILEB = 32 * HD * 2;
    constexpr int NBUF = SPLIT ? 4 : 2;
    constexpr int MOST = SPLIT ? 64 : 32;   // tiles whose rows are looked up at a time
    __shared__ __attribute__((aligned(16))) char lds[NBUF * 2 * TILEB];
    __shared__ uint32_t slots[MOST * 32];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int c = lane & 15, kq = lane >> 4;
    auto vswz = [](int key) { return HD == 128 ? (key & 7) : ((key >> 1) & 3); };

    const ListPlan pl = list_plan<false, SPLIT, !SPLIT, true>(p, ROWS, ATTN_TILE_FINE, ATTN_TILE_COARSE, blockIdx.x);
    if (!pl.found) return;
    const int first_pos = pl.me * pl.share, end = min(pl.total, first_pos + pl.share);
    const float sc = p.scale_log2e;

    // copies: row RPC * (wave + 4 i) + lane / NP of a tile, stored piece lane % NP (16-byte pieces of a K row and
    // 32-byte segments of a V row XORed with the key against bank conflicts)
    const int crow = lane / NP, cslot = lane % NP;
    uint32_t kp_at[COPIES], vp_at[COPIES];
#pragma unroll
    for (int i = 0; i < COPIES; ++i) {
        const int key = RPC * (wave + 4 * i) + crow;
        kp_at[i] = (uint32_t)(cslot ^ (key & (NP - 1))) * 16u;
        vp_at[i] = (uint32_t)(2 * ((cslot >> 1) ^ vswz(key)) + (cslot & 1)) * 16u;
    }
    // fragments: K (A operand: key 16 t + c, dims 32 j + 8 kq ..), V^T (dims 16 db + c of keys 4 kq .. and 16 + 4 kq ..)
    uint32_t k_at[NJ], v_at[NDB];
#pragma unroll
    for (int j = 0; j < NJ; ++j) k_at[j] = (uint32_t)(c * HD * 2 + ((4 * j + kq) ^ (c & (NP - 1))) * 16);
    const int rkey = 4 * kq + (c >> 2);
#pragma unroll
    for (int db = 0; db < NDB; ++db) v_at[db] = (uint32_t)(rkey * HD * 2 + (db ^ vswz(rkey)) * 32 + (c & 3) * 8);

    // The workgroup's share as pieces (consecutive steps of one unit).  Two cursors walk them: `ahead` looks up
    // the rows of the next tiles' keys, `now` is what is being computed.
    struct Cursor {
        SeqAt sq;
        int pos, unit, step, n;      // list position, unit, first step and steps of the piece
        int key, key_end;            // next key and end of the piece's keys
    };
    auto set_piece = [&](Cursor &q) {
        q.n = min(end - q.pos, q.sq.steps - q.step);
        q.key = pl.g * q.step;
        q.key_end = q.step + q.n == q.sq.steps ? q.sq.L : pl.g * (q.step + q.n);
        // (no further than the unit's last row sees: the row groups of a long query stop one after the other)
        if (q.sq.rg > 1) {
            const int r = q.sq.rg - 1 - q.unit % q.sq.rg, last = min(q.sq.ql, (ROWS * (r + 1) - 1) / p.Gq + 1);
            q.key_end = min(q.key_end, q.sq.L - q.sq.ql + last);
        }
    };
    auto next_piece = [&](Cursor &q) {
        q.pos += q.n;
        if (q.pos < end) {
            next_unit(p, q.sq, q.unit, q.step, ROWS, pl.g);
            set_piece(q);
        }
    };
    Cursor now;
    now.sq = pl.at;
    now.pos = first_pos;
    now.unit = (first_pos - pl.at.first) / pl.at.steps;
    now.step = (first_pos - pl.at.first) - now.unit * pl.at.steps;
    set_piece(now);
    Cursor ahead = now;

    // of the piece being computed
    bool fresh = true;                                     // its rows have not been set up yet
    bool active = false, ok = false;
    int tok = 0, hq = 0, kmax = -1, kmin = 0, kvh = 0;
    V8 qf[NJ];
    float m_run = 0.0f, l_run = 0.0f;
    float4_t o[NDB];
    auto begin_piece = [&]() {
        kvh = now.unit / now.sq.rg;
        const int rg = now.sq.rg - 1 - (now.unit - kvh * now.sq.rg);     // those with the most keys first
        const int rows_total = now.sq.ql * p.Gq, row0 = rg * ROWS + 16 * wave;
        const int row = row0 + c;
        active = row0 < rows_total;
        ok = row < rows_total;
        tok = ok ? row / p.Gq : 0;
        hq = ok ? row - tok * p.Gq : 0;
        kmax = ok ? now.sq.L - now.sq.ql + tok : -1;       // last position this row attends
        kmin = now.sq.L - now.sq.ql + row0 / p.Gq;
        const uint16_t *qp = (const uint16_t *)p.q + ((size_t)(now.sq.q0 + tok) * p.H + kvh * p.Gq + hq) * HD + 8 * kq;
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            uint4_t raw = {0u, 0u, 0u, 0u};
            if (ok) raw = *(const uint4_t *)(qp + 32 * j);
            qf[j] = __builtin_bit_cast(V8, raw);
        }
        m_run = -INFINITY;
        l_run = 0.0f;
#pragma unroll
        for (int db = 0; db < NDB; ++db) o[db] = float4_t{0.f, 0.f, 0.f, 0.f};
        fresh = false;
    };
    auto end_piece = [&]() {
        float l = l_run;
        l += __shfl_xor(l, 16, ODSD_WAVE);
        l += __shfl_xor(l, 32, ODSD_WAVE);
        if (ok) {
            if (now.n == now.sq.steps) {
                const float inv = l > 0.0f ? 1.0f / l : 0.0f;
                typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
                uint16_t *op = (uint16_t *)p.out + ((size_t)(now.sq.q0 + tok) * p.H + kvh * p.Gq + hq) * HD + 4 * kq;
#pragma unroll
                for (int db = 0; db < NDB; ++db)
                    *(u32x2 *)(op + 16 * db) = u32x2{AttnT<T>::pack2(o[db].x * inv, o[db].y * inv),
                                                     AttnT<T>::pack2(o[db].z * inv, o[db].w * inv)};
            } else {
                // (a piece that begins where its workgroup's share begins goes to the workgroup's first slot)
                float *part = p.part + (size_t)(2 * pl.me + (now.pos > first_pos ? 1 : 0)) * (ROWS * XROW) + (16 * wave + c) * XROW;
#pragma unroll
                for (int db = 0; db < NDB; ++db) *(float4_t *)(part + 16 * db + 4 * kq) = o[db];
                if (kq == 0) {
                    part[HD] = m_run;
                    part[HD + 1] = l;
                }
            }
        }
        next_piece(now);
        fresh = true;
    };

    while (now.pos < end) {
        if (fresh) begin_piece();
        // rows of K / V (slot * KVH + kvh) of the next tiles' keys, at most MOST tiles: positions past a
        // piece's last key repeat that key's row; an entry that is negative or beyond the cache reads slot 0
        int nt = 0;
        while (nt < MOST && ahead.pos < end) {
            const int L = ahead.sq.L, here = min(MOST - nt, max(0, (ahead.key_end - ahead.key + 31) / 32));
            const int ks = p.cu_k ? p.cu_k[ahead.sq.seq] : 0;
            const int h = ahead.unit / ahead.sq.rg;
            const int32_t *bt = p.block_tables + (size_t)ahead.sq.seq * p.max_blocks;
            for (int i = tid; i < 32 * here; i += 256) {
                const int pc = min(ahead.key + i, L - 1);
                uint32_t sl;
                if (p.cu_k) {
                    sl = (uint32_t)(ks + pc);
                } else {
                    const int blk = pc / p.block_size;
                    const int32_t b = bt[min(blk, p.max_blocks - 1)];
                    const int64_t s = (int64_t)b * p.block_size + (pc - blk * p.block_size);
                    sl = (b >= 0 && blk < p.max_blocks && s < p.num_slots) ? (uint32_t)s : 0u;
                }
                slots[32 * nt + i] = sl * (uint32_t)p.KVH + (uint32_t)h;
            }
            nt += here;
            ahead.key += 32 * here;
            if (ahead.key >= ahead.key_end) next_piece(ahead);
        }
        nt = __builtin_amdgcn_readfirstlane(nt);
        __syncthreads();
        // (Q has come in before the table entries; without this the compiler would wait for it, and with it for
        // every copy, at its first use)
#pragma unroll
        for (int j = 0; j < NJ; ++j) asm volatile("" : "+v"(qf[j]));
        auto copy_tile = [&](const int i) {
            char *dst = lds + i % NBUF * (2 * TILEB);
            uint32_t sl[COPIES];
#pragma unroll
            for (int u = 0; u < COPIES; ++u) sl[u] = slots[32 * i + RPC * (wave + 4 * u) + crow];
#pragma unroll
            for (int u = 0; u < COPIES; ++u) {
                const uint64_t off = (uint64_t)sl[u] * (HD * 2);
                dma16_from_to_lds((const char *)p.k_cache + off + kp_at[u], (lds_void *)(dst + RPC * (wave + 4 * u) * HD * 2));
                const char *vfrom = (const char *)p.v_cache + off + vp_at[u];
                lds_void *vto = (lds_void *)(dst + TILEB + RPC * (wave + 4 * u) * HD * 2);
                if (p.v_once) dma16_from_to_lds_nt(vfrom, vto);
                else dma16_from_to_lds(vfrom, vto);
            }
        };
#pragma unroll
        for (int i = 0; i < NBUF - 1; ++i)
            if (i < nt) copy_tile(i);
        for (int i = 0; i < nt; ++i) {
            while (now.key >= now.key_end) {               // (a piece without keys ends as it begins)
                if (fresh) begin_piece();
                end_piece();
            }
            if (fresh) begin_piece();
            // tile i has landed once only the copies of the younger tiles are outstanding
            if (NBUF > 3 && i + 2 < nt) ODSD_WAIT_VMCNT_LGKM0(2 * 2 * COPIES);
            else if (NBUF > 2 && i + 1 < nt) ODSD_WAIT_VMCNT_LGKM0(2 * COPIES);
            else ODSD_WAIT_VMCNT_LGKM0(0);
            __builtin_amdgcn_s_barrier();                  // ... for every wavefront, and all are done with tile i - 1
            if (i + NBUF - 1 < nt) copy_tile(i + NBUF - 1);
            if (active) {
                const char *kt = lds + i % NBUF * (2 * TILEB), *vt = kt + TILEB;
                const int k0 = now.key;
                float4_t st[2];
#pragma unroll
                for (int t = 0; t < 2; ++t) {
                    st[t] = float4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                    for (int j = 0; j < NJ; ++j)
                        st[t] = AttnT<T>::mfma(*(const V8 *)(kt + k_at[j] + t * 16 * HD * 2), qf[j], st[t]);
                }
                float a[8] = {st[0].x, st[0].y, st[0].z, st[0].w, st[1].x, st[1].y, st[1].z, st[1].w};
                if (k0 + 31 > kmin) {
#pragma unroll
                    for (int e = 0; e < 8; ++e)
                        a[e] = k0 + 16 * (e >> 2) + 4 * kq + (e & 3) <= kmax ? a[e] : -INFINITY;
                }
                const V8 pf = softmax_tile<T, NDB>(a, sc, m_run, l_run, o);
#pragma unroll
                for (int db = 0; db < NDB; ++db) {
                    const V8 vf = read_vt<V8>(vt + v_at[db], 16 * HD * 2);
                    o[db] = AttnT<T>::mfma(vf, pf, o[db]);
                }
            }
            now.key += 32;
        }
        // (pieces that end with the list, or had no keys at all)
        while (now.pos < end && now.key >= now.key_end) {
            if (fresh) begin_piece();
            end_piece();
        }
        ODSD_WAIT_VMCNT_LGKM0(0);
        __builtin_amdgcn_s_barrier();                      // buffers and slots are free again
    }
}

// Merge of the pieces of a unit: out[row] = sum_s exp2(m_s - m) O_s / sum_s exp2(m_s - m) l_s, pieces in
// order.  One workgroup per (sequence, KV head, unit, 1024 / HD rows): a thread owns 4 neighbouring output
// elements of a row and walks the pieces, 4 at a time.  Units that were finished in place are left alone.
// BY_SHARE: one workgroup per bound between two shares instead, and 1024 / HD rows; the first bound inside a unit
// does the work.  (For launches that allow for many row groups, which need not be there: 64 sequences of 8
// queries with the query lengths bounded by the 512 tokens of the call only, 900 keys: 131072 workgroups
// otherwise, 96 us the call.)
template <typename T, int HD, int ROWS, int FINE, int COARSE, bool BY_SHARE = false>
__global__ __launch_bounds__(256) void attn_merge_kernel(const AttnParams p) {
    constexpr int XROW = HD + 4;
    constexpr int TPR = HD / 4, RPW = 256 / TPR;
    int kvh, rg, a;                                                // a: list position of the unit's first step
    const ListPlan pl = list_plan<!BY_SHARE, true, false>(p, ROWS, FINE, COARSE, BY_SHARE ? blockIdx.x + 1 : blockIdx.x / p.KVH);
    const SeqAt &sq = pl.at;
    if (BY_SHARE) {
        if (!pl.found) return;
        const int at = ((int)blockIdx.x + 1) * pl.share - sq.first, unit = at / sq.steps;
        kvh = unit / sq.rg;
        rg = sq.rg - 1 - (unit - kvh * sq.rg);
        a = sq.first + unit * sq.steps;
    } else {
        kvh = blockIdx.x % p.KVH;
        rg = blockIdx.y;
        if (rg >= sq.rg) return;
        a = sq.first + (kvh * sq.rg + sq.rg - 1 - rg) * sq.steps;
    }
    const int wa = a / pl.share, wb = (a + sq.steps - 1) / pl.share;
    if (wa == wb || (BY_SHARE && wa != (int)blockIdx.x)) return;
    const int row = (int)blockIdx.z * RPW + (int)threadIdx.x / TPR, d = 4 * ((int)threadIdx.x % TPR);
    const int r = rg * ROWS + row;
    if (row >= ROWS || r >= sq.ql * p.Gq) return;
    const float *base = p.part + row * XROW;
    const size_t slot = (size_t)ROWS * XROW;
    auto piece = [&](const int w) { return base + (size_t)(2 * w + (w == wa && a > wa * pl.share ? 1 : 0)) * slot; };
    float m = -INFINITY, l = 0.0f;
    float4_t acc = {0.f, 0.f, 0.f, 0.f};
    constexpr int SB = 4;
    for (int w0 = wa; w0 <= wb; w0 += SB) {
        float ms[SB], ls[SB];
        float4_t os[SB];
#pragma unroll
        for (int u = 0; u < SB; ++u) {
            // (every load unconditional, on a clamped piece: loads under a branch serialise)
            const float *rp = piece(min(w0 + u, wb));
            const float2_t ml = *(const float2_t *)(rp + HD);
            ms[u] = ml.x;
            ls[u] = ml.y;
            os[u] = *(const float4_t *)(rp + d);
        }
#pragma unroll
        for (int u = 0; u < SB; ++u) {
            if (w0 + u > wb) {
                ms[u] = -INFINITY;
                ls[u] = 0.0f;
                os[u] = float4_t{0.f, 0.f, 0.f, 0.f};
            }
        }
        float mb = m;
#pragma unroll
        for (int u = 0; u < SB; ++u) mb = fmaxf(mb, ms[u]);
        const float ref = mb == -INFINITY ? 0.0f : mb;
        const float keep = __builtin_amdgcn_exp2f(m - ref);            // m = -inf -> 0
        l *= keep;
        acc.x *= keep; acc.y *= keep; acc.z *= keep; acc.w *= keep;
#pragma unroll
        for (int u = 0; u < SB; ++u) {
            const float f = __builtin_amdgcn_exp2f(ms[u] - ref);
            l += f * ls[u];
            acc.x += f * os[u].x; acc.y += f * os[u].y; acc.z += f * os[u].z; acc.w += f * os[u].w;
        }
        m = mb;
    }
    const float inv = l > 0.0f ? 1.0f / l : 0.0f;
    const int tok = r / p.Gq, hq = r - tok * p.Gq;
    typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
    *(u32x2 *)((uint16_t *)p.out + ((size_t)(sq.q0 + tok) * p.H + kvh * p.Gq + hq) * HD + d) =
        u32x2{AttnT<T>::pack2(acc.x * inv, acc.y * inv), AttnT<T>::pack2(acc.z * inv, acc.w * inv)};
}

// ---- host side -----------------------------------------------------------------------------------------
// Form of the kernel by the query rows of a sequence and the bytes that the keys can have
struct AttnForm {
    int rows;            // per unit
    int fine, coarse, whole;
    bool tile;
};
static int64_t attn_kv_bytes(int64_t n_seqs, int64_t max_keys, int kvh, int head_dim) {
    return n_seqs * max_keys * kvh * head_dim * 4;
}
static AttnForm attn_form(int64_t rows, int64_t kv_bytes) {
    // 17 to 32 rows: two row blocks per wavefront pay with many keys, the shared tiles with fewer (us, shared / own:
    // 32 / 8 heads, 64 sequences of up to 400 keys, 105 MB, 22.5 / 18.5, 700 31.5 / 25.9, 1000 41.4 / 34.0, 40 of
    // 1500 40.9 / 42.5; 16 / 8 heads of 64, 64 of 1000 33.3 / 21.4; 32 / 4 heads, 64 of 2000 68.3 / 62.6, but 16 of
    // 1000, 33 MB, 17.3 / 19.9)
    const bool wide = rows > 16 && rows <= 32 && kv_bytes > (96LL << 20);
    if (rows <= 16 || wide) return AttnForm{wide ? 32 : 16, ATTN_STREAM_FINE, ATTN_STREAM_COARSE, ATTN_STREAM_WHOLE, false};
    return AttnForm{64, ATTN_TILE_FINE, ATTN_TILE_COARSE, ATTN_TILE_WHOLE, true};
}

// Long queries (row groups at sight of more and more keys): nothing is split once the units fill the chip, from
// (keys - 320) / 4 units on, 300 at most (unsplit / split, us; 32 / 4 heads: 400 keys 50 units 13.2 / 13.9, 800 keys 68
// 21.0 / 18.2, 128 21.3 / 23.1, 1600 keys 200 36.9 / 33.7, 400 43.9 / 53.2, 3200 keys 200 70 / 52, 400 81 / 92, 3200
// 220 / 648).  But max_q_len may be far above what the sequences have, all tokens of the call by default; so only
// where the query can be more than 1 / LONG of the keys (16 sequences of 4000 keys, 8 queries, bounded by 128: 34
// split, 110 as one workgroup per unit before; the other way round 16 of 2000 keys with 100 queries of 4 heads take
// 105 split and would take 87 unsplit).  With LONG_RG row groups and more the units are found in the list, at
// most LISTED shares of them: workgroups without one end after its scan.
// In the other rules row groups are not counted.  List positions are 32 bits wide: a list that could grow past 2^30
// steps stays whole, with 2^18 units and more even on 131072 keys.
#define ATTN_LONG 16
#define ATTN_LONG_RG 4
#define ATTN_LISTED 16384
static bool attn_keep_whole(const AttnForm &f, int64_t n_seqs, int kvh, int64_t rg, int64_t max_q, int64_t max_keys) {
    const int64_t units = n_seqs * kvh, steps = (max_keys + f.fine - 1) / f.fine;
    if (max_keys <= f.whole || units >= ATTN_MANY || units * rg * steps > (1LL << 30)) return true;
    if (f.tile && ATTN_LONG * max_q > max_keys && 4 * units * rg >= min(max_keys - 320, (int64_t)1200)) return true;
    return f.tile ? max_keys <= min(192 + 5 * units, (int64_t)2048) : units >= 128 && max_keys <= 1024;
}

// What a call does, from its shape alone.  The size functions and the launch both ask here, with the same
// number of keys: the form, whether units are split and the workspace belong together.
struct AttnPlan {
    AttnForm f;
    int64_t rg, units;            // row groups per (sequence, KV head), units
    int shares;                   // workgroups that can get a share of the list
    int64_t kv_bytes;
    bool split;                   // units may be split: partial results and a merge
    size_t bytes;                 // workspace that splitting takes
};
// max_q, max_keys: query tokens and keys of a sequence at most; Gq: query heads per KV head
static AttnPlan attn_plan(int64_t n_seqs, int64_t max_q, int Gq, int64_t max_keys, int kvh, int head_dim) {
    AttnPlan pl;
    const int64_t rows = max_q * Gq;
    pl.kv_bytes = attn_kv_bytes(n_seqs, max_keys, kvh, head_dim);
    pl.f = attn_form(rows, pl.kv_bytes);
    pl.rg = (rows + pl.f.rows - 1) / pl.f.rows;
    pl.units = n_seqs * kvh * pl.rg;
    pl.split = !attn_keep_whole(pl.f, n_seqs, kvh, pl.rg, max_q, max_keys);
    // a list too short for the fine granularity is cut at the coarse one, and no workgroup has less than one step
    int64_t total = pl.units * ((max_keys + pl.f.fine - 1) / pl.f.fine);
    if (total < (int64_t)(pl.f.coarse / pl.f.fine) * ATTN_WG) total = pl.units * ((max_keys + pl.f.coarse - 1) / pl.f.coarse);
    pl.shares = (int)min(total, (int64_t)ATTN_WG);
    pl.bytes = pl.split ? odsd_round_up((size_t)2 * pl.shares * pl.f.rows * (head_dim + 4) * sizeof(float), 256) : 0;
    return pl;
}
static bool attn_plan_shape_ok(int32_t n_seqs, int32_t max_q_len, int64_t max_keys, int32_t num_heads,
                               int32_t num_kv_heads, int32_t head_dim) {
    if (n_seqs <= 0 || max_q_len <= 0 || max_keys <= 0 || num_heads <= 0 || num_kv_heads <= 0 ||
        num_heads % num_kv_heads || (head_dim != 64 && head_dim != 128))
        return false;
    return ((int64_t)max_q_len * (num_heads / num_kv_heads) + 63) / 64 <= 65535;
}
static size_t attn_workspace_bytes(int32_t n_seqs, int32_t max_q_len, int64_t max_keys, int32_t num_heads,
                                   int32_t num_kv_heads, int32_t head_dim) {
    if (!attn_plan_shape_ok(n_seqs, max_q_len, max_keys, num_heads, num_kv_heads, head_dim)) return 0;
    const AttnPlan pl = attn_plan(n_seqs, max_q_len, num_heads / num_kv_heads, max_keys, num_kv_heads, head_dim);
    return pl.split ? pl.bytes : 256;
}

extern "C" size_t odsd_paged_attention_workspace_bytes(int32_t n_seqs, int32_t max_q_len, int32_t num_heads,
                                                       int32_t num_kv_heads, int32_t head_dim,
                                                       int32_t block_size, int32_t max_blocks) {
    if (block_size <= 0 || max_blocks <= 0) return 0;
    return attn_workspace_bytes(n_seqs, max_q_len, (int64_t)max_blocks * block_size, num_heads, num_kv_heads, head_dim);
}

// p: everything but Gq, n_wg, part; max_keys: no sequence has more
static int attn_stream_launch(AttnParams &p, int32_t dtype, int head_dim, int64_t max_q, int64_t max_keys, bool aligned,
                              void *workspace, size_t workspace_bytes, hipStream_t st) {
    const AttnPlan pl = attn_plan(p.n_seqs, max_q, p.H / p.KVH, max_keys, p.KVH, head_dim);
    const AttnForm &f = pl.f;
    const int64_t rg = pl.rg, units = pl.units, kv_bytes = pl.kv_bytes;
    p.Gq = p.H / p.KVH;
    p.max_keys = (int)min(max_keys, (int64_t)1 << 30);               // (rounding up to a step stays within 32 bits)
    p.max_rg = (int)rg;
    if (rg > 65535) return ODSD_ERR_UNSUPPORTED;                      // grid.y of the merge
    // a unit per workgroup slot, or at most 480 keys: splitting levels the lengths out, but these calls can do
    // without it, and do when they bring no workspace for it
    const bool can_do_without = units >= ATTN_WG || max_keys <= 480;
    const bool no_workspace = !workspace || !odsd_aligned16(workspace) || workspace_bytes < pl.bytes;
    const bool merge = pl.split && !(can_do_without && no_workspace);
    if (merge) {
        if (!workspace) return ODSD_ERR_NULL;
        if (!odsd_aligned16(workspace)) return ODSD_ERR_ALIGN;
        if (workspace_bytes < pl.bytes) return ODSD_ERR_WORKSPACE;
        p.part = (float *)workspace;
        p.n_wg = ATTN_WG;
        p.whole = 0;
    } else {
        if (units > 0x7fffffff) return ODSD_ERR_UNSUPPORTED;
        // each a workgroup of its own, finished in place; the bound on the row groups may be far above what there
        // is, so with many of them the units are found in the list
        const bool list = rg >= ATTN_LONG_RG;
        p.n_wg = (int)(list ? min(units, (int64_t)ATTN_LISTED) : units);
        p.whole = list ? 0 : (int)rg;
    }
    const unsigned grid = (unsigned)(merge ? pl.shares : p.n_wg);
    // Up to 100 MB of keys may still be in the 256 MB memory-side cache from the call before; more are read past it:
    // 32 sequences of 2048 keys, 134 MB, 37.3 us where other keys came before (41.6 without the hint), 36.8 where the
    // same call did (34.2).  A model has other layers' keys in between.
    p.v_once = kv_bytes > (100 << 20);
    const dim3 mgrid((unsigned)(p.n_seqs * p.KVH), (unsigned)rg, (unsigned)((f.rows * head_dim + 1023) / 1024));
#define ATTN_GO(T, HDV, RBV)                                                                     \
    do {                                                                                         \
        if (aligned) attn_stream_kernel<T, HDV, RBV, true><<<grid, 256, 0, st>>>(p);             \
        else attn_stream_kernel<T, HDV, RBV, false><<<grid, 256, 0, st>>>(p);                    \
        if (merge) attn_merge_kernel<T, HDV, 16 * RBV, ATTN_STREAM_FINE, ATTN_STREAM_COARSE><<<mgrid, 256, 0, st>>>(p);           \
    } while (0)
#define ATTN_GO_RB(T, HDV)                                                                       \
    do {                                                                                         \
        if (f.rows == 16) ATTN_GO(T, HDV, 1);                                                    \
        else if (f.rows == 32) ATTN_GO(T, HDV, 2);                                               \
        else {                                                                                   \
            if (merge) attn_tile_kernel<T, HDV, true><<<grid, 256, 0, st>>>(p);                  \
            else attn_tile_kernel<T, HDV, false><<<grid, 256, 0, st>>>(p);                       \
            if (merge && units > 2 * ATTN_WG)                                                    \
                attn_merge_kernel<T, HDV, 64, ATTN_TILE_FINE, ATTN_TILE_COARSE, true><<<dim3(ATTN_WG - 1, 1, mgrid.z), 256, 0, st>>>(p); \
            else if (merge) attn_merge_kernel<T, HDV, 64, ATTN_TILE_FINE, ATTN_TILE_COARSE><<<mgrid, 256, 0, st>>>(p); \
        }                                                                                        \
    } while (0)
    if (dtype == ODSD_DT_F16) {
        if (head_dim == 128) ATTN_GO_RB(half_t, 128);
        else ATTN_GO_RB(half_t, 64);
    } else {
        if (head_dim == 128) ATTN_GO_RB(__bf16, 128);
        else ATTN_GO_RB(__bf16, 64);
    }
#undef ATTN_GO_RB
#undef ATTN_GO
    ODSD_CHECK_LAUNCH();
    return ODSD_OK;
}

extern "C" int odsd_paged_attention(const void *q, const void *k_cache, const void *v_cache,
                                    const int32_t *block_tables, const int32_t *context_lens,
                                    const int32_t *q_lens, int32_t n_seqs, int32_t max_q_len,
                                    int32_t num_heads, int32_t num_kv_heads, int32_t head_dim,
                                    int32_t block_size, int32_t max_blocks, int64_t num_slots,
                                    float softmax_scale, int32_t dtype, void *out, void *workspace,
                                    size_t workspace_bytes, void *stream) {
    if (n_seqs < 0 || max_q_len <= 0 || num_heads <= 0 || num_kv_heads <= 0 || num_heads % num_kv_heads ||
        block_size <= 0 || max_blocks <= 0 || num_slots <= 0 || !(softmax_scale > 0.0f))
        return ODSD_ERR_SHAPE;
    if (head_dim != 64 && head_dim != 128) return ODSD_ERR_UNSUPPORTED;
    if (dtype != ODSD_DT_BF16 && dtype != ODSD_DT_F16) return ODSD_ERR_DTYPE;
    if (n_seqs == 0) return ODSD_OK;
    if (!q || !k_cache || !v_cache || !block_tables || !context_lens || !out) return ODSD_ERR_NULL;
    if (!odsd_aligned16(q) || !odsd_aligned16(k_cache) || !odsd_aligned16(v_cache)) return ODSD_ERR_ALIGN;
    if ((int64_t)n_seqs * num_kv_heads > 0x7fffffffLL) return ODSD_ERR_SHAPE;
    AttnParams p{};
    p.q = q; p.k_cache = k_cache; p.v_cache = v_cache; p.out = out;
    p.q_lens = q_lens; p.context_lens = context_lens; p.block_tables = block_tables;
    p.n_seqs = n_seqs; p.H = num_heads; p.KVH = num_kv_heads; p.max_blocks = max_blocks;
    p.block_size = block_size; p.num_slots = num_slots;
    p.scale_log2e = softmax_scale * 1.4426950408889634f;
    return attn_stream_launch(p, dtype, head_dim, max_q_len, (int64_t)max_blocks * block_size, block_size % 32 == 0,
                              workspace, workspace_bytes, (hipStream_t)stream);
}

// ---- variable-length (prefill) form ----------------------------------------------------------------
extern "C" size_t odsd_varlen_attention_workspace_bytes(int32_t n_seqs, int32_t max_seqlen_q, int32_t max_seqlen_k,
                                                        int32_t num_heads, int32_t num_kv_heads, int32_t head_dim) {
    return attn_workspace_bytes(n_seqs, max_seqlen_q, max_seqlen_k, num_heads, num_kv_heads, head_dim);
}

extern "C" int odsd_varlen_attention(const void *q, const void *k, const void *v, const int32_t *cu_seqlens_q,
                                     const int32_t *cu_seqlens_k, int32_t n_seqs, int32_t max_seqlen_q,
                                     int32_t max_seqlen_k, int32_t num_heads, int32_t num_kv_heads,
                                     int32_t head_dim, float softmax_scale, int32_t dtype, void *out,
                                     void *workspace, size_t workspace_bytes, void *stream) {
    if (n_seqs < 0 || max_seqlen_q <= 0 || max_seqlen_k <= 0 || num_heads <= 0 || num_kv_heads <= 0 ||
        num_heads % num_kv_heads || !(softmax_scale > 0.0f))
        return ODSD_ERR_SHAPE;
    if (head_dim != 64 && head_dim != 128) return ODSD_ERR_UNSUPPORTED;
    if (dtype != ODSD_DT_BF16 && dtype != ODSD_DT_F16) return ODSD_ERR_DTYPE;
    if (n_seqs == 0) return ODSD_OK;
    if (!q || !k || !v || !cu_seqlens_q || !cu_seqlens_k || !out) return ODSD_ERR_NULL;
    if (!odsd_aligned16(q) || !odsd_aligned16(k) || !odsd_aligned16(v)) return ODSD_ERR_ALIGN;
    if ((int64_t)n_seqs * num_kv_heads > 0x7fffffffLL) return ODSD_ERR_SHAPE;
    AttnParams p{};
    p.q = q; p.k_cache = k; p.v_cache = v; p.out = out;
    p.cu_q = cu_seqlens_q; p.cu_k = cu_seqlens_k;
    p.n_seqs = n_seqs; p.H = num_heads; p.KVH = num_kv_heads;
    p.block_size = 32; p.max_blocks = (max_seqlen_k + 31) / 32; p.num_slots = 0;
    p.scale_log2e = softmax_scale * 1.4426950408889634f;
    const int64_t rows = (int64_t)max_seqlen_q * (num_heads / num_kv_heads);
    if ((rows + 63) / 64 > 65535) return ODSD_ERR_UNSUPPORTED;     // grid.y
    if (odsd_attn_prefill_supported(p, head_dim, max_seqlen_q, max_seqlen_k)) {
        odsd_launch_attn_prefill(p, dtype, head_dim, max_seqlen_q, (hipStream_t)stream);
        ODSD_CHECK_LAUNCH();
        return ODSD_OK;
    }
    return attn_stream_launch(p, dtype, head_dim, max_seqlen_q, max_seqlen_k, true, workspace, workspace_bytes, (hipStream_t)stream);
}
