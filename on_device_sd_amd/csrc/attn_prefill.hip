// Causal attention of a prefill step over packed sequences: many query rows per sequence.
//
// One workgroup of 4 wavefronts per (sequence, KV head, 128 query rows); a query row is one (token,
// query head) pair of the KV head's group.  A wavefront owns 32 rows and the workgroup walks the keys
// 64 at a time on v_mfma_f32_32x32x16:
//   * K and V tiles come by asynchronous global -> LDS copies (double buffered, one barrier per tile),
//     as stored, with 16-byte pieces (K) and 32-byte segments (V) of a row XORed with the key against
//     bank conflicts (measured: none; with the V swizzle of the decode kernel a third of the LDS cycles);
//   * S^T = K Q^T: a lane ends up with 32 of the 64 scores of ONE query row (lane % 32), its partner
//     lane ^ 32 with the others, in the order in which O^T = V^T P^T wants its B operand, so the
//     probabilities never leave the lane and the row's maximum, sum and rescaling factor are lane values;
//   * the scores of the next tile are computed in the step that exponentiates this one: one wavefront
//     then has matrix and vector work that do not wait for each other;
//   * V^T as the A operand through ds_read_b64_tr_b16 (no transposed copy).
// Against the decode / verify kernel, which ran these calls before: twice the rows per wavefront, so a
// fragment read from LDS feeds an MFMA of twice the flops, and a barrier covers four times the work.
// Bound by the two wavefronts a SIMD has room for: matrix unit busy 53 % and vector issue 41 % of the
// cycles with workgroups (46 % and 36 % of all), no bank conflict; two thirds of the vector instructions
// are the exponentials and their scaling.  (32-key tiles with three wavefronts per SIMD: + 3 % at 4096 tokens,
// - 10 % below 2000; raised wavefront priority round the MFMAs: - 1 to - 5 %.)
// Measured, causal flops, 32 query / 4 KV heads of 128, bf16, before -> now: 8192 tokens 812 -> 486 us
// (1130 TFLOP/s), 4096 tokens 236 -> 137, three sequences of 1200 to 3000 206 -> 120, 300 tokens
// 12.6 -> 9.0.
//
// Replaces the flash_attn_varlen_func call of the prefill branch (demo/src/layers/attention.py:229-240).
#include "attn.h"

#include "w4_gemm.h"
#include <type_traits>

// SPLIT == 2: 64 rows per workgroup; the four wavefronts are two row blocks x two halves of every tile's
// keys, and the halves are merged through LDS at the end.  For launches that do not fill the chip: twice
// the workgroups, and half the work between two barriers.
template <typename T, int HD, int SPLIT>
__global__ __launch_bounds__(256, 2) void attn_prefill_kernel(const AttnParams p) {
    typedef typename AttnT<T>::V8 V8;
    constexpr int KT = 64;                     // keys per tile
    constexpr int NJ = HD / 16;                // 16-dim steps of the score product
    constexpr int NDB = HD / 32;               // 32-dim blocks of the output
    constexpr int ROWB = HD * 2;               // bytes of a K or V row
    constexpr int TILEB = KT * ROWB;
    constexpr int NP = HD / 8;                 // 16-byte pieces of a row
    constexpr int RPC = 64 / NP;               // rows of one 1 KiB copy
    constexpr int NB = KT / 32 / SPLIT;        // 32-key blocks of a tile per wavefront
    constexpr int ROWS = 128 / SPLIT;          // query rows per workgroup
    constexpr int COPIES = KT / RPC / 4;       // copies per wavefront and matrix
    __shared__ __attribute__((aligned(16))) char lds[4 * TILEB];     // K tile 0, K tile 1, V tile 0, V tile 1

    const int seq = blockIdx.x / p.KVH, kvh = blockIdx.x % p.KVH;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int c = lane & 31, h = lane >> 5;
    const int Gq = p.H / p.KVH;
    const int k_start = p.cu_k[seq], L = p.cu_k[seq + 1] - k_start;
    const int q0 = p.cu_q[seq], ql = p.cu_q[seq + 1] - q0;
    const int rows_total = ql * Gq;
    // the row groups with the most keys first: the launch then ends with short ones
    const int rg = (int)(gridDim.y - 1 - blockIdx.y);
    if (ql <= 0 || rg * ROWS >= rows_total) return;
    const int rblk = SPLIT == 2 ? wave & 1 : wave, khalf = SPLIT == 2 ? wave >> 1 : 0;
    const int row = rg * ROWS + rblk * 32 + c;
    const bool row_ok = row < rows_total;
    const int tok = row_ok ? row / Gq : 0, hq = row_ok ? row % Gq : 0;
    const int D = p.KVH * HD;
    const float sc = p.scale_log2e;

    const int kmax = row_ok ? L - ql + tok : -1;       // last position this row attends
    int kmin_wave = row_ok ? kmax : 0x7fffffff;        // tiles that end at or before it need no mask
#pragma unroll
    for (int d = 16; d >= 1; d >>= 1) kmin_wave = min(kmin_wave, __shfl_xor(kmin_wave, d, ODSD_WAVE));
    kmin_wave = __builtin_amdgcn_readfirstlane(kmin_wave);
    const int last_tok = min(ql - 1, (rg * ROWS + ROWS - 1) / Gq);
    const int k_end = max(0, min(L, L - ql + last_tok + 1));
    const int n_tiles = (k_end + KT - 1) / KT;

    // copies of this wavefront: rows RPC * (wave + 4 i) + lane / NP of a tile, piece lane % NP
    const global_char *kb = (const global_char *)p.k_cache + ((size_t)k_start * D + (size_t)kvh * HD) * 2;
    const global_char *vb = (const global_char *)p.v_cache + ((size_t)k_start * D + (size_t)kvh * HD) * 2;
    const int crow = lane / NP, cslot = lane % NP;
    auto vswz = [](int key) { return (HD == 128 ? 2 * (key & 3) : 2 * ((key >> 1) & 1)) | ((key >> 2) & 1); };
    auto copy_k = [&](auto buf_c, const int k0) {
        constexpr int buf = decltype(buf_c)::value;
#pragma unroll
        for (int i = 0; i < COPIES; ++i) {
            const int key = RPC * (wave + 4 * i) + crow;
            const uint32_t base = (uint32_t)min(k0 + key, L - 1) * (uint32_t)(D * 2);
            const uint32_t kp = (uint32_t)(cslot ^ (key & (NP - 1)));
            dma16_to_lds(kb, base + kp * 16u, (lds_void *)(lds + buf * TILEB + RPC * (wave + 4 * i) * ROWB));
        }
    };
    auto copy_v = [&](auto buf_c, const int k0) {
        constexpr int buf = decltype(buf_c)::value;
#pragma unroll
        for (int i = 0; i < COPIES; ++i) {
            const int key = RPC * (wave + 4 * i) + crow;
            const uint32_t base = (uint32_t)min(k0 + key, L - 1) * (uint32_t)(D * 2);
            const uint32_t vp = (uint32_t)(2 * ((cslot >> 1) ^ vswz(key)) + (cslot & 1));
            dma16_to_lds(vb, base + vp * 16u, (lds_void *)(lds + (2 + buf) * TILEB + RPC * (wave + 4 * i) * ROWB));
        }
    };

    // LDS byte offsets of this lane's fragments: K (A operand: key c, dims 16 j + 8 h ..) and V^T
    // (dims 32 db + lane % 32 of 4 keys: lane c16 of a group of 16 addresses key c16 / 4, 4 dims)
    uint32_t k_at[NJ], v_at[NDB];
#pragma unroll
    for (int j = 0; j < NJ; ++j) k_at[j] = (uint32_t)(c * ROWB + ((2 * j + h) ^ (c & (NP - 1))) * 16);
    const int c16 = lane & 15, vkey = 4 * h + (c16 >> 2);
#pragma unroll
    for (int db = 0; db < NDB; ++db)
        v_at[db] = (uint32_t)(vkey * ROWB + ((2 * db + ((lane >> 4) & 1)) ^ vswz(vkey)) * 32 + (c16 & 3) * 8);

    float m_run = -INFINITY, l_run = 0.0f;
    float16_t o[NDB];
#pragma unroll
    for (int db = 0; db < NDB; ++db)
#pragma unroll
        for (int i = 0; i < 16; ++i) o[db][i] = 0.0f;

    V8 qf[NJ];
    auto load_q = [&]() {
        const uint16_t *qp = (const uint16_t *)p.q + ((size_t)(q0 + tok) * p.H + kvh * Gq + hq) * HD + 8 * h;
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            uint4_t raw = {0u, 0u, 0u, 0u};
            if (row_ok) raw = *(const uint4_t *)(qp + 16 * j);
            qf[j] = __builtin_bit_cast(V8, raw);
        }
    };

    // S^T of the tile in K buffer `buf`
    auto scores = [&](auto buf_c, float16_t (&st)[NB]) {
        constexpr int buf = decltype(buf_c)::value;
        const char *kt = lds + buf * TILEB + khalf * 32 * ROWB;
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
            for (int i = 0; i < 16; ++i) st[b][i] = 0.0f;
#pragma unroll
        for (int j = 0; j < NJ; ++j)
#pragma unroll
            for (int b = 0; b < NB; ++b) {
                const V8 kf = *(const V8 *)(kt + k_at[j] + b * 32 * ROWB);
                st[b] = AttnT<T>::mfma32(kf, qf[j], st[b]);
            }
    };
    // lane (c, h), register i of block b: key k0 + 32 b + 8 (i / 4) + 4 h + i % 4 of row c
    auto mask = [&](const int k0t, float16_t (&st)[NB]) {
        const int k0 = k0t + khalf * 32;
        if (k0 + 32 * NB - 1 > kmin_wave) {
#pragma unroll
            for (int b = 0; b < NB; ++b)
#pragma unroll
                for (int i = 0; i < 16; ++i)
                    st[b][i] = k0 + 32 * b + 8 * (i >> 2) + 4 * h + (i & 3) <= kmax ? st[b][i] : -INFINITY;
        }
    };
    // One step: softmax of tile `it` (scores in st), O += P V of it, and the scores of tile it + 1 into
    // sn, whose MFMAs run under the exponentials.
    auto step = [&](auto buf_c, auto more_c, const int it, float16_t (&st)[NB], float16_t (&sn)[NB]) {
        constexpr int buf = decltype(buf_c)::value;
        constexpr bool MORE = decltype(more_c)::value;
        const std::integral_constant<int, buf> cur;
        const std::integral_constant<int, buf ^ 1> oth;
        // K buffer `buf` was read for the last time in the step before, V buffer `oth` as well
        if constexpr (MORE) {
            copy_k(cur, (it + 2) * KT);
            copy_v(oth, (it + 1) * KT);
        }
        mask(it * KT, st);
        float mx = st[0][0];
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
            for (int i = 0; i < 16; ++i) mx = fmaxf(mx, st[b][i]);
        // The reference point of a row moves only when a score exceeds it by more than 2^8
        // (probabilities up to 256 are as exact in fp16 / bf16 as those below 1, the sums are fp32).
        if (__any(mx * sc > m_run + 8.0f)) {
            mx = fmaxf(mx, __shfl_xor(mx, 32, ODSD_WAVE));
            const float m_new = fmaxf(m_run, mx * sc);
            const float alpha = __builtin_amdgcn_exp2f(m_run - (m_new == -INFINITY ? 0.0f : m_new));
            l_run *= alpha;
            m_run = m_new;
#pragma unroll
            for (int db = 0; db < NDB; ++db)
#pragma unroll
                for (int i = 0; i < 16; ++i) o[db][i] *= alpha;
        }
        const float neg_ref = m_run == -INFINITY ? 0.0f : -m_run;
        if constexpr (MORE) scores(oth, sn);
        V8 pf[2 * NB];                                   // k-step s: keys 16 s + {4 h .. + 3, 8 + 4 h .. + 3}
        float ls = 0.0f;
#pragma unroll
        for (int s = 0; s < 2 * NB; ++s) {
            float pe[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) pe[i] = __builtin_amdgcn_exp2f(fmaf(st[s >> 1][8 * (s & 1) + i], sc, neg_ref));
            ls += ((pe[0] + pe[1]) + (pe[2] + pe[3])) + ((pe[4] + pe[5]) + (pe[6] + pe[7]));
            pf[s] = __builtin_bit_cast(V8, uint4_t{AttnT<T>::pack2(pe[0], pe[1]), AttnT<T>::pack2(pe[2], pe[3]),
                                                   AttnT<T>::pack2(pe[4], pe[5]), AttnT<T>::pack2(pe[6], pe[7])});
        }
        l_run += ls;
        const char *vt = lds + (2 + buf) * TILEB + khalf * 32 * ROWB;
#pragma unroll
        for (int s = 0; s < 2 * NB; ++s)
#pragma unroll
            for (int db = 0; db < NDB; ++db) {
                typedef short s4_t __attribute__((ext_vector_type(4)));
                typedef short s8_t __attribute__((ext_vector_type(8)));
                typedef __attribute__((address_space(3))) s4_t lds_s4;
                const s4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4 *)(vt + v_at[db] + (16 * s) * ROWB));
                const s4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4 *)(vt + v_at[db] + (16 * s + 8) * ROWB));
                const V8 vf = __builtin_bit_cast(V8, s8_t{lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w});
                o[db] = AttnT<T>::mfma32(vf, pf[s], o[db]);
            }
        // the copies have landed and every wavefront is done with the buffers it read
        if constexpr (MORE) {
            ODSD_WAIT_VMCNT_LGKM0(0);
            __builtin_amdgcn_s_barrier();
        }
    };

    if (n_tiles > 0) {
        const std::integral_constant<int, 0> b0;
        const std::integral_constant<int, 1> b1;
        const std::true_type yes;
        const std::false_type no;
        float16_t sa[NB], sb[NB];
        copy_k(b0, 0);
        copy_v(b0, 0);
        copy_k(b1, KT);
        load_q();
        ODSD_WAIT_VMCNT_LGKM0(0);
        __builtin_amdgcn_s_barrier();
        scores(b0, sa);
        // (K buffer 0 is refilled in the first step: every wavefront must have read it)
        ODSD_WAIT_VMCNT_LGKM0(0);
        __builtin_amdgcn_s_barrier();
        int it = 0;
        for (; it + 2 < n_tiles; it += 2) {
            step(b0, yes, it, sa, sb);
            step(b1, yes, it + 1, sb, sa);
        }
        if (it + 1 < n_tiles) {
            step(b0, yes, it, sa, sb);
            step(b1, no, it + 1, sb, sa);
        } else {
            step(b0, no, it, sa, sb);
        }
    }

    l_run += __shfl_xor(l_run, 32, ODSD_WAVE);
    if constexpr (SPLIT == 2) {
        // the second key half hands its sums to the first through LDS (free now): [dim pair register][lane]
        float *xch = (float *)lds + (size_t)rblk * (NDB * 16 + 2) * 64;
        __syncthreads();
        if (khalf == 1) {
#pragma unroll
            for (int db = 0; db < NDB; ++db)
#pragma unroll
                for (int i = 0; i < 16; ++i) xch[(db * 16 + i) * 64 + lane] = o[db][i];
            xch[(NDB * 16) * 64 + lane] = m_run;
            xch[(NDB * 16 + 1) * 64 + lane] = l_run;
        }
        __syncthreads();
        if (khalf == 1) return;
        const float m2 = xch[(NDB * 16) * 64 + lane], l2 = xch[(NDB * 16 + 1) * 64 + lane];
        const float m = fmaxf(m_run, m2), ref = m == -INFINITY ? 0.0f : m;
        const float f1 = __builtin_amdgcn_exp2f(m_run - ref), f2 = __builtin_amdgcn_exp2f(m2 - ref);
        l_run = l_run * f1 + l2 * f2;
#pragma unroll
        for (int db = 0; db < NDB; ++db)
#pragma unroll
            for (int i = 0; i < 16; ++i) o[db][i] = o[db][i] * f1 + xch[(db * 16 + i) * 64 + lane] * f2;
    }
    const float inv = l_run > 0.0f ? 1.0f / l_run : 0.0f;
    if (row_ok) {
        uint16_t *op = (uint16_t *)p.out + ((size_t)(q0 + tok) * p.H + kvh * Gq + hq) * HD + 4 * h;
#pragma unroll
        for (int db = 0; db < NDB; ++db)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
                const u32x2 v = {AttnT<T>::pack2(o[db][4 * q] * inv, o[db][4 * q + 1] * inv),
                                 AttnT<T>::pack2(o[db][4 * q + 2] * inv, o[db][4 * q + 3] * inv)};
                *(u32x2 *)(op + 32 * db + 8 * q) = v;
            }
    }
}

bool odsd_attn_prefill_supported(const AttnParams &p, int head_dim, int max_q, int max_k) {
    // byte offsets inside one sequence's keys are 32 bits wide
    if ((int64_t)max_k * p.KVH * head_dim * 2 >= (1LL << 32)) return false;
    const int64_t rows = (int64_t)max_q * (p.H / p.KVH);
    if (rows <= 64) return false;
    // Few query rows on many keys (a short chunk on top of a long prompt): a workgroup here walks all of
    // them in turn, 0.55 us per 64, while the decode / verify kernel slices them over the chip.
    return (int64_t)p.n_seqs * p.KVH * ((rows + 63) / 64) >= 128 || max_k <= 512;
}

void odsd_launch_attn_prefill(const AttnParams &p, int dtype, int head_dim, int max_q, hipStream_t st) {
    const int64_t rows = (int64_t)max_q * (p.H / p.KVH);
    const unsigned nx = (unsigned)(p.n_seqs * p.KVH);
    // up to 320 workgroups of 128 rows (256 CUs): halved ones are faster (300 tokens of 32 / 4 heads 9.0
    // against 10.8 us, 1000 tokens, 252 workgroups, 18.6 against 21.9; 1500 tokens, 376, 32.8 against 32.2)
    const bool split = (int64_t)nx * ((rows + 127) / 128) <= 320;
    const dim3 grid(nx, (unsigned)(split ? (rows + 63) / 64 : (rows + 127) / 128));
#define PREFILL_GO(T, HDV)                                                          \
    do {                                                                            \
        if (split) attn_prefill_kernel<T, HDV, 2><<<grid, 256, 0, st>>>(p);         \
        else attn_prefill_kernel<T, HDV, 1><<<grid, 256, 0, st>>>(p);               \
    } while (0)
    if (dtype == ODSD_DT_F16) {
        if (head_dim == 128) PREFILL_GO(half_t, 128);
        else PREFILL_GO(half_t, 64);
    } else {
        if (head_dim == 128) PREFILL_GO(__bf16, 128);
        else PREFILL_GO(__bf16, 64);
    }
#undef PREFILL_GO
}
