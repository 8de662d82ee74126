// The top-k selection shared by the router kernels and the expert kernels that route for themselves: the
// order-preserving integer key of a logit, the wavefront arg-max on (key, id), the selection of a token.
#pragma once
#include "common.h"

// total order on doubles as unsigned keys: larger value <=> larger key
__device__ __forceinline__ uint64_t order_key(double v) {
    if (v == 0.0) v = 0.0;   // -0 and +0 compare equal, so they must share a key
    const uint64_t b = (uint64_t)__double_as_longlong(v);
    return (b >> 63) ? ~b : (b | 0x8000000000000000ull);
}

// Wavefront arg-max on (key, -id) with DPP moves: every lane offers one candidate (a lane with nothing
// to offer passes key 0 -- no finite value maps to it -- and the largest id); the largest key wins,
// among equal keys the lowest id.  Returns the winner's id in every lane.
__device__ __forceinline__ int wave_argmax(const uint64_t key, int id) {
    uint32_t klo = (uint32_t)key, khi = (uint32_t)(key >> 32);
#define ODSD_ARGMAX_STEP(CTRL, ROWMASK)                                                                          \
    {                                                                                                            \
        const uint32_t olo = (uint32_t)__builtin_amdgcn_update_dpp((int)klo, (int)klo, CTRL, ROWMASK, 0xF, false); \
        const uint32_t ohi = (uint32_t)__builtin_amdgcn_update_dpp((int)khi, (int)khi, CTRL, ROWMASK, 0xF, false); \
        const int oe = __builtin_amdgcn_update_dpp(id, id, CTRL, ROWMASK, 0xF, false);                          \
        const uint64_t ok = ((uint64_t)ohi << 32) | olo, mk = ((uint64_t)khi << 32) | klo;                       \
        const bool better = ok > mk || (ok == mk && oe < id);                                                    \
        klo = better ? olo : klo;                                                                                \
        khi = better ? ohi : khi;                                                                                \
        id = better ? oe : id;                                                                                   \
    }
    ODSD_ARGMAX_STEP(0x111, 0xF)   // row_shr:1
    ODSD_ARGMAX_STEP(0x112, 0xF)   // row_shr:2
    ODSD_ARGMAX_STEP(0x114, 0xF)   // row_shr:4
    ODSD_ARGMAX_STEP(0x118, 0xF)   // row_shr:8   -> lane 15 of every row holds the row's best
    ODSD_ARGMAX_STEP(0x142, 0xA)   // row_bcast:15 into rows 1 and 3
    ODSD_ARGMAX_STEP(0x143, 0xC)   // row_bcast:31 into rows 2 and 3 -> lane 63 holds the best
#undef ODSD_ARGMAX_STEP
    return __builtin_amdgcn_readlane(id, 63);
}

// largest value of a 32-bit word over the wavefront, in every lane
__device__ __forceinline__ uint32_t wave_max_u32(uint32_t v) {
#define ODSD_MAX_STEP(CTRL, ROWMASK)                                                                      \
    {                                                                                                     \
        const uint32_t o = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, ROWMASK, 0xF, false);   \
        v = o > v ? o : v;                                                                                \
    }
    ODSD_MAX_STEP(0x111, 0xF)   // the lane pattern of wave_argmax
    ODSD_MAX_STEP(0x112, 0xF)
    ODSD_MAX_STEP(0x114, 0xF)
    ODSD_MAX_STEP(0x118, 0xF)
    ODSD_MAX_STEP(0x142, 0xA)
    ODSD_MAX_STEP(0x143, 0xC)
#undef ODSD_MAX_STEP
    return (uint32_t)__builtin_amdgcn_readlane((int)v, 63);
}

// wave_argmax, the upper halves of the keys first: two candidates that share sign, exponent and 20 bits of
// mantissa are rare, and a maximum of single words is one instruction per step instead of ten (K = 8 of
// E = 128: the top-k kernel 5.3 -> 4.3 us at T = 256).  Every lane's id must be its own.
__device__ __forceinline__ int wave_best(const uint64_t key, const int id) {
    const uint32_t hi = (uint32_t)(key >> 32);
    const uint32_t top = wave_max_u32(hi);
    const uint64_t who = __ballot(hi == top);
    if ((who & (who - 1)) == 0) return __builtin_amdgcn_readlane(id, __builtin_ctzll(who));
    return wave_argmax(key, id);
}

// V = logits per lane (experts lane, lane + 64, ...): 1, 2, 4 or 8 for E <= 64, 128, 256, 512
// Token t's logits into the lanes: partial sums in slice order; the loads of one slice batch are independent of each other.
template <int V>
__device__ __forceinline__ void sum_logits(const double *__restrict__ partial, const int t, int T, int E, int S, double (&lg)[V]) {
    const int lane = lane_id();
#pragma unroll
    for (int v = 0; v < V; ++v) lg[v] = 0.0;
    constexpr int SB = V <= 2 ? 8 : 4;   // slices loaded together
    for (int s0 = 0; s0 < S; s0 += SB) {
        double part[SB][V];
#pragma unroll
        for (int u = 0; u < SB; ++u)
#pragma unroll
            for (int v = 0; v < V; ++v) {
                const int e = lane + 64 * v;
                part[u][v] = (e < E && s0 + u < S) ? partial[((size_t)(s0 + u) * T + t) * E + e] : 0.0;
            }
#pragma unroll
        for (int u = 0; u < SB; ++u)
#pragma unroll
            for (int v = 0; v < V; ++v) lg[v] += part[u][v];
    }
}

// The n largest logits in descending order, ties to the lower expert: lane k < n keeps the k-th winner and its logit.
// Returns the bits of this lane's experts that were taken (those past E among them).
template <int V>
__device__ __forceinline__ uint32_t select_top(const double (&lg)[V], const int n, const int E, int &my_e, double &my_l, double &l_max) {
    const int lane = lane_id();
    uint64_t key[V];
    uint32_t taken = 0;   // bit v set: expert lane + 64 v already selected
#pragma unroll
    for (int v = 0; v < V; ++v) {
        key[v] = order_key(lg[v]);
        if (lane + 64 * v >= E) taken |= 1u << v;
    }
    my_e = 0;
    my_l = 0.0;
    l_max = 0.0;
    for (int k = 0; k < n; ++k) {
        // best remaining candidate of this lane: largest key, then lowest expert.  A lane with
        // nothing left offers key 0 (no finite logit maps to it) and the largest expert id.
        uint64_t bk = 0;
        int be = 0x7fffffff;
#pragma unroll
        for (int v = 0; v < V; ++v) {
            if (!((taken >> v) & 1u)) {
                if (be == 0x7fffffff || key[v] > bk) {
                    bk = key[v];
                    be = lane + 64 * v;
                }
            }
        }
        const int we = wave_best(bk, be);   // the same in every lane
        // the winner's logit sits in lane (we & 63), slot (we >> 6)
        double cand = lg[0];
#pragma unroll
        for (int v = 1; v < V; ++v) cand = (we >> 6) == v ? lg[v] : cand;
        const uint64_t cb = (uint64_t)__double_as_longlong(cand);
        const uint32_t wlo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)cb, we & 63);
        const uint32_t whi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(cb >> 32), we & 63);
        const double wl = __longlong_as_double((long long)(((uint64_t)whi << 32) | wlo));
        if ((we & 63) == lane) taken |= 1u << (we >> 6);
        if (lane == k) { my_e = we; my_l = wl; }
        if (k == 0) l_max = wl;
    }
    return taken;
}

// What lane k < K holds of the k-th winner, and its weight: in fp32, differences are taken in fp64 before the cast.
template <int V>
__device__ __forceinline__ void topk_weights(const double (&lg)[V], const int my_e, const double my_l, const double l_max,
                                             const int t, int E, int K, int renorm, int32_t *__restrict__ idx,
                                             float *__restrict__ w, int64_t *__restrict__ idx64) {
    const int lane = lane_id();
    float num = 0.0f;
    if (lane < K) num = expf((float)(my_l - l_max));
    float den;
    if (renorm) {
        den = wave_sum(num);
    } else {
        float part = 0.0f;
#pragma unroll
        for (int v = 0; v < V; ++v)
            if (lane + 64 * v < E) part += expf((float)(lg[v] - l_max));
        den = wave_sum(part);
    }
    if (lane < K) {
        const size_t o = (size_t)t * K + lane;
        idx[o] = my_e;
        w[o] = num / den;
        if (idx64) idx64[o] = (int64_t)my_e;
    }
}

// the selection for token t by one wavefront; lane k < K returns the k-th winner's expert id
// (idx null: nothing but that)
template <int V>
__device__ __forceinline__ int topk_token(const double *__restrict__ partial, const int t, int T, int E,
                                          int K, int S, int renorm, int32_t *__restrict__ idx,
                                          float *__restrict__ w, int64_t *__restrict__ idx64,
                                          double *__restrict__ logits) {
    const int lane = lane_id();

    double lg[V];
    sum_logits<V>(partial, t, T, E, S, lg);
    if (logits) {
#pragma unroll
        for (int v = 0; v < V; ++v)
            if (lane + 64 * v < E) logits[(size_t)t * E + lane + 64 * v] = lg[v];
    }
    int my_e;              // lane k keeps the k-th winner
    double my_l, l_max;
    select_top<V>(lg, K, E, my_e, my_l, l_max);

    if (!idx) return my_e;
    topk_weights<V>(lg, my_e, my_l, l_max, t, E, K, renorm, idx, w, idx64);
    return my_e;
}
