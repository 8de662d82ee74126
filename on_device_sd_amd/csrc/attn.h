// Pieces shared by the attention kernels: launch parameters and the element-type dependent operations.
#pragma once
#include "common.h"
#include <type_traits>

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float float2_t __attribute__((ext_vector_type(2)));
typedef float float16_t __attribute__((ext_vector_type(16)));

struct AttnParams {
    const void *q;             // [n_tokens, H, HD]
    const void *k_cache;       // [num_slots, KVH * HD]
    const void *v_cache;
    void *out;                 // [n_tokens, H, HD]
    const int32_t *q_lens;     // [n_seqs] or null (1 each)
    const int32_t *context_lens;
    const int32_t *block_tables;   // [n_seqs, max_blocks]
    int n_seqs, H, KVH, Gq, max_blocks, block_size;   // Gq: query heads per KV head
    int64_t num_slots;
    float scale_log2e;         // softmax scale * log2(e)
    // variable-length mode (prefill): q / k / v rows of sequence s are q[cu_q[s] ..], k[cu_k[s] ..]
    // (contiguous, no block table); both null in paged mode
    const int32_t *cu_q, *cu_k;
    int max_keys, max_rg;      // streaming kernels: the keys and row groups of a sequence that the launch is sized for
    int n_wg;                  // workgroups that share the work
    int whole;                 // no unit is split and a workgroup's number says which is its own: row groups per
                               // (sequence, KV head); 0: the units are found in the list
    int v_once;                // tile kernel: V is read nontemporally (the stream form always does)
    float *part;               // its partial results, two slots per workgroup: [rows][HD + 4]
};

template <typename T> struct AttnT;
template <> struct AttnT<half_t> {
    typedef half8_t V8;
    __device__ static __forceinline__ float4_t mfma(V8 a, V8 b, float4_t c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
    }
    __device__ static __forceinline__ float16_t mfma32(V8 a, V8 b, float16_t c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
    }
    // two values, round to nearest even, as one 32-bit word (a in the low half)
    __device__ static __forceinline__ uint32_t pack2(float a, float b) {
        typedef _Float16 h2 __attribute__((ext_vector_type(2)));
        typedef float f2 __attribute__((ext_vector_type(2)));
        return __builtin_bit_cast(uint32_t, __builtin_convertvector(f2{a, b}, h2));
    }
};
template <> struct AttnT<__bf16> {
    typedef bf16x8_t V8;
    __device__ static __forceinline__ float4_t mfma(V8 a, V8 b, float4_t c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
    }
    __device__ static __forceinline__ float16_t mfma32(V8 a, V8 b, float16_t c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
    }
    __device__ static __forceinline__ uint32_t pack2(float a, float b) {   // v_cvt_pk_bf16_f32
        typedef __bf16 b2 __attribute__((ext_vector_type(2)));
        typedef float f2 __attribute__((ext_vector_type(2)));
        return __builtin_bit_cast(uint32_t, __builtin_convertvector(f2{a, b}, b2));
    }
};


// causal attention over packed sequences with many query rows (attn_prefill.hip)
bool odsd_attn_prefill_supported(const AttnParams &p, int head_dim, int max_q, int max_k);
void odsd_launch_attn_prefill(const AttnParams &p, int dtype, int head_dim, int max_q, hipStream_t st);
