// Codes as matrix operands without scale and zero point, shared by the kernels that apply those to group sums.
#pragma once
#include "w4_gemm.h"

// Codes as fp16 without the per-weight scale and zero point.  (x & mask) | magic turns a nibble pair
// into fp16 values offset + q: the low nibbles of the two halves of a word with magic 0x6400
// (1024 + q, one unit in the last place = 1), the high nibbles with 0x5400 (64 + q, one unit in the
// last place = 1/16, so the nibble's 16 q is q).  Element order of the result is that of the MFMA A
// operand: (k0,k1) and (k4,k5) carry 1024 + q, (k2,k3) and (k6,k7) carry 64 + q.  The offsets are
// taken out again through the accumulator's start value (see group_sums), and scale and zero point
// are applied to the group's sum instead of to every weight: 5 vector instructions per 8 weights
// instead of 13.
struct RawConsts {
    uint32_t m_lo, m_hi, magic_lo, magic_hi;
};
__device__ __forceinline__ RawConsts raw_consts() {
    RawConsts c{0x000F000Fu, 0x00F000F0u, 0x64006400u, 0x54005400u};
    asm volatile("" : "+s"(c.m_lo), "+s"(c.m_hi), "+v"(c.magic_lo), "+v"(c.magic_hi));
    return c;
}
__device__ __forceinline__ half8_t raw_word(const RawConsts &c, const uint32_t x) {
    const uint32_t xs = x >> 8;
    const uint4_t t = {(x & c.m_lo) | c.magic_lo, (x & c.m_hi) | c.magic_hi, (xs & c.m_lo) | c.magic_lo,
                       (xs & c.m_hi) | c.magic_hi};
    return __builtin_bit_cast(half8_t, t);
}
#define ODSD_RAW_OFFSET_LO 1024.0f
#define ODSD_RAW_OFFSET_HI 64.0f

typedef float float2_t __attribute__((ext_vector_type(2)));

__device__ __forceinline__ uint64_t uniform_u64(const uint64_t v) {
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v), hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
    return ((uint64_t)hi << 32) | lo;
}

// Nothing moves across this point: the scheduling fence binds the machine scheduler, the empty
// statement with a memory clobber binds the instruction selector's ordering of a long straight-line
// block (without it the loads of many later steps are hoisted to the top of the unrolled stream and
// their results spilled).
#define ODSD_FENCE()                         \
    do {                                     \
        __builtin_amdgcn_sched_barrier(0);   \
        asm volatile("" ::: "memory");       \
        __builtin_amdgcn_sched_barrier(0);   \
    } while (0)
