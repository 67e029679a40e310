// Vector types and the quant-block -> f16 MFMA operand unpackers shared by the few-row GEMM kernels.
#pragma once

#include "common.h"

namespace {

typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
typedef _Float16 half4_t __attribute__((ext_vector_type(4)));
typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef float float4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));

__device__ __forceinline__ half2_t as_half2(uint32_t bits) { return __builtin_bit_cast(half2_t, bits); }

__device__ __forceinline__ half2_t splat(_Float16 v) {
    half2_t r = {v, v};
    return r;
}

// The f16 constants 1024.0 and 64.0 (as pairs) whose mantissas receive the nibbles.  They are
// passed through an empty asm once per kernel so the compiler sees VGPR values, not literals:
// (w & mask) | magic then selects as one v_and_or_b32 (mask in an SGPR) instead of two
// instructions with a literal each.
struct Q4KMagic {
    uint32_t lo, hi;
};
__device__ __forceinline__ Q4KMagic q4k_magic() {
    Q4KMagic m = {0x64006400u, 0x54005400u};
    asm volatile("" : "+v"(m.lo), "+v"(m.hi));
    return m;
}

// Eight f16 weights of one MFMA from two dwords of quant bytes.
//   HIGH = false: low nibbles,  1024 + q  via magic 0x6400, mask 0x000F
//   HIGH = true : high nibbles,   64 + q  via magic 0x5400, mask 0x00F0
// s2 = (s, s), c2 = (-1024 s, -1024 s) or (-64 s, -64 s).
template <bool HIGH>
__device__ __forceinline__ half8_t unpack_scale(uint32_t w0, uint32_t w1, half2_t s2, half2_t c2, uint32_t magic) {
    constexpr uint32_t mask = HIGH ? 0x00F000F0u : 0x000F000Fu;
    half2_t p0 = __builtin_elementwise_fma(as_half2((w0 & mask) | magic), s2, c2);
    half2_t p1 = __builtin_elementwise_fma(as_half2(((w0 >> 8) & mask) | magic), s2, c2);
    half2_t p2 = __builtin_elementwise_fma(as_half2((w1 & mask) | magic), s2, c2);
    half2_t p3 = __builtin_elementwise_fma(as_half2(((w1 >> 8) & mask) | magic), s2, c2);
    half8_t r = {p0[0], p0[1], p1[0], p1[1], p2[0], p2[1], p3[0], p3[1]};
    return r;
}

// ---- the Q4_K minima as one MFMA per super-block ----
// Lane (m, g) of the A operand holds the sums of row m's rounded activations over sub-blocks 2g and 2g + 1, each split
// into f16 parts, in k-slots {hi, hi', lo, lo', over, over', 0, 0}; the B operand holds the lane's two (negated) minima
// in the matching slots.  hi + lo carries 22 bits of the sum.  `over` (in units of 32) keeps a sum that would round past
// the largest f16 - 32 activations of about 2000 - finite; it is zero otherwise and then adds nothing.  The slab, tiled
// and expert kernels hold hi and lo alone (LDS, and the chain of a lightly loaded wave): such a sum is infinite there,
// its row's results come out NaN, and the wave computes its tile again with all three parts (q4k_again, gemm_fewrow.hip).
struct Q4KSumParts {
    _Float16 hi, lo, over;
};
__device__ __forceinline__ Q4KSumParts q4k_sum_parts(float sum) {
    Q4KSumParts p;
    p.over = fabsf(sum) >= 65520.0f ? static_cast<_Float16>(sum * 0.03125f) : static_cast<_Float16>(0.0f);
    const float rest = sum - 32.0f * static_cast<float>(p.over);
    p.hi = static_cast<_Float16>(rest);
    p.lo = static_cast<_Float16>(rest - static_cast<float>(p.hi));
    return p;
}
// Eight consecutive values of a row: added pairwise (the order in which the slab and the streaming kernel add them, four
// values to a thread), or one after the other (the expert kernels' order).
__device__ __forceinline__ float q4k_octet_sum(const _Float16 *h) {
    return ((static_cast<float>(h[0]) + static_cast<float>(h[1])) + (static_cast<float>(h[2]) + static_cast<float>(h[3]))) +
           ((static_cast<float>(h[4]) + static_cast<float>(h[5])) + (static_cast<float>(h[6]) + static_cast<float>(h[7])));
}
__device__ __forceinline__ float q4k_octet_sum_seq(const _Float16 *h) {
    float s = 0.0f;
#pragma unroll
    for (int i = 0; i < 8; i++) s += static_cast<float>(h[i]);
    return s;
}
// A lane's A operand from the sums of its two sub-blocks.
__device__ __forceinline__ half8_t q4k_sum_operand(float sum0, float sum1) {
    const Q4KSumParts s0 = q4k_sum_parts(sum0), s1 = q4k_sum_parts(sum1);
    const _Float16 zero = static_cast<_Float16>(0.0f);
    const half8_t a = {s0.hi, s1.hi, s0.lo, s1.lo, s0.over, s1.over, zero, zero};
    return a;
}
__device__ __forceinline__ half8_t q4k_min_operand(half2_t m) {
    const _Float16 k32 = static_cast<_Float16>(32.0f), zero = static_cast<_Float16>(0.0f);
    const half8_t b = {m[0], m[1], m[0], m[1], m[0] * k32, m[1] * k32, zero, zero};
    return b;
}

// Eight f16 weights of one MFMA: q = nibble | (two qh bits << 4), value round(q s).
//   HIGH = false: low nibbles, bits pre-shifted to 0..1:   1024 + q via magic 0x6400, c = -1024 s
//   HIGH = true : high nibbles (four bits up), qh bits go eight bits up: 64 + q via 0x5400, c = -64 s
template <bool HIGH>
__device__ __forceinline__ half8_t unpack6(uint32_t w0, uint32_t w1, uint32_t h0, uint32_t h1, half2_t s2, half2_t c2,
                                           uint32_t magic) {
    constexpr uint32_t mask = HIGH ? 0x00F000F0u : 0x000F000Fu;
    constexpr int up = HIGH ? 8 : 4;
    auto one = [&](uint32_t w, uint32_t h) {
        const uint32_t bits = ((w & mask) | magic) | ((h & 0x00030003u) << up);
        return __builtin_elementwise_fma(as_half2(bits), s2, c2);
    };
    const half2_t p0 = one(w0, h0), p1 = one(w0 >> 8, h0 >> 8), p2 = one(w1, h1), p3 = one(w1 >> 8, h1 >> 8);
    half8_t r = {p0[0], p0[1], p1[0], p1[1], p2[0], p2[1], p3[0], p3[1]};
    return r;
}

// ---- Q6_K in tiled, field-planar order: where a tile's 3360 bytes hold which field (dflash_repack_q6k_tiled) ----
constexpr int kQ6TileBytes = 16 * DFL_Q6_K_BYTES;  // 3360
constexpr int kQ6TQh = 2048, kQ6TSc = 3072, kQ6TD = 3328;
__host__ __device__ __forceinline__ int q6t_ql_piece(int row, int p) { return row * 128 + ((p ^ (row & 7)) << 4); }
__host__ __device__ __forceinline__ int q6t_qh_piece(int row, int p) { return kQ6TQh + row * 64 + ((p ^ ((row >> 1) & 3)) << 4); }

}  // namespace
