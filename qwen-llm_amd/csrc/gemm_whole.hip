// Whole-K few-row GEMM for the small matrices of a verify or draft layer (a few MB each):
//   Y[n_rows][n_out] = X[n_rows][n_in] . W^T,  X handed over in MFMA fragment order (common.h, "XF").
// Same contraction as encode_mat_mat_dispatch_dflash_verify (metal_forward/dispatch.rs:365-378, kernel
// kernels/mat_mat_fewrow_gen.metal:374-474); used inside the layer loops where the kernel that produces X can
// write it in fragment order.
//
// Why a second kernel family.  The streaming kernels (gemm_fewrow.hip) give every CU a contiguous run of
// (tile group x super-block) stages; where a run cuts a tile group the K sum is split over workgroups and a second
// launch adds the partial tiles.  For a 50 MB matrix that is the right shape.  For the 6-9 MB projections of a
// 2048-wide model it is two dependent launches of 7-10 us + 4 us in which every wave sees one or two stages: the
// time is launch latency, the trip for the first bytes, and a reduction through memory.  Here every (tile, stage)
// of the matrix is one wave-slot of ONE round of the chip:
//   * a workgroup owns `tl` output units over the whole K; wave = (tile lane, K slice), a slice is one or two
//     super-blocks; every load of a wave (weights straight into registers, the stage's eight activation fragments
//     with eight coalesced 16-byte loads from the XF buffer, which sits in L2) is issued before anything is waited for;
//   * the slices' partial tiles are added in LDS in slice order (deterministic), by the wave of slice 0, which writes Y.
// No partial tiles in memory, no second launch, no loop.  A (row, column) result depends on nothing but its own
// activation row and weight row, so a 16-row block and a single row give the same bits.
//
// Arithmetic: that of the streaming kernels (exact f16 integers from the quant bits, one packed fma with
// s = d * scale, f32 accumulation on v_mfma_f32_16x16x32_f16; the Q4_K minima and the Q6_K offset through a twin MFMA
// of the same activation fragment into a second accumulator that is subtracted at the end).  Where a target's Q4_K matrix
// has 16 super-blocks of K or more and one round of tiles (Q4S; dfl_whole_by_sums) the minima go by one MFMA over the activations' sub-block sums ahead of the
// eight: the same MFMAs are what a prompt's many-row product is made of (gemm_rows.hip, whose rows have this kernel's bits),
// and twins are half of them there.  The sums cost a wave 90 vector instructions a stage (4096 -> 5120 and 5120 -> 6144 9.1 -> 9.4 us a
// launch); matrices of short K, where a launch is 4 us and a prompt's product as short, keep the twins.
#include "common.h"
#include "mfma_unpack.h"

#include <hip/hip_ext.h>

#include <algorithm>
#include <cstdlib>
#include <type_traits>

namespace {

struct WholeArgs {
    const uint8_t *w;
    const uint8_t *xf;
    float *y;
    uint8_t *y_xf;
    int y_xf_kind;
    int n_out;   // rows of w (pair mode: 2 * ffn)
    int nb;      // super-blocks per row
    int n_rows;
    int ksplit;  // K slices per unit; waves per workgroup = ksplit * tl
    int tl;      // units per workgroup
    int n_units; // plain: ceil(tiles / R) units of R consecutive tiles; pair: ffn / 16 units of (gate tile, up tile)
    int pair_off;  // pair mode: tiles between a gate tile and its up tile; 0 = plain.  (The looping kernels: workgroups of the launch.)
    uint32_t row_bytes;  // Q6_K (GGUF row order): bytes per weight row
    // several 16-row blocks against the same weights (a prefill): block i reads xf + i * xf_stride bytes and writes
    // y + i * y_stride floats (y_xf + i * y_xf_stride bytes); the last block has rows_last rows, the others 16
    int n_blocks, rows_last;
    uint32_t xf_stride, y_xf_stride;
    size_t y_stride;
};
// As kernel parameters: what a wave needs for its first loads as words of their own, fourteen at most, which arrive in its
// scalar registers (a parameter that is a structure has to be loaded, a trip of 0.5 us to memory the host has just written,
// and a division by ksplit is some forty instructions, ahead of the first weight); the rest behind them.
// (a step of 40 layers, 80 such launches: 2689 -> 2664 us)
struct WholeTail {
    uint8_t *y_xf;
    int y_xf_kind, n_blocks, rows_last;
    uint32_t xf_stride, y_xf_stride;
    size_t y_stride;
};
#define DFL_WHOLE_PARAMS                                                                                                             \
    const uint8_t *w, const uint8_t *xf, float *y, uint32_t split, uint32_t by_ksplit, int nb, int n_out, int n_units, int pair_off, \
        uint32_t row_bytes, WholeTail tail
#define DFL_WHOLE_ARGS                                                                                                                        \
    WholeArgs {                                                                                                                               \
        w, xf, y, tail.y_xf, tail.y_xf_kind, n_out, nb, static_cast<int>(split >> 16), static_cast<int>(split & 255), static_cast<int>(split >> 8 & 255), \
            n_units, pair_off, row_bytes, tail.n_blocks, tail.rows_last, tail.xf_stride, tail.y_xf_stride, tail.y_stride                      \
    }
typedef void (*whole_kernel_t)(DFL_WHOLE_PARAMS);
// by_ksplit = ceil(65536 / ksplit): x / ksplit for 0 <= x <= 512 (a wave's index, a super-block's index times a slice's)
__device__ __forceinline__ int whole_div(int x, uint32_t by_ksplit) { return static_cast<int>(static_cast<uint32_t>(x) * by_ksplit >> 16); }
void whole_launch(whole_kernel_t fn, int grid, int threads, size_t lds, hipStream_t st, const WholeArgs &a, hipEvent_t start = nullptr,
                  hipEvent_t stop = nullptr) {
    const WholeTail tail = {a.y_xf, a.y_xf_kind, a.n_blocks, a.rows_last, a.xf_stride, a.y_xf_stride, a.y_stride};
    const uint32_t split = static_cast<uint32_t>(a.ksplit | a.tl << 8 | a.n_rows << 16), by_ksplit = (65536u + a.ksplit - 1) / a.ksplit;
    hipExtLaunchKernelGGL(fn, dim3(grid), dim3(threads), lds, st, start, stop, 0, a.w, a.xf, a.y, split, by_ksplit, a.nb, a.n_out, a.n_units, a.pair_off,
                          a.row_bytes, tail);
}

// ---- Q4_K, tiled order: [tile group of 256 rows][super-block][tile][row][144-byte block] ----
struct Q4W {
    u32x4_t hdr, q0, q1;
};
__device__ __forceinline__ void load_w(Q4W &r, const WholeArgs &a, int tile, int b, int lane) {
    const int n = lane & 15, g = lane >> 4;
    const uint8_t *p = a.w + ((static_cast<size_t>(tile >> 4) * a.nb + b) * 16 + (tile & 15)) * (16 * DFL_Q4_K_BYTES) +
                       n * DFL_Q4_K_BYTES;
    r.hdr = *reinterpret_cast<const u32x4_t *>(p);
    r.q0 = *reinterpret_cast<const u32x4_t *>(p + 16 + 32 * g);
    r.q1 = *reinterpret_cast<const u32x4_t *>(p + 32 + 32 * g);
}
// The same blocks in GGUF row order (the rows of a tile a row stride apart): the same operands, so the same products.
struct Q4R : Q4W {};
__device__ __forceinline__ void load_w(Q4R &r, const WholeArgs &a, int tile, int b, int lane) {
    const int row = min(tile * 16 + (lane & 15), a.n_out - 1), g = lane >> 4;  // rows past the matrix re-read its last row; never stored
    const uint8_t *p = a.w + static_cast<size_t>(row) * a.row_bytes + static_cast<size_t>(b) * DFL_Q4_K_BYTES;
    r.hdr = *reinterpret_cast<const u32x4_t *>(p);
    r.q0 = *reinterpret_cast<const u32x4_t *>(p + 16 + 32 * g);
    r.q1 = *reinterpret_cast<const u32x4_t *>(p + 32 + 32 * g);
}
// One super-block of one tile: lane (n = weight row, g = 64-value chunk) against the eight activation fragments.
__device__ __forceinline__ void compute(const Q4W &r, const half8_t (&af)[8], int lane, uint8_t *, uint32_t sc_sel, Q4KMagic magic,
                                        float4_t &acc, float4_t &acc_sub) {
    const int g = lane >> 4;
    const u32x4_t hdr = r.hdr;
    const uint32_t upper = 0u - static_cast<uint32_t>(g >> 1);
    const uint32_t sc_lo = hdr.y & 0x3F3F3F3Fu, sc_hi = (hdr.w & 0x0F0F0F0Fu) | ((hdr.y >> 2) & 0x30303030u);
    const uint32_t mn_lo = hdr.z & 0x3F3F3F3Fu, mn_hi = ((hdr.w >> 4) & 0x0F0F0F0Fu) | ((hdr.z >> 2) & 0x30303030u);
    const uint32_t sc_word = (sc_hi & upper) | (sc_lo & ~upper), mn_word = (mn_hi & upper) | (mn_lo & ~upper);
    const half2_t dm = __builtin_bit_cast(half2_t, hdr.x);
    const half2_t p_sc = as_half2(__builtin_amdgcn_perm(0x64646464u, sc_word, sc_sel));
    const half2_t p_mn = as_half2(__builtin_amdgcn_perm(0x64646464u, mn_word, sc_sel));
    const half2_t neg = dm * splat(static_cast<_Float16>(-1024.0f));
    const half2_t S = __builtin_elementwise_fma(p_sc, splat(dm[0]), splat(neg[0]));
    const half2_t M = __builtin_elementwise_fma(p_mn, splat(dm[1]), splat(neg[1]));
    const half2_t unbias = {static_cast<_Float16>(-1024.0f), static_cast<_Float16>(-64.0f)};
    const half2_t Cs = S * unbias;
    const half2_t s2l = splat(S[0]), c2l = splat(Cs[0]);
    const half2_t s2h = splat(S[1]), c2h = splat(Cs[1]);
    const _Float16 m_lo = M[0], m_hi = M[1];
    const half8_t bml = {m_lo, m_lo, m_lo, m_lo, m_lo, m_lo, m_lo, m_lo};
    const half8_t bmh = {m_hi, m_hi, m_hi, m_hi, m_hi, m_hi, m_hi, m_hi};
    const uint32_t qw[8] = {r.q0.x, r.q0.y, r.q0.z, r.q0.w, r.q1.x, r.q1.y, r.q1.z, r.q1.w};
#pragma unroll
    for (int t = 0; t < 4; t++) {
        const half8_t bl = unpack_scale<false>(qw[2 * t], qw[2 * t + 1], s2l, c2l, magic.lo);
        acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(af[t], bl, acc, 0, 0, 0);
        acc_sub = __builtin_amdgcn_mfma_f32_16x16x32_f16(af[t], bml, acc_sub, 0, 0, 0);
    }
#pragma unroll
    for (int t = 0; t < 4; t++) {
        const half8_t bh = unpack_scale<true>(qw[2 * t], qw[2 * t + 1], s2h, c2h, magic.hi);
        acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(af[4 + t], bh, acc, 0, 0, 0);
        acc_sub = __builtin_amdgcn_mfma_f32_16x16x32_f16(af[4 + t], bmh, acc_sub, 0, 0, 0);
    }
}

// The minima by the sums of the activations (the A operand of gemm_rows.hip's xf_sums_kernel, bit for bit): a lane's eight
// fragments are eight octets of its row, the first four one sub-block and the last four the next.
struct Q4S : Q4W {};
// h0 + h1 and h2 + h3 of a fragment's half (dwords (h0, h2) and (h1, h3)), each one rounding to f32
__device__ __forceinline__ float pair_sums(uint32_t a, uint32_t b) {
    float lo, hi;
    asm("v_fma_mix_f32 %0, %1, 1.0, %2 op_sel_hi:[1,0,1]" : "=v"(lo) : "v"(a), "v"(b));
    asm("v_fma_mix_f32 %0, %1, 1.0, %2 op_sel:[1,0,1] op_sel_hi:[1,0,1]" : "=v"(hi) : "v"(a), "v"(b));
    return lo + hi;
}
__device__ __forceinline__ half8_t sum_operand(const half8_t (&af)[8]) {
    float o[8];
#pragma unroll
    for (int t = 0; t < 8; t++) {
        const u32x4_t f = __builtin_bit_cast(u32x4_t, af[t]);
        o[t] = pair_sums(f.x, f.y) + pair_sums(f.z, f.w);
    }
    return q4k_sum_operand((o[0] + o[1]) + (o[2] + o[3]), (o[4] + o[5]) + (o[6] + o[7]));
}

// The same in two steps, for a launch that multiplies many row blocks with one set of weights: the B operands of a
// super-block's eight MFMAs once (unpack), then only the MFMAs per row block (mma), in compute()'s order.
struct Q4F {
    half8_t b[8];
    _Float16 m_lo, m_hi;
};
__device__ __forceinline__ void unpack(const Q4W &r, int lane, uint8_t *, uint32_t sc_sel, Q4KMagic magic, Q4F &f) {
    const int g = lane >> 4;
    const u32x4_t hdr = r.hdr;
    const uint32_t upper = 0u - static_cast<uint32_t>(g >> 1);
    const uint32_t sc_lo = hdr.y & 0x3F3F3F3Fu, sc_hi = (hdr.w & 0x0F0F0F0Fu) | ((hdr.y >> 2) & 0x30303030u);
    const uint32_t mn_lo = hdr.z & 0x3F3F3F3Fu, mn_hi = ((hdr.w >> 4) & 0x0F0F0F0Fu) | ((hdr.z >> 2) & 0x30303030u);
    const uint32_t sc_word = (sc_hi & upper) | (sc_lo & ~upper), mn_word = (mn_hi & upper) | (mn_lo & ~upper);
    const half2_t dm = __builtin_bit_cast(half2_t, hdr.x);
    const half2_t p_sc = as_half2(__builtin_amdgcn_perm(0x64646464u, sc_word, sc_sel));
    const half2_t p_mn = as_half2(__builtin_amdgcn_perm(0x64646464u, mn_word, sc_sel));
    const half2_t neg = dm * splat(static_cast<_Float16>(-1024.0f));
    const half2_t S = __builtin_elementwise_fma(p_sc, splat(dm[0]), splat(neg[0]));
    const half2_t M = __builtin_elementwise_fma(p_mn, splat(dm[1]), splat(neg[1]));
    const half2_t unbias = {static_cast<_Float16>(-1024.0f), static_cast<_Float16>(-64.0f)};
    const half2_t Cs = S * unbias;
    const half2_t s2l = splat(S[0]), c2l = splat(Cs[0]);
    const half2_t s2h = splat(S[1]), c2h = splat(Cs[1]);
    f.m_lo = M[0];
    f.m_hi = M[1];
    const uint32_t qw[8] = {r.q0.x, r.q0.y, r.q0.z, r.q0.w, r.q1.x, r.q1.y, r.q1.z, r.q1.w};
#pragma unroll
    for (int t = 0; t < 4; t++) {
        f.b[t] = unpack_scale<false>(qw[2 * t], qw[2 * t + 1], s2l, c2l, magic.lo);
        f.b[4 + t] = unpack_scale<true>(qw[2 * t], qw[2 * t + 1], s2h, c2h, magic.hi);
    }
}
__device__ __forceinline__ void mma(const Q4F &f, const half8_t (&af)[8], float4_t &acc, float4_t &acc_sub) {
    const half8_t bml = {f.m_lo, f.m_lo, f.m_lo, f.m_lo, f.m_lo, f.m_lo, f.m_lo, f.m_lo};
    const half8_t bmh = {f.m_hi, f.m_hi, f.m_hi, f.m_hi, f.m_hi, f.m_hi, f.m_hi, f.m_hi};
#pragma unroll
    for (int t = 0; t < 8; t++) {
        acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(af[t], f.b[t], acc, 0, 0, 0);
        acc_sub = __builtin_amdgcn_mfma_f32_16x16x32_f16(af[t], t < 4 ? bml : bmh, acc_sub, 0, 0, 0);
    }
}

struct Q4SF : Q4F {};
__device__ __forceinline__ void mma(const Q4SF &f, const half8_t (&af)[8], float4_t &acc, float4_t &) {
    const half2_t m = {-f.m_lo, -f.m_hi};
    acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(sum_operand(af), q4k_min_operand(m), acc, 0, 0, 0);
#pragma unroll
    for (int t = 0; t < 8; t++) acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(af[t], f.b[t], acc, 0, 0, 0);
}
__device__ __forceinline__ void compute(const Q4S &r, const half8_t (&af)[8], int lane, uint8_t *area, uint32_t sc_sel, Q4KMagic magic,
                                        float4_t &acc, float4_t &acc_sub) {
    Q4SF f;
    unpack(r, lane, area, sc_sel, magic, f);
    mma(f, af, acc, acc_sub);
}

// ---- Q6_K, GGUF row order: 210-byte blocks (ql[128], qh[64], scales[16], d), rows 2-byte aligned ----
// A tile's stage is 16 runs of 210 bytes a row stride apart.  They are loaded as 208 pieces of 16 bytes (13 per row,
// consecutive lanes taking consecutive pieces: row-contiguous requests) plus d, and pass through a wave-private LDS
// area with a 240-byte row stride, from which lane (n, g) picks its operands with aligned reads.  (Loading each lane's
// operands straight from memory, seven scattered unaligned loads, measured 8 us per launch against 4.8 us for the
// same bytes of Q4_K.)
constexpr int kQ6RowStride = 240;
constexpr int kQ6AreaBytes = 16 * kQ6RowStride;
typedef u32x4_t u32x4_unaligned_t __attribute__((aligned(2)));
struct Q6W {
    u32x4_t p[4];
    uint32_t d;
};
__device__ __forceinline__ void load_w(Q6W &r, const WholeArgs &a, int tile, int b, int lane) {
    const uint8_t *base = a.w + static_cast<size_t>(b) * DFL_Q6_K_BYTES;
    const int last = a.n_out - 1;  // rows past the matrix re-read its last row; never stored
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const int i = min(lane + 64 * j, 207);
        const int row = min(tile * 16 + i / 13, last);
        r.p[j] = *reinterpret_cast<const u32x4_unaligned_t *>(base + static_cast<size_t>(row) * a.row_bytes + 16 * (i % 13));
    }
    r.d = *reinterpret_cast<const uint16_t *>(base + static_cast<size_t>(min(tile * 16 + (lane & 15), last)) * a.row_bytes + 208);
}
// A lane's operands of one super-block of one weight row (lane (n, g): half h = g / 2, quarters (g & 1) and 2 + (g & 1)):
// 32 bytes of ql, 32 of qh, the four scales of its two quarters and d.
struct Q6Ops {
    u32x4_t qa, qb, ha, hb;
    uint32_t sc4, sc4h;  // low 16 bits: the two int8 scales of the low (high) quarter
    float d;
};
// The lane's operands out of a wave-private LDS area that holds the tile's sixteen raw 210-byte blocks, rows 240 bytes apart.
__device__ __forceinline__ Q6Ops q6_stage_through_lds(const Q6W &r, int lane, uint8_t *area) {
    const int n = lane & 15, g = lane >> 4, h = g >> 1, odd = g & 1;
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const int i = lane + 64 * j;
        if (i < 208) *reinterpret_cast<u32x4_t *>(area + (i / 13) * kQ6RowStride + 16 * (i % 13)) = r.p[j];
    }
    if (lane < 16) *reinterpret_cast<uint16_t *>(area + lane * kQ6RowStride + 208) = static_cast<uint16_t>(r.d);
    __builtin_amdgcn_wave_barrier();
    const uint8_t *rowp = area + n * kQ6RowStride;
    Q6Ops o;
    o.qa = *reinterpret_cast<const u32x4_t *>(rowp + 64 * h + 32 * odd);
    o.qb = *reinterpret_cast<const u32x4_t *>(rowp + 64 * h + 32 * odd + 16);
    o.ha = *reinterpret_cast<const u32x4_t *>(rowp + 128 + 32 * h);
    o.hb = *reinterpret_cast<const u32x4_t *>(rowp + 128 + 32 * h + 16);
    o.sc4 = (*reinterpret_cast<const uint32_t *>(rowp + 192 + 8 * h) >> (16 * odd)) & 0xffffu;
    o.sc4h = (*reinterpret_cast<const uint32_t *>(rowp + 192 + 8 * h + 4) >> (16 * odd)) & 0xffffu;
    o.d = __half2float(__ushort_as_half(*reinterpret_cast<const uint16_t *>(rowp + 208)));
    __builtin_amdgcn_wave_barrier();  // (the area is rewritten by this wave's next tile only after these reads: LDS runs a wave's accesses in order)
    return o;
}
__device__ __forceinline__ void q6_compute(const Q6Ops &o, const half8_t (&af)[8], int lane, Q4KMagic magic, float4_t &acc, float4_t &acc_sub) {
    const int odd = (lane >> 4) & 1;
    const int hs = 2 * odd;
    const uint32_t hq[8] = {o.ha.x >> hs, o.ha.y >> hs, o.ha.z >> hs, o.ha.w >> hs, o.hb.x >> hs, o.hb.y >> hs, o.hb.z >> hs, o.hb.w >> hs};
    const uint32_t ql[8] = {o.qa.x, o.qa.y, o.qa.z, o.qa.w, o.qb.x, o.qb.y, o.qb.z, o.qb.w};
    const float d = o.d;
    auto scale = [&](uint32_t pair, int j) { return static_cast<_Float16>(d * static_cast<float>(static_cast<int8_t>(pair >> (8 * j)))); };
    const _Float16 s_l0 = scale(o.sc4, 0), s_l1 = scale(o.sc4, 1), s_h0 = scale(o.sc4h, 0), s_h1 = scale(o.sc4h, 1);
#pragma unroll
    for (int t = 0; t < 4; t++) {
        const _Float16 sl = (t >> 1) ? s_l1 : s_l0;
        const half8_t bl = unpack6<false>(ql[2 * t], ql[2 * t + 1], hq[2 * t], hq[2 * t + 1], splat(sl),
                                          splat(sl * static_cast<_Float16>(-1024.0f)), magic.lo);
        acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(af[t], bl, acc, 0, 0, 0);
        const _Float16 of = sl * static_cast<_Float16>(32.0f);
        const half8_t bo = {of, of, of, of, of, of, of, of};
        acc_sub = __builtin_amdgcn_mfma_f32_16x16x32_f16(af[t], bo, acc_sub, 0, 0, 0);
    }
#pragma unroll
    for (int t = 0; t < 4; t++) {
        const _Float16 sh = (t >> 1) ? s_h1 : s_h0;
        const half8_t bh = unpack6<true>(ql[2 * t], ql[2 * t + 1], hq[2 * t] >> 4, hq[2 * t + 1] >> 4, splat(sh),
                                         splat(sh * static_cast<_Float16>(-64.0f)), magic.hi);
        acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(af[4 + t], bh, acc, 0, 0, 0);
        const _Float16 of = sh * static_cast<_Float16>(32.0f);
        const half8_t bo = {of, of, of, of, of, of, of, of};
        acc_sub = __builtin_amdgcn_mfma_f32_16x16x32_f16(af[4 + t], bo, acc_sub, 0, 0, 0);
    }
}
__device__ __forceinline__ void compute(const Q6W &r, const half8_t (&af)[8], int lane, uint8_t *area, uint32_t, Q4KMagic magic,
                                        float4_t &acc, float4_t &acc_sub) {
    q6_compute(q6_stage_through_lds(r, lane, area), af, lane, magic, acc, acc_sub);
}

// ---- Q6_K, tiled and field-planar: [tile group of 256 rows][super-block][tile 0..15][3360 bytes], a tile's sixteen
// blocks as four sections - ql [row][128], qh [row][64], scales [row][16], d [row] (f16) - every 16-byte piece aligned.
// The 16-byte pieces of a row's ql (qh) sit at piece index p ^ (row & 7) (p ^ ((row >> 1) & 3)): a layout that a wave
// can also read from LDS without bank conflicts.  Lane (n, g) fetches exactly its operands: four 16-byte loads, one of
// 8 bytes, one of 2, all aligned, a row's ql line shared by the four lanes of the row - no staging, no LDS.
struct Q6T {
    u32x4_t qa, qb, ha, hb;
    uint32_t s0, s1;
    uint32_t d;
};
__device__ __forceinline__ void load_w(Q6T &r, const WholeArgs &a, int tile, int b, int lane) {
    const int n = lane & 15, g = lane >> 4, h = g >> 1, odd = g & 1;
    const uint8_t *p = a.w + ((static_cast<size_t>(tile >> 4) * a.nb + b) * 16 + (tile & 15)) * kQ6TileBytes;
    r.qa = *reinterpret_cast<const u32x4_t *>(p + q6t_ql_piece(n, 4 * h + 2 * odd));
    r.qb = *reinterpret_cast<const u32x4_t *>(p + q6t_ql_piece(n, 4 * h + 2 * odd + 1));
    r.ha = *reinterpret_cast<const u32x4_t *>(p + q6t_qh_piece(n, 2 * h));
    r.hb = *reinterpret_cast<const u32x4_t *>(p + q6t_qh_piece(n, 2 * h + 1));
    const uint2 sc = *reinterpret_cast<const uint2 *>(p + kQ6TSc + n * 16 + 8 * h);
    r.s0 = sc.x;
    r.s1 = sc.y;
    r.d = *reinterpret_cast<const uint16_t *>(p + kQ6TD + n * 2);
}
__device__ __forceinline__ Q6Ops q6_ops(const Q6T &r, int lane) {
    const int odd = (lane >> 4) & 1;
    Q6Ops o;
    o.qa = r.qa;
    o.qb = r.qb;
    o.ha = r.ha;
    o.hb = r.hb;
    o.sc4 = (r.s0 >> (16 * odd)) & 0xffffu;
    o.sc4h = (r.s1 >> (16 * odd)) & 0xffffu;
    o.d = __half2float(__ushort_as_half(static_cast<uint16_t>(r.d)));
    return o;
}
__device__ __forceinline__ void compute(const Q6T &r, const half8_t (&af)[8], int lane, uint8_t *, uint32_t, Q4KMagic magic, float4_t &acc,
                                        float4_t &acc_sub) {
    q6_compute(q6_ops(r, lane), af, lane, magic, acc, acc_sub);
}

struct Q6F {
    half8_t b[8];
    _Float16 o[4];  // 32 s of the four scale pairs: low quarter's two, high quarter's two
};
__device__ __forceinline__ void q6_unpack(const Q6Ops &o, int lane, Q4KMagic magic, Q6F &f) {
    const int odd = (lane >> 4) & 1;
    const int hs = 2 * odd;
    const uint32_t hq[8] = {o.ha.x >> hs, o.ha.y >> hs, o.ha.z >> hs, o.ha.w >> hs, o.hb.x >> hs, o.hb.y >> hs, o.hb.z >> hs, o.hb.w >> hs};
    const uint32_t ql[8] = {o.qa.x, o.qa.y, o.qa.z, o.qa.w, o.qb.x, o.qb.y, o.qb.z, o.qb.w};
    const float d = o.d;
    auto scale = [&](uint32_t pair, int j) { return static_cast<_Float16>(d * static_cast<float>(static_cast<int8_t>(pair >> (8 * j)))); };
    const _Float16 s_l0 = scale(o.sc4, 0), s_l1 = scale(o.sc4, 1), s_h0 = scale(o.sc4h, 0), s_h1 = scale(o.sc4h, 1);
    const _Float16 k32 = static_cast<_Float16>(32.0f);
    f.o[0] = s_l0 * k32;
    f.o[1] = s_l1 * k32;
    f.o[2] = s_h0 * k32;
    f.o[3] = s_h1 * k32;
#pragma unroll
    for (int t = 0; t < 4; t++) {
        const _Float16 sl = (t >> 1) ? s_l1 : s_l0, sh = (t >> 1) ? s_h1 : s_h0;
        f.b[t] = unpack6<false>(ql[2 * t], ql[2 * t + 1], hq[2 * t], hq[2 * t + 1], splat(sl), splat(sl * static_cast<_Float16>(-1024.0f)),
                                magic.lo);
        f.b[4 + t] = unpack6<true>(ql[2 * t], ql[2 * t + 1], hq[2 * t] >> 4, hq[2 * t + 1] >> 4, splat(sh),
                                   splat(sh * static_cast<_Float16>(-64.0f)), magic.hi);
    }
}
__device__ __forceinline__ void unpack(const Q6W &r, int lane, uint8_t *area, uint32_t, Q4KMagic magic, Q6F &f) {
    q6_unpack(q6_stage_through_lds(r, lane, area), lane, magic, f);
}
__device__ __forceinline__ void unpack(const Q6T &r, int lane, uint8_t *, uint32_t, Q4KMagic magic, Q6F &f) {
    q6_unpack(q6_ops(r, lane), lane, magic, f);
}
__device__ __forceinline__ void mma(const Q6F &f, const half8_t (&af)[8], float4_t &acc, float4_t &acc_sub) {
#pragma unroll
    for (int t = 0; t < 8; t++) {
        acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(af[t], f.b[t], acc, 0, 0, 0);
        const _Float16 o = f.o[t >> 1];
        const half8_t bo = {o, o, o, o, o, o, o, o};
        acc_sub = __builtin_amdgcn_mfma_f32_16x16x32_f16(af[t], bo, acc_sub, 0, 0, 0);
    }
}
template <typename W>
struct FragsOf;
template <>
struct FragsOf<Q4W> {
    typedef Q4F type;
};
template <>
struct FragsOf<Q4R> {
    typedef Q4F type;
};
template <>
struct FragsOf<Q4S> {
    typedef Q4SF type;
};
template <>
struct FragsOf<Q6W> {
    typedef Q6F type;
};
template <>
struct FragsOf<Q6T> {
    typedef Q6F type;
};

__device__ __forceinline__ void load_xf(half8_t (&af)[8], const uint8_t *xf, int b, int lane) {
    const half8_t *p = reinterpret_cast<const half8_t *>(xf) + static_cast<size_t>(b) * 512 + lane;
#pragma unroll
    for (int t = 0; t < 8; t++) af[t] = p[t * 64];
}

// Where a wave's activation fragments come from: a buffer in fragment order (XfSrc), or the caller's rows, f32 or f16 in row order
// (RowSrc).  Rows come in row-contiguous loads and go through a wave-private LDS area to the fragments' places, rounded as
// pack_xf_kernel rounds them, so the products have the bits of a pack followed by the fragment-order launch.  (Each lane
// loading its own octets instead touches 64 cache lines a load: 16 f32 rows, 2048 -> 5120, 9.8 us against 5.9.)  Rows the call does
// not have stay what the area held: a row of the product depends on its own activation row only, and they are not stored.
struct XfSrc {};
template <typename XT>
struct RowSrc {};
constexpr int kRowAreaBytes = 16 * DFL_QK_K * 2;  // sixteen rows of a super-block in f16; row m's 16-byte slot o sits at o ^ m
typedef u32x4_t u32x4_row_t __attribute__((aligned(8)));
// kLone: where the one block has fewer than sixteen rows, the lanes of a row that is not there repeat its last one's (their products are not
// stored): a fragment of up to eight rows is then four cache lines, not eight, of which one row asks for a 16-byte piece each.
// One row, 2048 -> 5120 and 4096 -> 2048 in Q6_K: 6.15 -> 5.65 us a launch.  (Leaving those lanes out by the mask: 5.7, and sixteen
// rows 0.1 us slower; the lane worked out ahead of the weights' loads: sixteen rows 0.2 us slower.)
template <typename W, bool kLone>
__device__ __forceinline__ void load_act(XfSrc, half8_t (&af)[8], const WholeArgs &a, const uint8_t *xf, int b, int lane, uint8_t *) {
    load_xf(af, xf, b, kLone ? (lane & 48) | min(lane & 15, a.n_rows - 1) : lane);
}
// One super-block of the rows, row-contiguous: f32 a row a load, f16 two rows a load.
template <typename XT>
struct RowsRaw {
    static constexpr int kLoads = 16 * sizeof(XT) / 4, kRowsPerLoad = 16 / kLoads;
    u32x4_t v[kLoads];
};
template <typename XT>
__device__ __forceinline__ void rows_load(RowsRaw<XT> &r, const XT *xb, size_t stride, int n_rows, int lane) {
#pragma unroll
    for (int i = 0; i < RowsRaw<XT>::kLoads; i++)
        if (i * RowsRaw<XT>::kRowsPerLoad < n_rows) {
            if constexpr (sizeof(XT) == 4)
                r.v[i] = *reinterpret_cast<const u32x4_t *>(xb + i * stride + 4 * lane);
            else
                r.v[i] = *reinterpret_cast<const u32x4_row_t *>(xb + min(2 * i + (lane >> 5), n_rows - 1) * stride + 8 * (lane & 31));
        }
}
// Rows 16 / kParts * part .. as f16 into the area, row m (from the part's first) at 512 m, its 16-byte slot o at o ^ m, a slot's eight values in
// fragment order (0 2 1 3 4 6 5 7).
template <typename XT, int kParts>
__device__ __forceinline__ void rows_to_lds(const RowsRaw<XT> &r, int part, int n_rows, int lane, uint8_t *area) {
    constexpr int kPer = RowsRaw<XT>::kLoads / kParts;
#pragma unroll
    for (int j = 0; j < kPer; j++) {
        const int i = part * kPer + j;
        if (i * RowsRaw<XT>::kRowsPerLoad < n_rows) {
            const u32x4_t v = r.v[i];
            if constexpr (sizeof(XT) == 4) {
                const float4_t f = __builtin_bit_cast(float4_t, v);
                *reinterpret_cast<half4_t *>(area + j * 512 + ((lane >> 1) ^ j) * 16 + (lane & 1) * 8) =
                    half4_t{static_cast<_Float16>(f[0]), static_cast<_Float16>(f[2]), static_cast<_Float16>(f[1]), static_cast<_Float16>(f[3])};
            } else {
                const int m = 2 * j + (lane >> 5), o = lane & 31;
                *reinterpret_cast<u32x4_t *>(area + m * 512 + (o ^ m) * 16) =
                    u32x4_t{__builtin_amdgcn_perm(v.y, v.x, 0x05040100u), __builtin_amdgcn_perm(v.y, v.x, 0x07060302u),
                            __builtin_amdgcn_perm(v.w, v.z, 0x05040100u), __builtin_amdgcn_perm(v.w, v.z, 0x07060302u)};
            }
        }
    }
    __builtin_amdgcn_wave_barrier();
}
template <typename W, bool, typename XT>
__device__ __forceinline__ void load_act(RowSrc<XT>, half8_t (&af)[8], const WholeArgs &a, const uint8_t *x, int b, int lane, uint8_t *area) {
    RowsRaw<XT> raw;
    rows_load(raw, reinterpret_cast<const XT *>(x) + b * DFL_QK_K, static_cast<size_t>(a.nb) * DFL_QK_K, a.n_rows, lane);
    rows_to_lds<XT, 1>(raw, 0, a.n_rows, lane, area);
    constexpr bool q6 = std::is_same<typename FragsOf<W>::type, Q6F>::value;
    const int m = lane & 15, g = lane >> 4;
    // (octets of a lane: common.h, "XF")
#pragma unroll
    for (int t = 0; t < 8; t++) {
        const int o = q6 ? 16 * (g >> 1) + 8 * (t >> 2) + 4 * (g & 1) + (t & 3) : 8 * g + t;
        af[t] = *reinterpret_cast<const half8_t *>(area + m * 512 + (o ^ m) * 16);
    }
    __builtin_amdgcn_wave_barrier();  // (a wave's LDS accesses run in order: what comes next may overwrite the area)
}
template <typename X>
struct AreaBytes {
    static constexpr int value = kQ6AreaBytes;
};
template <typename XT>
struct AreaBytes<RowSrc<XT>> {
    static constexpr int value = kRowAreaBytes;  // (a Q6_K tile's stage passes through it behind the activations)
};
static_assert(kRowAreaBytes >= kQ6AreaBytes, "one area for both");

// W: Q4W or Q6W.  R: tiles per wave and stage (they share the stage's activation fragments).
// kMulti: several 16-row blocks per launch (a.n_blocks): 1 = every wave has one stage (K of at most 16 super-blocks), 2 = one or
// two; the single-block instances (0) keep the registers of a kernel without the loop.  (A prefill takes 1 with R = 1 in the tiled
// orders, whose weights a wave holds; the others serve dflash_gemm_fewrow_xf.)
template <typename W, int R, int kMulti, typename X = XfSrc>
__global__ void __launch_bounds__(1024) gemm_whole_kernel(DFL_WHOLE_PARAMS) {
    const WholeArgs a = DFL_WHOLE_ARGS;
    // [16 waves][R] partial tiles; Q6_K: then a staging area per wave
    extern __shared__ float4_t red[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int tlane = whole_div(wave, by_ksplit), kslice = wave - tlane * a.ksplit;
    const int unit = blockIdx.x * a.tl + tlane;
    const bool active = unit < a.n_units;
    const int n = lane & 15, g = lane >> 4;
    const int b0 = whole_div(a.nb * kslice, by_ksplit), b1 = whole_div(a.nb * (kslice + 1), by_ksplit);  // one or two stages (host)
    const bool two = kMulti != 1 && b1 - b0 > 1;
    const int n_tiles = (a.n_out + 15) >> 4;
    int tile[R];
#pragma unroll
    for (int r = 0; r < R; r++) tile[r] = min(a.pair_off ? unit + r * a.pair_off : unit * R + r, n_tiles - 1);
    float4_t acc[R], acc_sub[R];
    const uint32_t sc_sel = (lane & 16) ? 0x04030402u : 0x04010400u;
    const Q4KMagic magic = q4k_magic();
    uint8_t *area = reinterpret_cast<uint8_t *>(red + 16 * R * 64) + wave * AreaBytes<X>::value;
    // (every load in flight together where the registers hold them; else one tile at a time)
    constexpr bool kEarly = sizeof(W) * R <= 96;
    W w0[kEarly ? R : 1], w1[kEarly ? R : 1];
    if (kEarly && active) {
        // the weights come from HBM, the activations from L2: weights first; they stay in registers for every block
#pragma unroll
        for (int r = 0; r < (kEarly ? R : 1); r++) load_w(w0[r], a, tile[r], b0, lane);
        if (two) {
#pragma unroll
            for (int r = 0; r < (kEarly ? R : 1); r++) load_w(w1[r], a, tile[r], b0 + 1, lane);
        }
    }
    const int n_blocks = kMulti ? a.n_blocks : 1;
    half8_t af[8];
    if (kEarly && active) load_act<W, kMulti == 0>(X(), af, a, a.xf, b0, lane, area);
    // many row blocks, one tile per wave: the B operands are unpacked once and stay in registers in place of the raw weights
    constexpr bool kFrags = kMulti != 0 && kEarly && R == 1;
    typename FragsOf<W>::type f0, f1;
    if (kFrags && active) {
        unpack(w0[0], lane, area, sc_sel, magic, f0);
        if (two) unpack(w1[0], lane, area, sc_sel, magic, f1);
    }
    for (int blk = 0; blk < n_blocks; blk++) {
        const uint8_t *xf = a.xf + static_cast<size_t>(blk) * a.xf_stride;
        const int n_rows = blk + 1 == n_blocks ? a.rows_last : 16;
#pragma unroll
        for (int r = 0; r < R; r++) acc[r] = acc_sub[r] = float4_t{0, 0, 0, 0};
        if (active) {
            if constexpr (kFrags) {
                mma(f0, af, acc[0], acc_sub[0]);
                if (two) {
                    load_act<W, kMulti == 0>(X(), af, a, xf, b0 + 1, lane, area);
                    mma(f1, af, acc[0], acc_sub[0]);
                }
                if (blk + 1 < n_blocks) load_act<W, kMulti == 0>(X(), af, a, xf + a.xf_stride, b0, lane, area);
            } else if constexpr (kEarly) {
                // (af holds this block's first stage: loaded above, or behind the previous block's products)
#pragma unroll
                for (int r = 0; r < R; r++) compute(w0[r], af, lane, area, sc_sel, magic, acc[r], acc_sub[r]);
                if (two) {
                    load_act<W, kMulti == 0>(X(), af, a, xf, b0 + 1, lane, area);
#pragma unroll
                    for (int r = 0; r < R; r++) compute(w1[r], af, lane, area, sc_sel, magic, acc[r], acc_sub[r]);
                }
                // the next block's fragments travel while this block's partial tiles are summed and written
                if (kMulti != 0 && blk + 1 < n_blocks) load_act<W, kMulti == 0>(X(), af, a, xf + a.xf_stride, b0, lane, area);
            } else {
                for (int b = b0; b < b1; b++) {
                    load_act<W, kMulti == 0>(X(), af, a, xf, b, lane, area);
#pragma unroll
                    for (int r = 0; r < R; r++) {
                        W w;
                        load_w(w, a, tile[r], b, lane);
                        compute(w, af, lane, area, sc_sel, magic, acc[r], acc_sub[r]);
                    }
                }
            }
        }
        if (blk) __syncthreads();  // the previous block's partial tiles have been summed
#pragma unroll
        for (int r = 0; r < R; r++) red[(wave * R + r) * 64 + lane] = acc[r] - acc_sub[r];
        __syncthreads();
        if (kslice != 0 || !active) continue;
        float4_t sum[R];
#pragma unroll
        for (int r = 0; r < R; r++) {
            sum[r] = red[(wave * R + r) * 64 + lane];
            for (int s = 1; s < a.ksplit; s++) sum[r] += red[((wave + s) * R + r) * 64 + lane];
        }
        float *y = a.y ? a.y + static_cast<size_t>(blk) * a.y_stride : nullptr;
        if (!a.pair_off) {
#pragma unroll
            for (int r = 0; r < R; r++) {
                const int col = (unit * R + r) * 16 + n;
                if (col < a.n_out) {
#pragma unroll
                    for (int i = 0; i < 4; i++)
                        if (4 * g + i < n_rows) y[static_cast<size_t>(4 * g + i) * a.n_out + col] = sum[r][i];
                }
            }
            continue;
        }
        if constexpr (R == 2) {
            // SwiGLU of the (gate tile, up tile) pair: out[m][16 unit + n] = silu(gate) * up
            const int ffn = a.n_out >> 1;
            float4_t out;
#pragma unroll
            for (int i = 0; i < 4; i++) out[i] = sum[0][i] / (1.0f + expf(-sum[0][i])) * sum[1][i];
            const int col = unit * 16 + n;
            if (y && col < ffn) {
#pragma unroll
                for (int i = 0; i < 4; i++)
                    if (4 * g + i < n_rows) y[static_cast<size_t>(4 * g + i) * ffn + col] = out[i];
            }
            if (a.y_xf) {
                // the tile through this wave's own LDS slot: lane (m, octet) then holds eight consecutive columns of a row
                // (the slot's partial tile has been read: by this wave, above)
                float *f = reinterpret_cast<float *>(&red[wave * R * 64]);
                red[wave * R * 64 + lane] = out;
                __builtin_amdgcn_wave_barrier();
                if (lane < 32) {
                    const int m = lane >> 1, oct = lane & 1;
                    float v[8];
#pragma unroll
                    for (int i = 0; i < 8; i++) v[i] = f[((8 * oct + i) + 16 * (m >> 2)) * 4 + (m & 3)];
                    dfl_xf_store(a.y_xf + static_cast<size_t>(blk) * a.y_xf_stride, a.y_xf_kind, m, unit * 16 + 8 * oct, v[0], v[1], v[2],
                                 v[3], v[4], v[5], v[6], v[7]);
                }
            }
        }
    }
}

// A DFlash-2 sublayer's coefficient projection and its side-0 convolution (kernel size 2) as one launch: dyn[row][side][tap][group] =
// row . W^T as gemm_whole_kernel has it, then y[row][c] = sum_tap (base[0][tap][c] + dyn[row][0][tap][c / group_size]) * x[row - tap][c] as
// dflash2_conv_kernel has it, in fragment order for the projection that reads it.  Workgroup (part, j), j < n_groups / 16: the
// coefficients of groups 16 j .. + 15 for both taps (two tiles, its waves share K), then the convolution of 256 of their channels
// (every part computes the coefficients again: 64 KB of rows and two tiles of weights out of L2).  Behind those, part 0 of j >= n_groups / 16
// stores two tiles of side 1, which the norm that adds the sublayer's result reads (side 0's go nowhere else).
// What bounds it: the product's launch; the convolution's operands arrive under it.  4.8 + 3.4 us as two launches, 6.2 now.
__global__ void __launch_bounds__(1024)
    gemm_conv_kernel(const uint8_t *w, const uint8_t *xf, const float *x, const float *base, int nb, int n_groups, uint32_t by_group, int group_size,
                     int n_rows, int n_waves, float *dyn, uint8_t *y_xf, int y_xf_kind) {
    __shared__ float4_t red[16 * 64];
    __shared__ float coef[2][16][16];  // [tap][row][group]
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n = lane & 15, g = lane >> 4, jj = n_groups >> 4, h = nb * DFL_QK_K;
    const int half = wave >= nb, kslice = half ? wave - nb : wave;
    const bool conv = static_cast<int>(blockIdx.y) < jj;
    if (!conv && blockIdx.x) return;
    const int tile = conv ? half * jj + blockIdx.y : 2 * jj + 2 * (blockIdx.y - jj) + half;
    WholeArgs a = {};
    a.w = w;
    a.nb = nb;
    Q4W wt;
    load_w(wt, a, tile, kslice, lane);
    half8_t af[8];
    load_xf(af, xf, kslice, lane);
    // the convolution's operands of this wave's first row: four channels a lane
    const int c0 = 256 * blockIdx.x + 4 * lane, c = conv ? 16 * group_size * blockIdx.y + c0 : 0, t0 = min(wave, n_rows - 1);
    float4_t b0 = {0, 0, 0, 0}, b1 = b0, x0 = b0, x1 = b0;
    if (conv) {
        b0 = *reinterpret_cast<const float4_t *>(base + c);
        b1 = *reinterpret_cast<const float4_t *>(base + h + c);
        x0 = *reinterpret_cast<const float4_t *>(x + static_cast<size_t>(t0) * h + c);
        x1 = *reinterpret_cast<const float4_t *>(x + static_cast<size_t>(max(t0 - 1, 0)) * h + c);
    }
    dfl_have(dyn, y_xf, y_xf_kind);
    float4_t acc = {0, 0, 0, 0}, acc_sub = {0, 0, 0, 0};
    compute(wt, af, lane, nullptr, (lane & 16) ? 0x04030402u : 0x04010400u, q4k_magic(), acc, acc_sub);
    red[wave * 64 + lane] = acc - acc_sub;
    __syncthreads();
    if (kslice == 0) {
        float4_t sum = red[wave * 64 + lane];
        for (int s = 1; s < nb; s++) sum += red[(wave + s) * 64 + lane];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int row = 4 * g + i;
            if (conv)
                coef[half][row][n] = sum[i];
            else if (row < n_rows)
                dyn[static_cast<size_t>(row) * (4 * n_groups) + tile * 16 + n] = sum[i];
        }
    }
    if (!conv) return;
    __syncthreads();
    const int grp = static_cast<int>(__umulhi(c0, by_group));  // c0 / group_size
    for (int t = wave; t < n_rows; t += n_waves) {
        if (t != wave) {
            x0 = *reinterpret_cast<const float4_t *>(x + static_cast<size_t>(t) * h + c);
            x1 = *reinterpret_cast<const float4_t *>(x + static_cast<size_t>(t - 1) * h + c);
        }
        const float d0 = coef[0][t][grp], d1 = coef[1][t][grp];
        float4_t y;
#pragma unroll
        for (int e = 0; e < 4; e++) {
            y[e] = __builtin_fmaf(b0[e] + d0, x0[e], 0.0f);
            if (t) y[e] = __builtin_fmaf(b1[e] + d1, x1[e], y[e]);
        }
        dfl_xf_store_pair(y_xf, y_xf_kind, t, c & ~7, y[0], y[1], y[2], y[3]);
    }
}

// The same product for a matrix of many more tiles than one round of the chip (an output head: 151936 rows), K of at
// most 16 super-blocks: a workgroup walks units blockIdx.x * tl + tlane, + gridDim.x * tl, ...  A wave's K slice is
// the same super-block in every unit, so its eight activation fragments are loaded ONCE and stay in registers; the
// weights of the next unit travel while the current one is unpacked and multiplied; the slices' partial tiles meet
// in one of two LDS buffers in turn (one barrier per unit: a buffer is rewritten two units later, behind the barrier
// of the unit in between).  Same sums, in the same order, as gemm_whole_kernel with twin products.
template <typename W>
__global__ void __launch_bounds__(1024) gemm_whole_loop_kernel(DFL_WHOLE_PARAMS) {
    const WholeArgs a = DFL_WHOLE_ARGS;
    extern __shared__ float4_t red[];  // [2][16 waves][64]; Q6_K in row order: then a staging area per wave
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int tlane = whole_div(wave, by_ksplit), kslice = wave - tlane * a.ksplit;
    const int n = lane & 15, g = lane >> 4;
    const int b0 = whole_div(a.nb * kslice, by_ksplit);  // one stage per wave (host: nb <= 16, so ksplit == nb and every slice is one super-block)
    const bool has_stage = whole_div(a.nb * (kslice + 1), by_ksplit) > b0;
    const int n_tiles = (a.n_out + 15) >> 4;
    const int stride = a.pair_off * a.tl;
    const uint32_t sc_sel = (lane & 16) ? 0x04030402u : 0x04010400u;
    const Q4KMagic magic = q4k_magic();
    uint8_t *area = reinterpret_cast<uint8_t *>(red + 2 * 16 * 64) + wave * kQ6AreaBytes;
    int unit = static_cast<int>(blockIdx.x) * a.tl + tlane;
    W w_cur, w_next;
    if (unit < n_tiles && has_stage) load_w(w_cur, a, unit, b0, lane);
    half8_t af[8];
    if (has_stage) load_xf(af, a.xf, b0, lane);
    for (int it = 0;; it++) {
        const int next = unit + stride;
        if (next < n_tiles && has_stage) load_w(w_next, a, next, b0, lane);
        float4_t acc = {0, 0, 0, 0}, acc_sub = {0, 0, 0, 0};
        if (unit < n_tiles && has_stage) compute(w_cur, af, lane, area, sc_sel, magic, acc, acc_sub);
        float4_t *buf = red + (it & 1) * (16 * 64);
        buf[wave * 64 + lane] = acc - acc_sub;
        __syncthreads();
        if (kslice == 0 && unit < n_tiles) {
            float4_t sum = buf[wave * 64 + lane];
            for (int s = 1; s < a.ksplit; s++) sum += buf[(wave + s) * 64 + lane];
            const int col = unit * 16 + n;
            if (col < a.n_out) {
#pragma unroll
                for (int i = 0; i < 4; i++)
                    if (4 * g + i < a.n_rows) a.y[static_cast<size_t>(4 * g + i) * a.n_out + col] = sum[i];
            }
        }
        // (the same decision in every wave of the workgroup: its first unit lane's next index)
        if (static_cast<int>(blockIdx.x) * a.tl + (it + 1) * stride >= n_tiles) break;
        unit = next;
        w_cur = w_next;
    }
}

// The looping kernel for the tiled Q6_K order with the weights brought in through LDS instead of registers: a wave
// streams its (tile, super-block) pieces - 3360 contiguous bytes, 210 pieces of 16 - with direct-to-LDS loads into a
// private ring of two buffers and picks its operands out of them with aligned, conflict-free reads (that is what the
// order's piece rotation is for).  No registers are tied up by bytes in flight, so two units travel per wave (the
// register version holds one and already spills); "landed" is an s_waitcnt vmcnt of the younger unit's four loads
// (loads return in order; a Y store of the previous unit that is still in flight only makes the wait stricter).
typedef const __attribute__((address_space(1))) void *gptr_t;
typedef __attribute__((address_space(3))) void *lptr_t;
constexpr int kQ6RingDepth = 2;
constexpr int kVmcnt4 = (4 & 0xF) | 0x0F70, kVmcnt0 = 0x0F70;  // s_waitcnt vmcnt(n), the other counters left alone (gfx9 encoding)
constexpr size_t kQ6LoopLds = static_cast<size_t>(2) * 16 * 64 * sizeof(float4_t) + static_cast<size_t>(16) * kQ6RingDepth * kQ6TileBytes;
__global__ void __launch_bounds__(1024) gemm_q6t_loop_kernel(DFL_WHOLE_PARAMS) {
    const WholeArgs a = DFL_WHOLE_ARGS;
    extern __shared__ float4_t red[];  // [2][16 waves][64], then the rings [16 waves][kQ6RingDepth][3360 bytes]
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int tlane = whole_div(wave, by_ksplit), kslice = wave - tlane * a.ksplit;
    const int n = lane & 15, g = lane >> 4, h = g >> 1, odd = g & 1;
    const int b0 = kslice;  // (host: nb <= 16, so ksplit == nb and every slice is one super-block)
    const int n_tiles = (a.n_out + 15) >> 4;
    const int stride = a.pair_off * a.tl;
    const Q4KMagic magic = q4k_magic();
    uint8_t *ring = reinterpret_cast<uint8_t *>(red + 2 * 16 * 64) + static_cast<size_t>(wave) * (kQ6RingDepth * kQ6TileBytes);
    auto issue = [&](int unit, int slot) {  // the unit's 210 pieces into ring buffer `slot`
        const uint8_t *src = a.w + ((static_cast<size_t>(unit >> 4) * a.nb + b0) * 16 + (unit & 15)) * kQ6TileBytes + lane * 16;
        uint8_t *dst = ring + slot * kQ6TileBytes;
        __builtin_amdgcn_global_load_lds((gptr_t)(src), (lptr_t)(dst), 16, 0, 0);
        __builtin_amdgcn_global_load_lds((gptr_t)(src + 1024), (lptr_t)(dst + 1024), 16, 0, 0);
        __builtin_amdgcn_global_load_lds((gptr_t)(src + 2048), (lptr_t)(dst + 2048), 16, 0, 0);
        // (the fourth load carries the last 18 pieces: a lane's 16 bytes land at the buffer address + 16 lane whatever it
        // reads, so the other lanes stay out of it; the wave still issues four loads, which is what the count below needs)
        if (lane < 18) __builtin_amdgcn_global_load_lds((gptr_t)(src + 3072), (lptr_t)(dst + 3072), 16, 0, 0);
    };
    int unit = static_cast<int>(blockIdx.x) * a.tl + tlane;
    half8_t af[8];
    load_xf(af, a.xf, b0, lane);
    __builtin_amdgcn_s_waitcnt(kVmcnt0);  // (the fragments are in registers: from here on only weight loads and Y stores are counted)
    if (unit < n_tiles) issue(unit, 0);
    for (int it = 0;; it++) {
        const int next = unit + stride;
        const int slot = it & 1;
        if (next < n_tiles) issue(next, slot ^ 1);  // (that buffer's unit was consumed one iteration ago: its reads are complete)
        float4_t acc = {0, 0, 0, 0}, acc_sub = {0, 0, 0, 0};
        if (unit < n_tiles) {
            if (next < n_tiles)
                __builtin_amdgcn_s_waitcnt(kVmcnt4);
            else
                __builtin_amdgcn_s_waitcnt(kVmcnt0);
            const uint8_t *t = ring + slot * kQ6TileBytes;
            Q6Ops o;
            o.qa = *reinterpret_cast<const u32x4_t *>(t + q6t_ql_piece(n, 4 * h + 2 * odd));
            o.qb = *reinterpret_cast<const u32x4_t *>(t + q6t_ql_piece(n, 4 * h + 2 * odd + 1));
            o.ha = *reinterpret_cast<const u32x4_t *>(t + q6t_qh_piece(n, 2 * h));
            o.hb = *reinterpret_cast<const u32x4_t *>(t + q6t_qh_piece(n, 2 * h + 1));
            const uint2 sc = *reinterpret_cast<const uint2 *>(t + kQ6TSc + n * 16 + 8 * h);
            o.sc4 = (sc.x >> (16 * odd)) & 0xffffu;
            o.sc4h = (sc.y >> (16 * odd)) & 0xffffu;
            o.d = __half2float(__ushort_as_half(*reinterpret_cast<const uint16_t *>(t + kQ6TD + n * 2)));
            q6_compute(o, af, lane, magic, acc, acc_sub);
        }
        float4_t *buf = red + slot * (16 * 64);
        buf[wave * 64 + lane] = acc - acc_sub;
        __syncthreads();
        if (kslice == 0 && unit < n_tiles) {
            float4_t sum = buf[wave * 64 + lane];
            for (int s = 1; s < a.ksplit; s++) sum += buf[(wave + s) * 64 + lane];
            const int col = unit * 16 + n;
            if (col < a.n_out) {
#pragma unroll
                for (int i = 0; i < 4; i++)
                    if (4 * g + i < a.n_rows) a.y[static_cast<size_t>(4 * g + i) * a.n_out + col] = sum[i];
            }
        }
        if (static_cast<int>(blockIdx.x) * a.tl + (it + 1) * stride >= n_tiles) break;
        unit = next;
    }
}

// The public operator on a Q4_K matrix of many rounds of tiles, K of at most 24 super-blocks, rows in row order: one workgroup per
// CU walks units of one tile, its waves share K.  A wave keeps the fragments and the sub-block sums of its one or two
// super-blocks in registers for every tile, so a tile costs it nothing but weights, which it streams through a private
// ring of LDS slots (a slot: one super-block of the tile, 144 pieces of 16 bytes, three direct-to-LDS loads); the slices' partial tiles
// meet in one of two LDS buffers in turn, one barrier per tile, a different wave adding each time.  No partial tiles in memory, no second launch.
// What bounds it: the stream of the weights (46 KB a tile of K = 5120 at 5.3 - 5.6 TB/s over the chip) behind a start of 4 us, in which every
// CU takes in all of the rows; where the tiles are a few rounds, the last one, for which only some CUs have a tile.
// us a call, weights cold, streaming kernel and reduction : this one, 1 row f32 / 16 rows f16 / 16 rows f32:
//   tiled Q4_K  5120 -> 17408 17.9 :17.0 20.2 :17.2 20.5 :19.4   2560 -> 16384 12.2 : 9.2 13.3 :10.2 13.4 :10.8   2048 -> 40000 17.0 :13.0 20.3 :14.4 20.3 :15.9
//   row order   5120 -> 17408 18.1 :17.7 19.8 :18.2 19.9 :20.3   2560 -> 16384 12.6 : 9.4 14.4 :10.1 14.4 :11.3   2048 -> 40000 17.0 :13.5 19.2 :15.1 19.2 :16.6
// Sixteen f32 rows are twice the bytes to bring in ahead of the first product, and against weights in row order, two super-blocks a wave,
// that is all that the launch saves, or 2 % more; the line looks at the matrix alone, so that a row has its bits whatever its type and company.
// (no stage ahead of the rows, or four: 18.3 and 18.5 for 16 f16 rows, 5120 -> 17408).
// A stage has landed when no more loads are under way than were issued behind it: they return in order, and a Y store among them only makes it stricter.
constexpr int kWideSlot = 16 * DFL_Q4_K_BYTES;  // 2304 bytes
constexpr int kWideSlots = 6;                        // at most (the counts below)
__device__ __forceinline__ void wide_wait(int ahead) {  // at most `ahead` stages (three loads each) still under way, ahead uniform
    if (ahead <= 0)
        __builtin_amdgcn_s_waitcnt(kVmcnt0);
    else if (ahead == 1)
        __builtin_amdgcn_s_waitcnt(0x0F70 | 3);
    else if (ahead == 2)
        __builtin_amdgcn_s_waitcnt(0x0F70 | 6);
    else if (ahead == 3)
        __builtin_amdgcn_s_waitcnt(0x0F70 | 9);
    else if (ahead == 4)
        __builtin_amdgcn_s_waitcnt(0x0F70 | 12);
    else
        __builtin_amdgcn_s_waitcnt(0x0F70 | 15);
}
// The fragments of one super-block out of its rows: in one go through 8 KB of LDS, or eight rows at a time through 4 KB.
template <typename XT, int kParts>
__device__ __forceinline__ void wide_fragments(half8_t (&af)[8], const RowsRaw<XT> &raw, int n_rows, int lane, uint8_t *area) {
    const int g = lane >> 4;
#pragma unroll
    for (int part = 0; part < kParts; part++) {
        rows_to_lds<XT, kParts>(raw, part, n_rows, lane, area);
        const int m = lane & (16 / kParts - 1);
        half8_t v[8];
#pragma unroll
        for (int t = 0; t < 8; t++) v[t] = *reinterpret_cast<const half8_t *>(area + m * 512 + ((8 * g + t) ^ m) * 16);
#pragma unroll
        for (int t = 0; t < 8; t++) {
            asm volatile("" : "+v"(v[t]));  // (read by every lane: a select, not a branch around each read)
            af[t] = kParts == 1 || ((lane & 15) >> 3) == part ? v[t] : af[t];
        }
        __builtin_amdgcn_wave_barrier();
    }
}
// kLen: super-blocks a wave has at most (two: at most twelve waves, whose registers hold both).
template <typename XT, bool kTiled, int kLen, int kSlots>
__global__ void __launch_bounds__(kLen == 2 ? 768 : 1024) gemm_q4k_wide_kernel(DFL_WHOLE_PARAMS) {
    const WholeArgs a = DFL_WHOLE_ARGS;
    extern __shared__ float4_t red[];  // [2][waves][64], then the rings [wave][kSlots][kWideSlot]
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), waves = a.ksplit * a.tl;
    const int tlane = whole_div(wave, by_ksplit), kslice = wave - tlane * a.ksplit;
    const int n = lane & 15, g = lane >> 4;
    const int b0 = whole_div(a.nb * kslice, by_ksplit), len = whole_div(a.nb * (kslice + 1), by_ksplit) - b0;  // one or two super-blocks (host)
    const int n_tiles = (a.n_out + 15) >> 4, stride = a.pair_off * a.tl;
    const int first = static_cast<int>(blockIdx.x) * a.tl, unit0 = first + tlane;
    const int units = unit0 < n_tiles ? (n_tiles - 1 - unit0) / stride + 1 : 0;  // of this wave
    const int rounds = (n_tiles - 1 - first) / stride + 1;                       // of the workgroup (its first tile lane has the most)
    const int n_stages = units * len;
    uint8_t *ring = reinterpret_cast<uint8_t *>(red + 2 * waves * 64) + static_cast<size_t>(wave) * (kSlots * kWideSlot);
    // the next stage to issue: super-block b0 + i_b of tile i_tile, into slot i_slot
    int issued = 0, i_b = 0, i_tile = unit0, i_slot = 0;
    int r0 = 0, r1 = 0, r2 = 0, p0 = 0, p1 = 0, p2 = 0;  // row order: the lane's three pieces of a stage, rows and bytes in them
    if constexpr (!kTiled) {
        r0 = lane / 9, p0 = 16 * (lane - 9 * r0);
        r1 = (lane + 64) / 9, p1 = 16 * (lane + 64 - 9 * r1);
        r2 = (lane + 128) / 9, p2 = 16 * (lane + 128 - 9 * r2);  // (lanes past 15 issue nothing)
    }
    auto issue = [&]() {
        uint8_t *dst = ring + i_slot * kWideSlot;
        const int tile = min(i_tile, n_tiles - 1);  // (past the last: one of the first stages, which go out whatever there is; not read)
        if constexpr (kTiled) {
            const uint8_t *src = a.w + ((static_cast<size_t>(tile >> 4) * a.nb + b0 + i_b) * 16 + (tile & 15)) * kWideSlot + lane * 16;
            __builtin_amdgcn_global_load_lds((gptr_t)(src), (lptr_t)(dst), 16, 0, 0);
            __builtin_amdgcn_global_load_lds((gptr_t)(src + 1024), (lptr_t)(dst + 1024), 16, 0, 0);
            if (lane < 16) __builtin_amdgcn_global_load_lds((gptr_t)(src + 2048), (lptr_t)(dst + 2048), 16, 0, 0);
        } else {
            // (rows past the matrix re-read its last row; never stored)
            const uint8_t *src = a.w + static_cast<size_t>(b0 + i_b) * DFL_Q4_K_BYTES;
            const int t = tile * 16, last = a.n_out - 1;
            __builtin_amdgcn_global_load_lds((gptr_t)(src + static_cast<size_t>(min(t + r0, last)) * a.row_bytes + p0), (lptr_t)(dst), 16, 0, 0);
            __builtin_amdgcn_global_load_lds((gptr_t)(src + static_cast<size_t>(min(t + r1, last)) * a.row_bytes + p1), (lptr_t)(dst + 1024), 16, 0, 0);
            if (lane < 16)
                __builtin_amdgcn_global_load_lds((gptr_t)(src + static_cast<size_t>(min(t + r2, last)) * a.row_bytes + p2), (lptr_t)(dst + 2048), 16, 0, 0);
        }
        issued++;
        if (++i_slot == kSlots) i_slot = 0;
        if (++i_b == len) {
            i_b = 0;
            i_tile += stride;
        }
    };
    // The rows first (they come from L2), behind them the first stages, as many as leave the rows' way through LDS alone; the others
    // once the fragments stand.
    constexpr int kAreaSlots = kLen == 2 ? 4 : 2;  // 8 KB, or 4 KB where there are three slots to a wave
    half8_t af0[8] = {}, af1[kLen == 2 ? 8 : 1] = {}, am0, am1;
    {
        uint8_t *area = ring + (kSlots - kAreaSlots) * kWideSlot;
        static_assert(kAreaSlots * kWideSlot >= 16 * 512 / (kLen == 2 ? 1 : 2), "the rows' area");
        const XT *xb = reinterpret_cast<const XT *>(a.xf) + static_cast<size_t>(b0) * DFL_QK_K;
        const size_t xs = static_cast<size_t>(a.nb) * DFL_QK_K;
        RowsRaw<XT> raw0, raw1;
        rows_load(raw0, xb, xs, a.n_rows, lane);
        if constexpr (kLen == 2)
            if (len > 1) rows_load(raw1, xb + DFL_QK_K, xs, a.n_rows, lane);
        // (a fixed number of stages without a branch: the compiler then waits for the rows alone, not for what is behind them)
        issue();
        if constexpr (kSlots - kAreaSlots > 1) issue();
        wide_fragments<XT, kLen == 2 ? 1 : 2>(af0, raw0, a.n_rows, lane, area);
        if constexpr (kLen == 2) {
            if (len > 1) {
                wide_fragments<XT, 1>(af1, raw1, a.n_rows, lane, area);
            }
            am1 = sum_operand(af1);
        }
        am0 = sum_operand(af0);
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // (the area's last reads are done: its slots may be loaded into)
    while (issued < n_stages && issued < kSlots) issue();

    const uint32_t sc_sel = (lane & 16) ? 0x04030402u : 0x04010400u;
    const Q4KMagic magic = q4k_magic();
    int done = 0, slot = 0;
    float4_t acc;
    auto stage = [&](const half8_t (&af)[8], const half8_t &am) {
        wide_wait(issued - done - 1);
        const u32x4_t *p = reinterpret_cast<const u32x4_t *>(ring + slot * kWideSlot) + n * 9;
        Q4S w;
        w.hdr = p[0];
        w.q0 = p[1 + 2 * g];
        w.q1 = p[2 + 2 * g];
        Q4SF f;
        unpack(w, lane, nullptr, sc_sel, magic, f);
        const half2_t mn = {-f.m_lo, -f.m_hi};
        acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(am, q4k_min_operand(mn), acc, 0, 0, 0);
#pragma unroll
        for (int t = 0; t < 8; t++) acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(af[t], f.b[t], acc, 0, 0, 0);
        done++;
        if (++slot == kSlots) slot = 0;
        if (issued < n_stages) issue();  // (into the slot just read: its operands are in registers)
    };
    for (int it = 0; it < rounds; it++) {
        const int unit = unit0 + it * stride;
        acc = float4_t{0, 0, 0, 0};
        if (it < units) {
            stage(af0, am0);
            if constexpr (kLen == 2)
                if (len > 1) stage(af1, am1);
        }
        float4_t *buf = red + (it & 1) * (waves * 64);
        buf[wave * 64 + lane] = acc;
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        // the slices take turns at the sum (a buffer is rewritten two rounds later, behind the barrier of the round between)
        if (kslice == it % a.ksplit && it < units) {
            const float4_t *part = buf + tlane * a.ksplit * 64 + lane;
            float4_t sum = part[0];
            for (int s = 1; s < a.ksplit; s++) sum += part[s * 64];
            const int col = unit * 16 + n;
            if (col < a.n_out) {
#pragma unroll
                for (int i = 0; i < 4; i++)
                    if (4 * g + i < a.n_rows) a.y[static_cast<size_t>(4 * g + i) * a.n_out + col] = sum[i];
            }
        }
    }
    if (issued > n_stages) __builtin_amdgcn_s_waitcnt(kVmcnt0);  // (nothing is under way into LDS when the wave ends)
}

// Row-major activations -> XF: one thread per (row, eight consecutive values).
template <typename XT>
__global__ void __launch_bounds__(256) pack_xf_kernel(const XT *__restrict__ x, int n_rows, int n_in, int kind, uint8_t *__restrict__ xf) {
    const int oct = blockIdx.x * 256 + threadIdx.x, m = blockIdx.y;
    if (8 * oct >= n_in || m >= n_rows) return;
    const XT *p = x + static_cast<size_t>(m) * n_in + 8 * oct;
    dfl_xf_store(xf, kind, m, 8 * oct, static_cast<float>(p[0]), static_cast<float>(p[1]), static_cast<float>(p[2]), static_cast<float>(p[3]),
                 static_cast<float>(p[4]), static_cast<float>(p[5]), static_cast<float>(p[6]), static_cast<float>(p[7]));
}

struct EnvInt {
    const char *name;
    bool set;
    int value;
    explicit EnvInt(const char *n) : name(n), set(false), value(0) {
        if (const char *e = getenv(n)) {
            set = true;
            value = atoi(e);
        }
    }
    int get(int fallback) const { return set ? value : fallback; }
};
#define env_int(name, fallback) ([]() -> const EnvInt & { static const EnvInt e(name); return e; }().get(fallback))

struct WholePlan {
    int kind, ksplit, tl, R, n_units, n_wg;
    bool loop;  // more units than one round: gemm_whole_loop_kernel (one stage per wave, plain product)
};

// The split of a matrix over waves, or kind == DFL_XF_NONE where this path does not take it.
WholePlan whole_plan(const dflash_ctx *ctx, int32_t w_type, int64_t n_in, int64_t n_out, int64_t pair_ffn) {
    WholePlan p = {DFL_XF_NONE, 0, 0, 0, 0, 0, false};
    if (!env_int("DFLASH_GEMM_WHOLE", 1)) return p;
    const int kind = w_type == DFLASH_TYPE_Q4_K_TILED ? DFL_XF_Q4K
                     : (w_type == DFLASH_TYPE_Q6_K || w_type == DFLASH_TYPE_Q6_K_TILED) ? DFL_XF_Q6K
                                                                                       : DFL_XF_NONE;
    if (kind == DFL_XF_NONE || n_in <= 0 || n_in % DFL_QK_K || n_out <= 0 || n_out >= (1 << 24)) return p;
    const int nb = static_cast<int>(n_in / DFL_QK_K);
    if (nb > 32) return p;  // more than two stages per wave
    if (pair_ffn && (n_out != 2 * pair_ffn || pair_ffn % 16)) return p;
    const int ksplit = nb < 16 ? nb : 16, tl = 16 / ksplit;
    const int tiles = static_cast<int>((n_out + 15) / 16);
    int R = pair_ffn ? 2 : 1;
    int n_units = pair_ffn ? static_cast<int>(pair_ffn / 16) : tiles;
    // one round of the chip: at most one workgroup per CU (a wave's registers leave room for one)
    // (a quarter of a round more, 320 workgroups on 256 CUs, measured slower than two tiles per wave on 160: 10.1 -> 8.6 us
    // for 4096 -> 5120 Q4_K, 14.9 -> 14.0 us for 5120 -> 5120 Q6_K; DFLASH_WHOLE_TOL_PCT=25 for the former rule)
    static const int env_tol = env_int("DFLASH_WHOLE_TOL_PCT", 0);
    const int max_wg = ctx->n_cu + ctx->n_cu * env_tol / 100;
    if (!pair_ffn && (n_units + tl - 1) / tl > max_wg) {
        R = 2;
        n_units = (tiles + 1) / 2;
    }
    const int n_wg = (n_units + tl - 1) / tl;
    if (n_wg > max_wg) {
        // many rounds: the looping kernel, where every wave keeps one super-block of the activations (K <= 16 super-blocks)
        if (pair_ffn || nb > 16 || !env_int("DFLASH_GEMM_WHOLE_LOOP", 1)) return p;
        p = {kind, ksplit, tl, 1, tiles, std::min((tiles + tl - 1) / tl, ctx->n_cu), true};
        return p;
    }
    p = {kind, ksplit, tl, R, n_units, n_wg, false};
    return p;
}

}  // namespace

int dfl_whole_kind(const dflash_ctx *ctx, int32_t w_type, int64_t n_in, int64_t n_out, int64_t pair_ffn) {
    return whole_plan(ctx, w_type, n_in, n_out, pair_ffn).kind;
}

bool dfl_whole_by_sums(const dflash_ctx *ctx, int32_t w_type, int64_t n_in, int64_t n_out, int64_t pair_ffn) {
    if (w_type != DFLASH_TYPE_Q4_K_TILED || n_in < 16 * DFL_QK_K) return false;
    const WholePlan p = whole_plan(ctx, w_type, n_in, n_out, pair_ffn);
    return p.kind != DFL_XF_NONE && !p.loop;
}

bool dfl_whole_holds_weights(const dflash_ctx *ctx, int32_t w_type, int64_t n_in, int64_t n_out) {
    const WholePlan p = whole_plan(ctx, w_type, n_in, n_out, 0);
    return p.kind != DFL_XF_NONE && !p.loop && p.R == 1 && n_in / DFL_QK_K <= p.ksplit;
}

int32_t dfl_gemm_whole(dflash_ctx *ctx, int32_t w_type, const void *w, const void *xf, float *y, int64_t n_in, int64_t n_out,
                       int32_t n_rows, int64_t pair_ffn, void *y_xf, int y_xf_kind, hipStream_t st, bool by_sums) {
    return dfl_gemm_whole_blocks(ctx, w_type, w, xf, y, n_in, n_out, n_rows, pair_ffn, y_xf, y_xf_kind, st, by_sums);
}

int32_t dfl_gemm_whole_blocks(dflash_ctx *ctx, int32_t w_type, const void *w, const void *xf, float *y, int64_t n_in, int64_t n_out,
                              int32_t n_rows_total, int64_t pair_ffn, void *y_xf, int y_xf_kind, hipStream_t st, bool by_sums) {
    const int32_t n_blocks = (n_rows_total + 15) / 16;
    const int32_t n_rows = n_rows_total - 16 * (n_blocks - 1);  // rows of the last block
    if (n_rows_total < 1 || n_blocks > 4096) return dfl_fail(ctx, DFLASH_ERR_BAD_SHAPE, "gemm_whole: %d rows", n_rows_total);
    const WholePlan p = whole_plan(ctx, w_type, n_in, n_out, pair_ffn);
    if (p.kind == DFL_XF_NONE) return dfl_fail(ctx, DFLASH_ERR_UNSUPPORTED, "gemm_whole: type %d, %lld -> %lld not taken", w_type,
                                               static_cast<long long>(n_in), static_cast<long long>(n_out));
    if (!w || !xf || n_rows < 1 || n_rows > 16 || (!y && !(pair_ffn && y_xf)))
        return dfl_fail(ctx, DFLASH_ERR_BAD_SHAPE, "gemm_whole: null operand or n_rows %d", n_rows);
    const bool q6_tiled = w_type == DFLASH_TYPE_Q6_K_TILED;
    if (reinterpret_cast<uintptr_t>(xf) % 16 || reinterpret_cast<uintptr_t>(w) % ((p.kind == DFL_XF_Q4K || q6_tiled) ? 16 : 2) ||
        (y_xf && reinterpret_cast<uintptr_t>(y_xf) % 16))
        return dfl_fail(ctx, DFLASH_ERR_ALIGNMENT, "gemm_whole: operand alignment");
    if (y_xf && (!pair_ffn || (y_xf_kind != DFL_XF_Q4K && y_xf_kind != DFL_XF_Q6K)))
        return dfl_fail(ctx, DFLASH_ERR_UNSUPPORTED, "gemm_whole: fragment-order output needs the SwiGLU pair mode and a kind");
    WholeArgs a;
    a.w = static_cast<const uint8_t *>(w);
    a.xf = static_cast<const uint8_t *>(xf);
    a.y = y;
    a.y_xf = static_cast<uint8_t *>(y_xf);
    a.y_xf_kind = y_xf_kind;
    a.n_out = static_cast<int>(n_out);
    a.nb = static_cast<int>(n_in / DFL_QK_K);
    a.n_rows = n_rows;
    a.ksplit = p.ksplit;
    a.tl = p.tl;
    a.n_units = p.n_units;
    a.pair_off = pair_ffn ? static_cast<int>(pair_ffn / 16) : 0;
    a.row_bytes = static_cast<uint32_t>(a.nb) * DFL_Q6_K_BYTES;
    a.n_blocks = n_blocks;
    a.rows_last = n_rows;
    a.xf_stride = static_cast<uint32_t>(dfl_xf_bytes(n_in));
    a.y_xf_stride = static_cast<uint32_t>(dfl_xf_bytes(pair_ffn ? pair_ffn : 256));
    a.y_stride = static_cast<size_t>(16) * (pair_ffn ? pair_ffn : n_out);
    const int threads = 64 * p.ksplit * p.tl;
    const size_t red_bytes = static_cast<size_t>(16) * p.R * 64 * sizeof(float4_t);
    const size_t lds = red_bytes + ((p.kind == DFL_XF_Q6K && !q6_tiled) ? static_cast<size_t>(16) * kQ6AreaBytes : 0);
    if (p.loop) {
        if (n_blocks > 1) return dfl_fail(ctx, DFLASH_ERR_UNSUPPORTED, "gemm_whole: a matrix of %d tiles takes one block of rows per call", p.n_units);
        const bool q6_ring = q6_tiled && kQ6LoopLds <= ctx->lds_bytes && env_int("DFLASH_Q6T_RING", 1);
        const whole_kernel_t lf = p.kind == DFL_XF_Q4K ? gemm_whole_loop_kernel<Q4W>
                            : q6_ring            ? gemm_q6t_loop_kernel
                            : q6_tiled           ? gemm_whole_loop_kernel<Q6T>
                                                 : gemm_whole_loop_kernel<Q6W>;
        const size_t llds = q6_ring ? kQ6LoopLds
                                    : static_cast<size_t>(2) * 16 * 64 * sizeof(float4_t) +
                                          ((p.kind == DFL_XF_Q6K && !q6_tiled) ? static_cast<size_t>(16) * kQ6AreaBytes : 0);
        if (llds > ctx->lds_bytes) return dfl_fail(ctx, DFLASH_ERR_UNSUPPORTED, "gemm_whole: %zu bytes of LDS needed", llds);
        if (llds > 48 * 1024)
            if (const int32_t rc = dfl_raise_lds_limit(ctx, reinterpret_cast<const void *>(lf), llds)) return rc;
        dfl_timed timer(ctx, st, DFL_T_GEMM);
        a.pair_off = p.n_wg;
        whole_launch(lf, p.n_wg, 64 * p.ksplit * p.tl, llds, st, a);
        DFL_HIP_CHECK(ctx, hipGetLastError());
        return DFLASH_OK;
    }
    by_sums = by_sums && dfl_whole_by_sums(ctx, w_type, n_in, n_out, pair_ffn);
    const int multi = n_blocks > 1 ? (a.nb > p.ksplit ? 2 : 1) : 0;
    if (multi && by_sums && (p.R != 1 || multi != 1))
        return dfl_fail(ctx, DFLASH_ERR_UNSUPPORTED, "gemm_whole: several blocks by sums only past weights a wave holds");
#define DFL_WHOLE_PICK(WT, RR) (multi == 0 ? gemm_whole_kernel<WT, RR, 0> : multi == 1 ? gemm_whole_kernel<WT, RR, 1> : gemm_whole_kernel<WT, RR, 2>)
    const whole_kernel_t fn = p.kind == DFL_XF_Q4K && by_sums ? (p.R == 2 ? gemm_whole_kernel<Q4S, 2, 0> : multi ? gemm_whole_kernel<Q4S, 1, 1> : gemm_whole_kernel<Q4S, 1, 0>)
                        : p.kind == DFL_XF_Q4K          ? (p.R == 2 ? DFL_WHOLE_PICK(Q4W, 2) : DFL_WHOLE_PICK(Q4W, 1))
                        : q6_tiled           ? (p.R == 2 ? DFL_WHOLE_PICK(Q6T, 2) : DFL_WHOLE_PICK(Q6T, 1))
                                             : (p.R == 2 ? DFL_WHOLE_PICK(Q6W, 2) : DFL_WHOLE_PICK(Q6W, 1));
#undef DFL_WHOLE_PICK
    if (lds > ctx->lds_bytes) return dfl_fail(ctx, DFLASH_ERR_UNSUPPORTED, "gemm_whole: %zu bytes of LDS needed", lds);
    if (lds > 48 * 1024)
        if (const int32_t rc = dfl_raise_lds_limit(ctx, reinterpret_cast<const void *>(fn), lds)) return rc;
    dfl_timed timer(ctx, st, DFL_T_GEMM);
    whole_launch(fn, p.n_wg, threads, lds, st, a);
    DFL_HIP_CHECK(ctx, hipGetLastError());
    return DFLASH_OK;
}

bool dfl_gemm_conv_takes(const dflash_ctx *ctx, int32_t w_type, int64_t h, int32_t kernel_size, int32_t group_size, int32_t y_xf_kind) {
    if (w_type != DFLASH_TYPE_Q4_K_TILED || y_xf_kind == DFL_XF_NONE || kernel_size != 2 || h < 256 || h % 256 || h > 8 * DFL_QK_K) return false;
    if (group_size < 16 || group_size % 16 || h % group_size || (h / group_size) % 16) return false;
    return whole_plan(ctx, w_type, h, 4 * (h / group_size), 0).kind == DFL_XF_Q4K;
}

int32_t dfl_gemm_conv(dflash_ctx *ctx, const void *w, const void *xf, const float *x, const float *base, int64_t h, int32_t group_size, int32_t n_rows,
                      float *dyn, void *y_xf, int y_xf_kind, hipStream_t st) {
    if (!dfl_gemm_conv_takes(ctx, DFLASH_TYPE_Q4_K_TILED, h, 2, group_size, y_xf_kind) || n_rows < 1 || n_rows > 16)
        return dfl_fail(ctx, DFLASH_ERR_UNSUPPORTED, "gemm_conv: %lld channels in groups of %d, %d rows", static_cast<long long>(h), group_size, n_rows);
    if (!w || !xf || !x || !base || !dyn || !y_xf) return dfl_fail(ctx, DFLASH_ERR_INVALID_INPUT, "gemm_conv: null pointer");
    for (const void *p : {w, xf, static_cast<const void *>(x), static_cast<const void *>(base), static_cast<const void *>(y_xf)})
        if (reinterpret_cast<uintptr_t>(p) % 16) return dfl_fail(ctx, DFLASH_ERR_ALIGNMENT, "gemm_conv: operand alignment");
    if (dfl_ranges_overlap(xf, dfl_xf_bytes(h), y_xf, dfl_xf_bytes(h))) return dfl_fail(ctx, DFLASH_ERR_ALIAS, "gemm_conv: the result overlaps the rows");
    const int nb = static_cast<int>(h / DFL_QK_K), groups = static_cast<int>(h / group_size);
    const uint32_t by_group = static_cast<uint32_t>(((1ull << 32) + group_size - 1) / group_size);  // (exact for channels below 16 group_size <= h <= 2048)
    dfl_timed timer(ctx, st, DFL_T_GEMM);
    gemm_conv_kernel<<<dim3(16 * group_size / 256, 2 * (groups / 16)), 128 * nb, 0, st>>>(
        static_cast<const uint8_t *>(w), static_cast<const uint8_t *>(xf), x, base, nb, groups, by_group, group_size, n_rows, 2 * nb, dyn,
        static_cast<uint8_t *>(y_xf), y_xf_kind);
    DFL_HIP_CHECK(ctx, hipGetLastError());
    return DFLASH_OK;
}

// ---- the public operator on rows in row order ----
namespace {
// One launch in place of the streaming kernel and its reduction, where the tiles are one round of the chip, in the smallest
// workgroups that hold them so.  The line depends on the matrix alone, not on its order, the rows or their type, so neither do the
// bits.  us of the GPU per call, streaming : direct, 1 row f32 / 16 rows f16 / 16 rows f32:
//   one tile per wave   Q6_K 2048 -> 512   7.3 : 4.2   7.9 : 4.9   7.9 : 5.4    tiled Q4_K 4096 -> 4096  8.4 : 4.4   9.7 : 5.5   9.7 : 6.1
//                       Q6_K 6144 -> 2048 10.0 : 8.1  11.1 :10.3  11.1 :11.1    Q4_K in row order 6144 -> 2048  8.9 : 6.5  10.0 : 8.2   9.9 : 9.2
//     beyond 24 super-blocks  Q6_K 8192 -> 1024   9.9 : 8.8  10.7 :11.0  10.8 :12.4 (two stages a wave, each with its rows to bring in)
//     beyond 22, few tiles, us a call  Q6_K 6144 -> 512  9.0 : 7.9   9.1 :10.0   9.0 :11.2   -> 1024  9.1 : 8.1   9.2 :10.1   9.0 :11.3
//                                      from half a round of tiles on a single row gains what sixteen lose:  -> 2048  9.4 : 8.3  10.2 :11.2  10.3 :11.5
//   two tiles per wave  tiled Q4_K 4096 -> 5120  8.9 : 5.8  10.1 : 7.1  10.2 : 7.7    in row order  9.1 : 6.6  10.8 : 8.0  10.8 : 8.9
//     beyond 16 super-blocks  5120 -> 5120  8.7 : 8.3  10.1 :10.2  10.2 :10.7    Q6_K, 4096 -> 5120  11.5 :13.4 (its registers spill)
WholePlan rows_direct_plan(const dflash_ctx *ctx, int32_t w_type, int64_t n_in, int64_t n_out) {
    WholePlan p = {DFL_XF_NONE, 0, 0, 0, 0, 0, false};
    if (!env_int("DFLASH_GEMM_WHOLE", 1)) return p;
    const int kind = w_type == DFLASH_TYPE_Q6_K ? DFL_XF_Q6K : (w_type == DFLASH_TYPE_Q4_K || w_type == DFLASH_TYPE_Q4_K_TILED) ? DFL_XF_Q4K : DFL_XF_NONE;
    const int nb = static_cast<int>(n_in / DFL_QK_K);
    if (kind == DFL_XF_NONE || n_in % DFL_QK_K || nb < 1 || nb > 24 || n_out < 1 || n_out >= (1 << 24)) return p;
    const int ksplit = nb < 16 ? nb : 16, tiles = static_cast<int>((n_out + 15) / 16);
    if (kind == DFL_XF_Q6K && nb > 22 && 2 * tiles < ctx->n_cu) return p;
    for (int R = 1; R <= (kind == DFL_XF_Q4K && nb <= 16 ? 2 : 1); R++)
        for (int tl = 1; tl <= 16 / ksplit; tl++) {
            const int units = (tiles + R - 1) / R, n_wg = (units + tl - 1) / tl;
            if (n_wg > ctx->n_cu) continue;
            p = {kind, ksplit, tl, R, units, n_wg, false};
            // (lines of LDS: the partial tiles and a wave's rows)
            if (static_cast<size_t>(16) * R * 64 * sizeof(float4_t) + static_cast<size_t>(ksplit) * tl * kRowAreaBytes > ctx->lds_bytes) p.kind = DFL_XF_NONE;
            return p;
        }
    return p;
}
// The looping kernel's: K shared by one or two super-blocks a wave, as many waves as the ring leaves room for.
struct WidePlan {
    int ksplit, tl, slots, n_wg;
};
WidePlan rows_wide_plan(const dflash_ctx *ctx, int32_t w_type, int64_t n_in, int64_t n_out) {
    WidePlan p = {0, 0, 0, 0};
    if (!env_int("DFLASH_GEMM_WHOLE", 1) || !env_int("DFLASH_GEMM_WHOLE_LOOP", 1)) return p;
    const int nb = static_cast<int>(n_in / DFL_QK_K);
    if ((w_type != DFLASH_TYPE_Q4_K && w_type != DFLASH_TYPE_Q4_K_TILED) || n_in % DFL_QK_K || nb < 1 || nb > 24 || n_out < 1 || n_out >= (1 << 24)) return p;
    const int tiles = static_cast<int>((n_out + 15) / 16);
    // (two super-blocks a wave take in the rows in 2 us more: from three rounds on; 5120 -> 6144, 16 rows f32, tiled 11.5 :12.1)
    if (nb > 16 && tiles < 3 * ctx->n_cu) return p;
    const int ksplit = nb > 16 ? (nb + 1) / 2 : nb, tl = 16 / ksplit > 0 && nb <= 16 ? 16 / ksplit : 1, waves = ksplit * tl;
    const size_t red = static_cast<size_t>(2) * waves * 64 * sizeof(float4_t);
    if (red >= ctx->lds_bytes) return p;
    const int slots = std::min<int>(kWideSlots, static_cast<int>((ctx->lds_bytes - red) / (static_cast<size_t>(waves) * kWideSlot)));
    if (slots < (nb > 16 ? 5 : 3)) return p;
    p = {ksplit, tl, slots == 5 && nb <= 16 ? 4 : slots, std::min((tiles + tl - 1) / tl, ctx->n_cu)};
    return p;
}
template <typename W, typename XT>
whole_kernel_t rows_direct_fn(int R) {
    if constexpr (!std::is_same<W, Q6W>::value)
        if (R == 2) return gemm_whole_kernel<W, 2, 0, RowSrc<XT>>;
    return gemm_whole_kernel<W, 1, 0, RowSrc<XT>>;
}
}  // namespace

bool dfl_gemm_direct_takes(const dflash_ctx *ctx, int32_t w_type, int64_t n_in, int64_t n_out) {
    return rows_direct_plan(ctx, w_type, n_in, n_out).kind != DFL_XF_NONE || rows_wide_plan(ctx, w_type, n_in, n_out).ksplit;
}

int32_t dfl_gemm_direct(dflash_ctx *ctx, int32_t w_type, const void *w, const void *x, int32_t x_type, float *y, int64_t n_in, int64_t n_out,
                        int32_t n_rows, hipStream_t st) {
    const WholePlan p = rows_direct_plan(ctx, w_type, n_in, n_out);
    const WidePlan wp = rows_wide_plan(ctx, w_type, n_in, n_out);
    if ((p.kind == DFL_XF_NONE && !wp.ksplit) || n_rows < 1 || n_rows > 16)
        return dfl_fail(ctx, DFLASH_ERR_UNSUPPORTED, "gemm_direct: type %d, %lld -> %lld not taken", w_type, static_cast<long long>(n_in),
                        static_cast<long long>(n_out));
    if (reinterpret_cast<uintptr_t>(x) % (x_type == DFLASH_TYPE_F32 ? 16 : 8))
        return dfl_fail(ctx, DFLASH_ERR_ALIGNMENT, "gemm_fewrow: activations must be 16-byte (f32) / 8-byte (f16) aligned");
    const bool q6 = w_type == DFLASH_TYPE_Q6_K, f32 = x_type == DFLASH_TYPE_F32;
    WholeArgs a = {};
    a.w = static_cast<const uint8_t *>(w);
    a.xf = static_cast<const uint8_t *>(x);
    a.y = y;
    a.n_out = static_cast<int>(n_out);
    a.nb = static_cast<int>(n_in / DFL_QK_K);
    a.n_rows = n_rows;
    a.ksplit = p.ksplit;
    a.tl = p.tl;
    a.n_units = p.n_units;
    a.row_bytes = static_cast<uint32_t>(a.nb) * (q6 ? DFL_Q6_K_BYTES : DFL_Q4_K_BYTES);
    a.n_blocks = 1;
    a.rows_last = n_rows;
    if (p.kind == DFL_XF_NONE) {
        a.ksplit = wp.ksplit;
        a.tl = wp.tl;
        const int waves = wp.ksplit * wp.tl;
        const bool tiled = w_type == DFLASH_TYPE_Q4_K_TILED;
        const size_t wlds = static_cast<size_t>(2) * waves * 64 * sizeof(float4_t) + static_cast<size_t>(waves) * wp.slots * kWideSlot;
        const bool two = a.nb > 16;
#define DFL_WIDE_PICK(XT, LEN, SLOTS) (tiled ? gemm_q4k_wide_kernel<XT, true, LEN, SLOTS> : gemm_q4k_wide_kernel<XT, false, LEN, SLOTS>)
#define DFL_WIDE_PICK4(XT) (two ? (wp.slots == 6 ? DFL_WIDE_PICK(XT, 2, 6) : DFL_WIDE_PICK(XT, 2, 5)) \
                                : (wp.slots == 6 ? DFL_WIDE_PICK(XT, 1, 6) : wp.slots == 4 ? DFL_WIDE_PICK(XT, 1, 4) : DFL_WIDE_PICK(XT, 1, 3)))
        const whole_kernel_t wfn = f32 ? DFL_WIDE_PICK4(float) : DFL_WIDE_PICK4(_Float16);
#undef DFL_WIDE_PICK4
#undef DFL_WIDE_PICK
        if (const int32_t rc = dfl_raise_lds_limit(ctx, reinterpret_cast<const void *>(wfn), wlds)) return rc;
        dfl_timed timer(ctx, st, DFL_T_GEMM);
        const dfl_stamp sp(ctx, DFL_T_KERNEL_Q4K_TILED);
        a.pair_off = wp.n_wg;
        whole_launch(wfn, wp.n_wg, 64 * waves, wlds, st, a, sp.start, sp.stop);
        DFL_HIP_CHECK(ctx, hipGetLastError());
        return DFLASH_OK;
    }
    const size_t lds = static_cast<size_t>(16) * p.R * 64 * sizeof(float4_t) + static_cast<size_t>(p.ksplit) * p.tl * kRowAreaBytes;
    const whole_kernel_t fn = q6 ? (f32 ? rows_direct_fn<Q6W, float>(p.R) : rows_direct_fn<Q6W, _Float16>(p.R))
                     : w_type == DFLASH_TYPE_Q4_K_TILED ? (f32 ? rows_direct_fn<Q4W, float>(p.R) : rows_direct_fn<Q4W, _Float16>(p.R))
                                                        : (f32 ? rows_direct_fn<Q4R, float>(p.R) : rows_direct_fn<Q4R, _Float16>(p.R));
    if (lds > 48 * 1024)
        if (const int32_t rc = dfl_raise_lds_limit(ctx, reinterpret_cast<const void *>(fn), lds)) return rc;
    dfl_timed timer(ctx, st, DFL_T_GEMM);
    hipEvent_t start = nullptr, stop = nullptr;
    if (!q6) {  // (Q4_K's slot, whichever kernel the matrix takes)
        const dfl_stamp stamp(ctx, DFL_T_KERNEL_Q4K_TILED);
        start = stamp.start;
        stop = stamp.stop;
    }
    whole_launch(fn, p.n_wg, 64 * p.ksplit * p.tl, lds, st, a, start, stop);
    DFL_HIP_CHECK(ctx, hipGetLastError());
    return DFLASH_OK;
}

namespace {
// One thread per (row, super-block) of the tiled matrix: the row-order block's fields to their places (rows past the
// matrix: zero blocks, d = 0).
__global__ void __launch_bounds__(256)
    q6k_repack_tiled_kernel(const uint8_t *__restrict__ w, uint8_t *__restrict__ out, int n_out, int nb, int64_t n_items) {
    const int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
    if (i >= n_items) return;
    const int b = static_cast<int>(i % nb);
    const int64_t row = i / nb;
    const int tile = static_cast<int>(row >> 4), r = static_cast<int>(row & 15);
    uint8_t *t = out + ((static_cast<size_t>(tile >> 4) * nb + b) * 16 + (tile & 15)) * kQ6TileBytes;
    const bool live = row < n_out;
    const uint8_t *src = w + (static_cast<size_t>(live ? row : 0) * nb + b) * DFL_Q6_K_BYTES;  // 2-byte aligned
    const uint16_t *s16 = reinterpret_cast<const uint16_t *>(src);
    auto put = [&](int dst_off, int src_off16) {  // one 16-byte piece
        uint16_t *d16 = reinterpret_cast<uint16_t *>(t + dst_off);
        for (int k = 0; k < 8; k++) d16[k] = live ? s16[src_off16 + k] : static_cast<uint16_t>(0);
    };
    for (int p = 0; p < 8; p++) put(q6t_ql_piece(r, p), 8 * p);
    for (int p = 0; p < 4; p++) put(q6t_qh_piece(r, p), 64 + 8 * p);
    put(kQ6TSc + r * 16, 96);
    *reinterpret_cast<uint16_t *>(t + kQ6TD + r * 2) = live ? s16[104] : static_cast<uint16_t>(0);
}
}  // namespace

extern "C" size_t dflash_q6k_tiled_bytes(int64_t n_in, int64_t n_out) {
    if (n_in <= 0 || n_out <= 0 || n_in % DFL_QK_K) return 0;
    const size_t groups = (static_cast<size_t>(n_out) + 255) / 256;
    return groups * static_cast<size_t>(n_in / DFL_QK_K) * 16 * kQ6TileBytes;
}

extern "C" int32_t dflash_repack_q6k_tiled(dflash_ctx *ctx, const void *w, void *w_tiled, int64_t n_in, int64_t n_out,
                                           dflash_stream_t stream) {
    if (!ctx) return DFLASH_ERR_INVALID_INPUT;
    if (!w || !w_tiled) return dfl_fail(ctx, DFLASH_ERR_INVALID_INPUT, "repack_q6k_tiled: null pointer");
    if (n_in <= 0 || n_out <= 0 || n_in % DFL_QK_K || n_in > 0x7fffffffll || n_out > 0x7fffffffll)
        return dfl_fail(ctx, DFLASH_ERR_BAD_SHAPE, "repack_q6k_tiled: n_in %lld / n_out %lld", static_cast<long long>(n_in),
                        static_cast<long long>(n_out));
    if (reinterpret_cast<uintptr_t>(w) % 2 || reinterpret_cast<uintptr_t>(w_tiled) % 128)
        return dfl_fail(ctx, DFLASH_ERR_ALIGNMENT, "repack_q6k_tiled: source must be 2-byte, destination 128-byte aligned");
    const size_t out_bytes = dflash_q6k_tiled_bytes(n_in, n_out);
    const int nb = static_cast<int>(n_in / DFL_QK_K);
    const size_t in_bytes = static_cast<size_t>(n_out) * nb * DFL_Q6_K_BYTES;
    if (dfl_ranges_overlap(w_tiled, out_bytes, w, in_bytes)) return dfl_fail(ctx, DFLASH_ERR_ALIAS, "repack_q6k_tiled: buffers overlap");
    // a tiled tensor goes to the fast kernels unconditionally: it must be one they can take
    if (const int32_t rc = dflash_check_scale_range(ctx, DFLASH_TYPE_Q6_K, w, in_bytes / DFL_Q6_K_BYTES, nullptr, stream)) return rc;
    const int64_t n_items = static_cast<int64_t>((static_cast<size_t>(n_out) + 255) / 256 * 256) * nb;
    const int64_t blocks = (n_items + 255) / 256;
    if (blocks > 0x7fffffffll) return dfl_fail(ctx, DFLASH_ERR_BAD_SHAPE, "repack_q6k_tiled: matrix too large");
    q6k_repack_tiled_kernel<<<static_cast<unsigned>(blocks), 256, 0, static_cast<hipStream_t>(stream)>>>(
        static_cast<const uint8_t *>(w), static_cast<uint8_t *>(w_tiled), static_cast<int>(n_out), nb, n_items);
    DFL_HIP_CHECK(ctx, hipGetLastError());
    return DFLASH_OK;
}

extern "C" size_t dflash_xf_bytes(int64_t n_in) { return n_in > 0 && n_in % DFL_QK_K == 0 ? dfl_xf_bytes(n_in) : 0; }

namespace {
// The public entries take a range-checked tensor only (there is no f32 kernel behind them): the tiled order, or
// DFLASH_TYPE_Q6_K | DFLASH_TYPE_RANGE_CHECKED.  Returns the bare type, or -1.
int32_t xf_public_type(int32_t w_type) {
    if (w_type == DFLASH_TYPE_Q4_K_TILED || w_type == DFLASH_TYPE_Q6_K_TILED) return w_type;
    if (w_type == (DFLASH_TYPE_Q6_K | DFLASH_TYPE_RANGE_CHECKED)) return DFLASH_TYPE_Q6_K;
    return -1;
}
}  // namespace

extern "C" int32_t dflash_gemm_fewrow_xf_kind(dflash_ctx *ctx, int32_t w_type, int64_t n_in, int64_t n_out) {
    const int32_t t = xf_public_type(w_type);
    return ctx && t >= 0 ? dfl_whole_kind(ctx, t, n_in, n_out, 0) : DFL_XF_NONE;
}

extern "C" int32_t dflash_pack_xf(dflash_ctx *ctx, const void *x, int32_t x_type, int32_t n_rows, int64_t n_in, int32_t kind,
                                  void *xf, dflash_stream_t stream) {
    if (!ctx) return DFLASH_ERR_INVALID_INPUT;
    if (!x || !xf || n_rows < 1 || n_rows > 16 || n_in <= 0 || n_in % DFL_QK_K || n_in > (1 << 24))
        return dfl_fail(ctx, DFLASH_ERR_BAD_SHAPE, "pack_xf: n_rows %d, n_in %lld", n_rows, static_cast<long long>(n_in));
    if (kind != DFL_XF_Q4K && kind != DFL_XF_Q6K) return dfl_fail(ctx, DFLASH_ERR_UNSUPPORTED, "pack_xf: kind %d", kind);
    if (x_type != DFLASH_TYPE_F32 && x_type != DFLASH_TYPE_F16) return dfl_fail(ctx, DFLASH_ERR_UNSUPPORTED, "pack_xf: x_type %d", x_type);
    if (reinterpret_cast<uintptr_t>(xf) % 16) return dfl_fail(ctx, DFLASH_ERR_ALIGNMENT, "pack_xf: xf must be 16-byte aligned");
    const size_t x_bytes = static_cast<size_t>(n_rows) * n_in * (x_type == DFLASH_TYPE_F32 ? 4 : 2);
    if (dfl_ranges_overlap(x, x_bytes, xf, dfl_xf_bytes(n_in))) return dfl_fail(ctx, DFLASH_ERR_ALIAS, "pack_xf: xf overlaps x");
    hipStream_t st = static_cast<hipStream_t>(stream);
    const dim3 grid(static_cast<unsigned>((n_in / 8 + 255) / 256), n_rows);
    if (x_type == DFLASH_TYPE_F32)
        pack_xf_kernel<float><<<grid, 256, 0, st>>>(static_cast<const float *>(x), n_rows, static_cast<int>(n_in), kind, static_cast<uint8_t *>(xf));
    else
        pack_xf_kernel<_Float16><<<grid, 256, 0, st>>>(static_cast<const _Float16 *>(x), n_rows, static_cast<int>(n_in), kind,
                                                     static_cast<uint8_t *>(xf));
    DFL_HIP_CHECK(ctx, hipGetLastError());
    return DFLASH_OK;
}

extern "C" int32_t dflash_gemm_fewrow_xf(dflash_ctx *ctx, int32_t w_type, const void *w, const void *xf, float *y, int64_t n_in,
                                         int64_t n_out, int32_t n_rows, dflash_stream_t stream) {
    if (!ctx) return DFLASH_ERR_INVALID_INPUT;
    const int32_t tagged = w_type;
    w_type = xf_public_type(tagged);
    if (w_type < 0)
        return dfl_fail(ctx, DFLASH_ERR_UNSUPPORTED,
                        "gemm_fewrow_xf: type tag %d: only DFLASH_TYPE_Q4_K_TILED, DFLASH_TYPE_Q6_K_TILED and DFLASH_TYPE_Q6_K | "
                        "DFLASH_TYPE_RANGE_CHECKED (a tensor that passed dflash_check_scale_range) are taken",
                        tagged);
    if (dfl_whole_kind(ctx, w_type, n_in, n_out, 0) == DFL_XF_NONE)
        return dfl_fail(ctx, DFLASH_ERR_UNSUPPORTED, "gemm_fewrow_xf: type %d, %lld -> %lld is not taken by the whole-K kernels", w_type,
                        static_cast<long long>(n_in), static_cast<long long>(n_out));
    if (n_in > 0 && n_out > 0 && y && xf && w) {
        const size_t wb = w_type == DFLASH_TYPE_Q4_K_TILED   ? dflash_q4k_tiled_bytes(n_in, n_out)
                          : w_type == DFLASH_TYPE_Q6_K_TILED ? dflash_q6k_tiled_bytes(n_in, n_out)
                                                             : dflash_row_bytes(w_type, n_in) * n_out;
        const size_t yb = static_cast<size_t>(n_rows > 0 ? n_rows : 1) * n_out * sizeof(float);
        const size_t xb = static_cast<size_t>(n_rows > 16 ? (n_rows + 15) / 16 : 1) * dfl_xf_bytes(n_in);
        if (dfl_ranges_overlap(y, yb, xf, xb) || dfl_ranges_overlap(y, yb, w, wb))
            return dfl_fail(ctx, DFLASH_ERR_ALIAS, "gemm_fewrow_xf: y aliases an input");
    }
    return dfl_gemm_whole(ctx, w_type, w, xf, y, n_in, n_out, n_rows, 0, nullptr, DFL_XF_NONE, static_cast<hipStream_t>(stream));
}
