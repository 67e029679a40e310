// The wide Q4_K product of a dense layer's FFN: silu(x . gate^T) * (x . up^T) for up to sixteen rows, gate and up one fused
// matrix in the tiled order, many more tiles than one round of the chip (5120 -> 2 x 17408: 100 MB).  Same contraction as
// encode_mat_mat_dispatch_dflash_verify (metal_forward/dispatch.rs:365-378) on both halves, and the SwiGLU that follows.
#include "common.h"
#include "lds_read.h"
#include "mfma_unpack.h"

#include <algorithm>

namespace {

typedef const __attribute__((address_space(1))) void *gptr_t;
typedef __attribute__((address_space(3))) void *lptr_t;

constexpr int kTile = 16 * DFL_Q4_K_BYTES;  // sixteen weight rows of a super-block: 2304 bytes
constexpr int kStage = 16 * kTile;          // a tile group's
constexpr int kXStage = 8192 + 1024;        // a super-block of the rows: fragments (XF) and sub-block sums (XS)
constexpr int kChunk = 4;                   // super-blocks of the rows between two barriers
constexpr int kChunkLoads = kChunk * 9;
constexpr int kPerMost = 7;  // units a workgroup has under way: fourteen waves and the one that brings in the rows
constexpr int kDepth = 2;    // stages a wave has under way
constexpr size_t kXBytes = 2 * static_cast<size_t>(kChunk) * kXStage;

constexpr int vmcnt(int n) { return ((n & 0xF) | ((n & 0x30) << 10)) | 0x0F70; }  // s_waitcnt vmcnt(n) (gfx9 encoding)

__device__ __forceinline__ uint32_t lds_at(const void *p) {
    return static_cast<uint32_t>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) const void *)(p)));
}
// A lane's operands of a super-block: its weight row's header and 32 quant bytes, the minima's A operand and the eight fragments.
struct Operands {
    u32x4_t hdr, q0, q1;
    half8_t a_min, af[8];
};
__device__ __forceinline__ void read_operands(Operands &o, uint32_t blk, uint32_t blk_q, uint32_t x) {
    o.hdr = lds_read<u32x4_t, 0>(blk);
    o.q0 = lds_read<u32x4_t, 16>(blk_q);
    o.q1 = lds_read<u32x4_t, 32>(blk_q);
    o.a_min = lds_read<half8_t, 8192>(x);
    static_for<0, 8>([&](auto t) { o.af[decltype(t)::value] = lds_read<half8_t, 1024 * decltype(t)::value>(x); });
}
__device__ __forceinline__ void weights_arrived(Operands &o) {  // (what follows may load into their place)
    lds_arrived<11>(o.hdr);
    lds_arrived<10>(o.q0);
    lds_arrived<9>(o.q1);
    asm volatile("" ::: "memory");
}
// The minima's MFMA, then the eight of the scaled nibbles, into one accumulator (the order of the many-row product with sums,
// gemm_rows.hip, whose rows have these bits).
__device__ __forceinline__ void products(Operands &o, int g, uint32_t sc_sel, Q4KMagic magic, float4_t &acc) {
    const u32x4_t hdr = o.hdr;
    const uint32_t upper = 0u - static_cast<uint32_t>(g >> 1);
    const uint32_t sc_lo = hdr.y & 0x3F3F3F3Fu, sc_hi = (hdr.w & 0x0F0F0F0Fu) | ((hdr.y >> 2) & 0x30303030u);
    const uint32_t mn_lo = hdr.z & 0x3F3F3F3Fu, mn_hi = ((hdr.w >> 4) & 0x0F0F0F0Fu) | ((hdr.z >> 2) & 0x30303030u);
    const uint32_t sc_word = (sc_hi & upper) | (sc_lo & ~upper), mn_word = (mn_hi & upper) | (mn_lo & ~upper);
    const half2_t dm = __builtin_bit_cast(half2_t, hdr.x);
    const half2_t p_sc = as_half2(__builtin_amdgcn_perm(0x64646464u, sc_word, sc_sel));
    const half2_t p_mn = as_half2(__builtin_amdgcn_perm(0x64646464u, mn_word, sc_sel));
    const half2_t neg = dm * splat(static_cast<_Float16>(-1024.0f));
    const half2_t S = __builtin_elementwise_fma(p_sc, splat(dm[0]), splat(neg[0]));
    const half2_t M = __builtin_elementwise_fma(p_mn, splat(-dm[1]), splat(-neg[1]));
    const half2_t unbias = {static_cast<_Float16>(-1024.0f), static_cast<_Float16>(-64.0f)};
    const half2_t Cs = S * unbias;
    const half2_t s2l = splat(S[0]), c2l = splat(Cs[0]), s2h = splat(S[1]), c2h = splat(Cs[1]);
    const uint32_t qw[8] = {o.q0.x, o.q0.y, o.q0.z, o.q0.w, o.q1.x, o.q1.y, o.q1.z, o.q1.w};
    lds_arrived<8>(o.a_min);
    acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(o.a_min, q4k_min_operand(M), acc, 0, 0, 0);
    static_for<0, 8>([&](auto i) {
        constexpr int t = decltype(i)::value, j = t & 3;
        const half8_t b = t < 4 ? unpack_scale<false>(qw[2 * j], qw[2 * j + 1], s2l, c2l, magic.lo) : unpack_scale<true>(qw[2 * j], qw[2 * j + 1], s2h, c2h, magic.hi);
        lds_arrived<7 - t>(o.af[t]);
        acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(o.af[t], b, acc, 0, 0, 0);
    });
}

// A wave owns a tile (a unit is a tile of gate and the same one of up: two waves) over the whole K and streams it through a ring of
// its own with direct-to-LDS loads; one more wave brings in the rows, kChunk super-blocks at a time, for all of them.  One
// barrier a chunk hands a buffer of rows over: behind it chunk k + 1 has landed and chunk k's place is free.  (The row loads are
// not among the loads that a wave with weights counts, which return in order.)  What a wave reads of a stage it has in registers
// ahead of the products, and the slot is loaded into again at once.
// Units that are left over when every workgroup has as many as any are cut by weight rows, `cut` ways, over as many workgroups.
// What bounds it: the stream, which without the products takes 20-21 us for the 100 MB of 5120 -> 2 x 17408 (5.0 TB/s), 3.5 of them the start; with
// them 24-25 (dispatch stamps; the streaming kernel 26.5-27.8 and its reduction 4.2-5): 114 vector instructions a stage and wave, ten waves on four SIMDs.
// Measured on the way, same matrix: two super-blocks of rows a barrier 28 (four 25.2; ring of six; of two, which leaves the rows' loads
// less to stand behind, 25.2 : 25.7 for one of three); leftover units whole, on every fourth CU 24.8; words in LDS in place of the barriers 28-31 (polling
// takes LDS cycles from everybody); the sub-block sums made here by the wave that brings in the rows 26.1.
struct DenseSplit {
    int per_wg, left, cut;  // units of every workgroup; units left over, and the parts of each: workgroup i < left * cut has one
};
__global__ void __launch_bounds__(64 * (2 * kPerMost + 1))
    gemm_q4k_dense_pair_kernel(const uint8_t *__restrict__ w, const uint8_t *__restrict__ xf, const uint8_t *__restrict__ xs, int nb, int per, int up_tiles,
                               int n_rows, DenseSplit split, int ffn, _Float16 *__restrict__ y) {
    extern __shared__ uint8_t lds[];  // rows [2][kChunk][kXStage], up tiles [per][64] float4, rings [wave][kDepth][kTile]
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), wg = blockIdx.x;
    const int part_of = split.per_wg * gridDim.x + wg / split.cut;  // the unit of which this workgroup has a part
    const int n_units = split.per_wg + (wg < split.left * split.cut ? 1 : 0);
    const int n_rounds = (n_units + per - 1) / per, n_chunks = (nb + kChunk - 1) / kChunk, total = n_rounds * n_chunks;
    auto barrier = [] {
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    if (wave >= 2 * per) {
        int c = 0, slot = 0;
        auto load = [&]() {  // nine loads of a kilobyte for a super-block (past the last, that one again)
#pragma unroll
            for (int i = 0; i < kChunk; i++) {
                const int b = min(c * kChunk + i, nb - 1);
                uint8_t *dst = lds + (slot * kChunk + i) * kXStage;
                const uint8_t *src = xf + static_cast<size_t>(b) * 8192 + lane * 16;
#pragma unroll
                for (int t = 0; t < 8; t++) __builtin_amdgcn_global_load_lds((gptr_t)(src + t * 1024), (lptr_t)(dst + t * 1024), 16, 0, 0);
                __builtin_amdgcn_global_load_lds((gptr_t)(xs + static_cast<size_t>(b) * 1024 + lane * 16), (lptr_t)(dst + 8192), 16, 0, 0);
            }
            if (++c == n_chunks) c = 0;
            slot ^= 1;
        };
        load();
        load();  // (two chunks at least: the host's rule)
        __builtin_amdgcn_s_waitcnt(vmcnt(kChunkLoads));
        barrier();
        for (int k = 0; k < total; k++) {
            __builtin_amdgcn_s_waitcnt(vmcnt(0));  // chunk k + 1
            barrier();
            if (k + 2 < total) load();
        }
        return;
    }
    const int half = wave >= per, first = wave - half * per;
    const int n = lane & 15, g = lane >> 4;
    uint8_t *ring = lds + kXBytes + static_cast<size_t>(per) * 1024 + static_cast<size_t>(wave) * kDepth * kTile;
    const int units = n_units > first ? (n_units - first + per - 1) / per : 0;  // of this wave: first, first + per, ...
    // The next stage to issue: super-block i_b of the wave's unit i_unit.  Three loads whatever there is, so that the waits need not
    // ask: of a part every lane past it takes its last piece again, and past the last unit there is one piece, which nobody reads.
    int i_b = 0, i_unit = first, i_slot = 0, step = kStage;
    const uint8_t *src = w;
    uint32_t off[3] = {0, 0, 0};
    auto seek = [&]() {
        const bool part = i_unit >= split.per_wg, any = i_unit < n_units;
        const int tile = (part ? part_of : wg * split.per_wg + i_unit) + half * up_tiles;
        const int last = !any ? 0 : part ? 144 / split.cut - 1 : 143;
        src = any ? w + static_cast<size_t>(tile >> 4) * nb * kStage + (tile & 15) * kTile + (part ? (wg % split.cut) * (kTile / split.cut) : 0) : w;
        step = any ? kStage : 0;
#pragma unroll
        for (int j = 0; j < 3; j++) off[j] = 16u * static_cast<uint32_t>(min(64 * j + lane, last));
    };
    seek();
    auto issue = [&]() {
        uint8_t *dst = ring + i_slot * kTile;
        __builtin_amdgcn_global_load_lds((gptr_t)(src + off[0]), (lptr_t)(dst), 16, 0, 0);
        __builtin_amdgcn_global_load_lds((gptr_t)(src + off[1]), (lptr_t)(dst + 1024), 16, 0, 0);
        if (lane < 16) __builtin_amdgcn_global_load_lds((gptr_t)(src + off[2]), (lptr_t)(dst + 2048), 16, 0, 0);
        src += step;
        i_slot ^= 1;
    };
    auto next = [&]() {  // (apart from the loads: nothing read from LDS is under way here)
        if (++i_b == nb) {
            i_b = 0;
            i_unit += per;
            seek();
        }
    };
    issue();
    next();
    issue();
    next();
    const uint32_t sc_sel = (lane & 16) ? 0x04030402u : 0x04010400u;
    const Q4KMagic magic = q4k_magic();
    float4_t *xchg = reinterpret_cast<float4_t *>(lds + kXBytes) + first * 64 + lane;
    const uint32_t x_at = lds_at(lds) + lane * 16, ring_at = lds_at(ring);
    int slot = 0, xslot = 0;
    barrier();
    for (int r = 0; r < n_rounds; r++) {
        const bool active = r < units;
        const int row = first + r * per >= split.per_wg ? n & (16 / split.cut - 1) : n;  // (a part's rows are the slot's first)
        float4_t acc = {0, 0, 0, 0};
        for (int c = 0; c < n_chunks; c++, xslot ^= 1) {
            if (active) {
                const int len = min(kChunk, nb - c * kChunk);
                uint32_t x = x_at + xslot * (kChunk * kXStage);
                for (int s = 0; s < len; s++, x += kXStage, slot ^= 1) {
                    __builtin_amdgcn_s_waitcnt(vmcnt(3));  // the stage has landed when only the one behind it is under way
                    const uint32_t blk = ring_at + slot * kTile + row * DFL_Q4_K_BYTES;
                    Operands o;
                    read_operands(o, blk, blk + 32 * g, x);
                    weights_arrived(o);
                    issue();  // (into the slot just read)
                    products(o, g, sc_sel, magic, acc);
                    next();
                }
            }
            if (c + 1 == n_chunks && active && half) *xchg = acc;
            barrier();
        }
        if (active && !half) {
            const float4_t up = *xchg;
            const int u = first + r * per;
            const bool part = u >= split.per_wg;
            const int col = (part ? part_of : wg * split.per_wg + u) * 16 + n;
            if (part && n / (16 / split.cut) != wg % split.cut) continue;
#pragma unroll
            for (int i = 0; i < 4; i++) {
                float o = acc[i] / (1.0f + expf(-acc[i])) * up[i];
                asm volatile("" : "+v"(o));  // (rounded to f32 first: the product is not fused into the conversion)
                if (4 * g + i < n_rows) y[static_cast<size_t>(4 * g + i) * ffn + col] = static_cast<_Float16>(o);
            }
        }
    }
    __builtin_amdgcn_s_waitcnt(vmcnt(0));  // (nothing is under way into LDS when the wave ends)
}

struct DensePlan {
    int units, n_wg, per;
    DenseSplit split;
    size_t lds;
};
DensePlan dense_plan(const dflash_ctx *ctx, int32_t w_type, int64_t n_in, int64_t ffn) {
    DensePlan p = {0, 0, 0, {0, 0, 1}, 0};
    if (w_type != DFLASH_TYPE_Q4_K_TILED || n_in <= 0 || n_in % DFL_QK_K || ffn <= 0 || ffn % 16 || ffn > (1 << 22)) return p;
    if (n_in > 8192 || n_in / DFL_QK_K <= kChunk) return p;  // (a norm leaves rows of at most 8192 values in fragment order)
    const int units = static_cast<int>(ffn / 16);
    p.n_wg = std::min(units, ctx->n_cu);
    p.split.per_wg = units / p.n_wg;
    p.split.left = units - p.split.per_wg * p.n_wg;
    while (p.split.left && p.split.cut < 16 && p.split.left * p.split.cut * 2 <= p.n_wg) p.split.cut *= 2;
    const int most = p.split.per_wg + (p.split.left ? 1 : 0), rounds = (most + kPerMost - 1) / kPerMost;
    p.per = (most + rounds - 1) / rounds;
    p.lds = kXBytes + static_cast<size_t>(p.per) * (1024 + 2 * kDepth * kTile);
    if (p.lds > ctx->lds_bytes) return p;
    p.units = units;
    return p;
}

}  // namespace

// Every shape that a whole-K launch does not take and that gives each CU a unit.  us a layer, streaming kernel and its reduction : this one,
// 1 row and 16 rows (q/k/v, attention, norms and down among them): 5120 -> 2 x 17408 90.5 : 90.6  99.0 : 95.4, 12288 78.8 : 76.6  85.0 : 81.2,
// 8192 67.0 : 66.3  73.9 : 70.0, 6144 63.5 : 63.4  69.2 : 66.3; 4096 -> 2 x 14336 68.3 : 65.6  72.6 : 69.0, 8192 55.7 : 54.3  61.8 : 56.9;
// 2560 -> 2 x 9728 54.2 : 52.5  57.7 : 54.3; 2048 -> 2 x 11264 50.2 : 47.9  53.5 : 49.7; 8192 -> 2 x 28672 154.7 : 150.9  164.5 : 156.1.
bool dfl_gemm_dense_pair_takes(const dflash_ctx *ctx, int32_t w_type, int64_t n_in, int64_t ffn) {
    return dense_plan(ctx, w_type, n_in, ffn).units >= ctx->n_cu;
}

int32_t dfl_gemm_dense_pair(dflash_ctx *ctx, int32_t w_type, const void *w, const void *xf, const void *xs, void *y_f16, int64_t n_in, int64_t ffn,
                            int32_t n_rows, hipStream_t st) {
    const DensePlan p = dense_plan(ctx, w_type, n_in, ffn);
    if (!p.units || n_rows < 1 || n_rows > 16) return dfl_fail(ctx, DFLASH_ERR_UNSUPPORTED, "gemm_dense_pair: shape not taken");
    if (!w || !xf || !xs || !y_f16) return dfl_fail(ctx, DFLASH_ERR_INVALID_INPUT, "gemm_dense_pair: null pointer");
    if (reinterpret_cast<uintptr_t>(w) % 128 || reinterpret_cast<uintptr_t>(xf) % 16 || reinterpret_cast<uintptr_t>(xs) % 16)
        return dfl_fail(ctx, DFLASH_ERR_ALIGNMENT, "gemm_dense_pair: tiled Q4_K weights must be 128-byte aligned, rows 16-byte aligned");
    if (const int32_t rc = dfl_raise_lds_limit(ctx, reinterpret_cast<const void *>(gemm_q4k_dense_pair_kernel), p.lds)) return rc;
    dfl_timed timer(ctx, st, DFL_T_GEMM);
    gemm_q4k_dense_pair_kernel<<<p.n_wg, 64 * (2 * p.per + 1), p.lds, st>>>(
        static_cast<const uint8_t *>(w), static_cast<const uint8_t *>(xf), static_cast<const uint8_t *>(xs), static_cast<int>(n_in / DFL_QK_K), p.per,
        p.units, n_rows, p.split, static_cast<int>(ffn), static_cast<_Float16 *>(y_f16));
    DFL_HIP_CHECK(ctx, hipGetLastError());
    return DFLASH_OK;
}
