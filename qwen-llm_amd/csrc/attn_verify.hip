// Block-causal verify attention: the 16 draft rows of a block attend the whole prefix and
// each other causally, over an f16 KV cache, GQA.
//
// Replaces the reference's per-row loop (metal_dflash.rs:9963-10062: scatter one K/V row,
// then one single-query decode attention, sixteen times; kernels attn_v4.metal /
// attn.metal:266-336) with one pass that streams the KV cache once for all 16 rows:
//     o[i][h] = softmax(q[i][h] . K[0..L+i, kv(h)] * scale) . V[0..L+i, kv(h)]
//
// Mapping onto CDNA4 (split-KV flash decoding on MFMA):
//  * grid = (KV splits) x (KV heads); a workgroup owns one KV head and one contiguous chunk of
//    key positions; each of its waves owns one query head of the GQA group, i.e. a 16-row tile
//    (the block's rows are exactly the 16-wide side of v_mfma_f32_16x16x32_f16).
//  * K and V stream HBM -> LDS once per workgroup in stages of 32 keys (direct-to-LDS loads into a
//    ring of buffers, the next stages in flight while one is consumed), so the group's heads share
//    one copy; both tiles are bank-swizzled on the way in so that MFMA operand reads are conflict-free.
//  * scores are computed transposed, S^T = K . Q^T: K rows are the A operand, Q^T stays in
//    registers for the whole kernel (pre-multiplied by scale*log2(e), rounded to f16 as the
//    reference's decode kernel does, attn_v4.metal:20-31).  The result leaves every lane holding
//    one query row and eight consecutive keys of the stage, which is exactly the B operand of the
//    second product O^T = V^T . P^T, so probabilities never move between lanes.
//  * V is cached transposed, [kv head][dim][position]: the A operand of O^T wants 8 consecutive
//    positions of one dim, 16 contiguous bytes there.
//  * online softmax in base 2 on the lanes' own values; the running maximum is shared by the
//    four lanes of a row with two cross-lane exchanges per stage, the accumulator rescale is
//    skipped while no row's maximum moves, and stages every row sees in full skip the mask.
//  * each workgroup writes (m, l, O) partials; a second small kernel merges the splits.
#include "common.h"
#include "lds_read.h"
#include "rope_head.h"

#include <cmath>
#include <algorithm>
#include <cstdlib>

namespace {

typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef _Float16 half4_t __attribute__((ext_vector_type(4)));
typedef float float4_t __attribute__((ext_vector_type(4)));

constexpr float kLog2e = 1.4426950408889634f;

// exchange with the lane 16 / 32 positions away (the other lanes that hold the same query row)
__device__ __forceinline__ float xor_lane(float v, int mask) {
    return __shfl_xor(v, mask, 64);
}

typedef const __attribute__((address_space(1))) void *gptr_t;
typedef __attribute__((address_space(3))) void *lptr_t;

constexpr int kAttnBufs = 4;  // LDS ring: two stages in flight, the one whose scores are computed, the one whose values are read

// s_waitcnt vmcnt(n) lgkmcnt(0) (gfx9 encoding)
constexpr int attn_vmcnt(int n) { return ((n & 0xF) | ((n & 0x30) << 10)) | 0x0070; }

// LDS reads sixteen lanes of 16 bytes a clock (64 banks of 4 bytes) when they fall into sixteen different sixteenths of 256
// bytes.  K: 16-byte chunk j of key row r sits at chunk j ^ swz(r): the sixteen lanes of an MFMA operand read rows 8 (n >> 2) +
// (n & 3) at the same j, whole multiples of 256 bytes apart from heads of 128 on (sixteen values; heads of 64 have eight
// chunks a row, two rows to 256 bytes, and eight values do).  V^T: chunk g of dim d sits at g ^ ((d >> 1) & 3): the lanes read
// sixteen dims, 64 bytes apart, at the same g.  Measured, reads of this pattern: 222 bytes a clock and CU (124 with eight values
// for K and V as it comes; contiguous lanes 217).
template <int CH>
__device__ __forceinline__ int attn_swz(int r) { return (r & 3) | ((r >> 1) & (CH >= 16 ? 12 : 4)); }
__device__ __forceinline__ int attn_swz_v(int d) { return (d >> 1) & 3; }

// Keys per KV split for n_pos visible positions: an even share of `want` splits, rounded up to
// whole 32-key stages, at least min_chunk.  Host and kernels use the same rule, so a launch whose
// context length is only known on the device (a captured graph) can size its grid for the largest
// context and let surplus workgroups leave.
__host__ __device__ __forceinline__ int64_t attn_chunk(int64_t n_pos, int64_t want, int64_t min_chunk) {
    // (32-bit division where the positions fit: the 64-bit one is 150 instructions at the head of every workgroup)
    int64_t chunk = n_pos + want <= 0x7fffffff ? static_cast<uint32_t>(n_pos + want - 1) / static_cast<uint32_t>(want) : (n_pos + want - 1) / want;
    chunk = (chunk + 31) / 32 * 32;
    return chunk < min_chunk ? min_chunk : chunk;
}
__host__ __device__ __forceinline__ int attn_splits(int64_t n_pos, int64_t want, int64_t min_chunk) {
    const int64_t chunk = attn_chunk(n_pos, want, min_chunk);
    return static_cast<int>(n_pos <= 0x7fffffff ? (static_cast<uint32_t>(n_pos) + static_cast<uint32_t>(chunk) - 1) / static_cast<uint32_t>(chunk)
                                                : (n_pos + chunk - 1) / chunk);
}

// Eight consecutive query values (16-byte aligned): asked for ahead of everything else and read behind the first stages'
// requests.  Asm loads with a wait of the kernel's own: the compiler, which cannot know how many stage loads follow
// them, would wait for those as well.  (The build refuses this kernel if it uses scratch: see build.py.)
template <typename TQ>
struct AttnQ8;
template <>
struct AttnQ8<float> {
    float4_t a, b;
    template <int OFF>
    __device__ __forceinline__ void load(const float *p) {
        asm volatile("global_load_dwordx4 %0, %1, off offset:%2" : "=v"(a) : "v"(p), "n"(OFF * 4) : "memory");
        asm volatile("global_load_dwordx4 %0, %1, off offset:%2" : "=v"(b) : "v"(p), "n"(OFF * 4 + 16) : "memory");
    }
    __device__ __forceinline__ void arrived() { asm volatile("" : "+v"(a), "+v"(b)); }
    __device__ __forceinline__ float get(int i) const { return i < 4 ? a[i] : b[i - 4]; }
};
template <>
struct AttnQ8<_Float16> {
    half8_t a;
    template <int OFF>
    __device__ __forceinline__ void load(const _Float16 *p) {
        asm volatile("global_load_dwordx4 %0, %1, off offset:%2" : "=v"(a) : "v"(p), "n"(OFF * 2) : "memory");
    }
    __device__ __forceinline__ void arrived() { asm volatile("" : "+v"(a)); }
    __device__ __forceinline__ float get(int i) const { return static_cast<float>(a[i]); }
};
template <int S, int KS, typename TQ>
__device__ __forceinline__ void attn_load_q(AttnQ8<TQ> *v, const TQ *p) {
    if constexpr (S < KS) {
        v[S].template load<32 * S>(p);
        attn_load_q<S + 1, KS>(v, p);
    }
}

#ifdef DFLASH_TRACE
// Debug build only: per-workgroup time stamps (100 MHz constant clock).
__device__ unsigned long long *g_attn_trace = nullptr;  // [n_wg][16]
#define ATT_TR(i)                                                                                                   \
    do {                                                                                                            \
        if (threadIdx.x == 0 && g_attn_trace)                                                                       \
            g_attn_trace[(blockIdx.y * gridDim.x + blockIdx.x) * 16 + (i)] = wall_clock64();                        \
    } while (0)
#else
#define ATT_TR(i) \
    do {          \
    } while (0)
#endif

// s_waitcnt vmcnt(n), lgkmcnt(0) for a wave-uniform n: at most n loads into LDS still on their way, and this wave's LDS
// reads done (the barrier that follows hands what they read to the next loads)
__device__ __forceinline__ void attn_wait(int n) {
    switch (n) {
#define DFL_W(N) case N: __builtin_amdgcn_s_waitcnt(attn_vmcnt(N)); break
        DFL_W(1); DFL_W(2); DFL_W(3); DFL_W(4); DFL_W(5); DFL_W(6); DFL_W(7); DFL_W(8); DFL_W(10); DFL_W(11); DFL_W(12);
        DFL_W(14); DFL_W(15); DFL_W(16); DFL_W(18); DFL_W(21); DFL_W(22); DFL_W(24); DFL_W(32); DFL_W(33); DFL_W(48);
#undef DFL_W
        case 64: case 96: __builtin_amdgcn_s_waitcnt(attn_vmcnt(63)); break;
        default: __builtin_amdgcn_s_waitcnt(attn_vmcnt(0)); break;
    }
}

// Splits are merged in order: what came before times `old`, plus the next one's result times `next`.
struct AttnMerge {
    float m, old, next;
    __device__ __forceinline__ AttnMerge(float m_before, float m_next) {
        m = fmaxf(m_before, m_next);
        old = m_before == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(m_before - m);
        next = m_next == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(m_next - m);
    }
    __device__ __forceinline__ float add(float before, float v) const { return __builtin_fmaf(next, v, old * before); }
};

// A lane's dims 16 t + 4 g + i of row n, as f16 in fragment order: it has four dims of an octet, the lane 16 away the other
// four; even lane rows take tile t's octets, odd ones tile t + 1's.
template <int DT>
__device__ __forceinline__ void attn_store_xf(float4_t (&tot)[DT], void *out_xf, int kind, int n, int g, int dim0, bool live) {
#pragma unroll
    for (int t = 0; t < DT; t += 2) {
#pragma unroll
        for (int i = 0; i < 4; i++) {
            float lo = tot[t][i], hi = tot[t + 1][i];
            dfl_swap16(lo, hi);
            tot[t][i] = lo;
            tot[t + 1][i] = hi;
        }
        const float4_t a = tot[t], b = tot[t + 1];
        if (live) dfl_xf_store(out_xf, kind, n, dim0 + 16 * (t + (g & 1)) + 8 * (g >> 1), a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]);
    }
}

// ROPE: the block's rows come as the projections leave them, [row][query heads | key heads | value heads] in f32.  A wave norms and
// rotates its head's queries in registers; where a workgroup's keys reach into the block, two waves more make the block's keys and
// values of its KV head, put them over what the cache still holds there in LDS, and (in the first part of a group) into the
// cache.  Elsewhere those two waves end at once.  The arithmetic is that of qk_norm_rope_kernel, bit for bit; sines and cosines
// come from a table of the block, [row][cosines, sines], made once a block, which waits with the norm's weights in the ring's last
// buffer, ahead of the stage that comes there.
// What bounds it: the launch of the rotation was one trip to memory with little to do; here that trip is the one the first stages
// are on anyway, and what is left is 450 vector instructions a wave ahead of the first scores (heads of 256).  Rotation and attention,
// behind 2 k of context: 16 rows of 16 / 2 heads of 256 3.9 + 11.2 -> 12.5 us, one row 3.5 + 7.9 -> 9.6, 16 rows of 32 / 8 heads
// of 128 4.9 + 7.7 -> 9.4.  (The block's keys and values by the heads' waves, behind their queries: 14.0, 10.5 and 10.5; by one wave of
// a workgroup of one, through LDS: 12 us more a launch.)
struct AttnRope {
    const float *table, *q_w, *k_w;
    float eps;
};
// A lane of an MFMA's query operand holds elements 32 s + 8 g + j of head row n in r[s][j]: the sum of squares over the row in the order
// of RopeHead (chains of the elements 64 apart, then lanes 32, 16, 8, 4, 2, 1 apart, of which the first and the last three are this
// lane's own elements here): the same bits.
template <int KS>
__device__ __forceinline__ float attn_row_squares(const float (&r)[KS][8]) {
    float t[8];
#pragma unroll
    for (int j = 0; j < 8; j++) {
        float c0 = r[0][j] * r[0][j], c1 = r[1][j] * r[1][j];
#pragma unroll
        for (int k = 1; k < KS / 2; k++) {
            c0 = __builtin_fmaf(r[2 * k][j], r[2 * k][j], c0);
            c1 = __builtin_fmaf(r[2 * k + 1][j], r[2 * k + 1][j], c1);
        }
        if constexpr (KS == 2) asm volatile("" : "+v"(c0), "+v"(c1));  // (a product and a sum, two roundings: the sum there crosses lanes)
        t[j] = c0 + c1;
    }
    // (elements 16 apart are lanes 32 apart, elements 8 apart lanes 16 apart; j ^ 1 then sits in the other half of the wave, j ^ 2 in
    // the other half of that)
    float u[4], w[2];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        dfl_swap32(t[2 * i], t[2 * i + 1]);
        u[i] = t[2 * i] + t[2 * i + 1];
    }
#pragma unroll
    for (int i = 0; i < 2; i++) {
        dfl_swap16(u[2 * i], u[2 * i + 1]);
        w[i] = u[2 * i] + u[2 * i + 1];
    }
    float v = w[0] + w[1], a = v, b = v;
    dfl_swap16(a, b);
    v = a + b;
    a = v, b = v;
    dfl_swap32(a, b);
    return a + b;
}
// ... and its norm and rotation: tab(c), w(c) are the 16-byte chunk c of the row's cosines and sines, and of the weights; put(s, j, value).
template <int KS, typename Tab, typename W, typename Put>
__device__ __forceinline__ void attn_rotate(const float (&r)[KS][8], int g, float eps, Tab tab, W w, Put put) {
    constexpr int kHalf = 4 * KS;  // chunks of half a head
    const float by = dfl_head_scale<32 * KS>(attn_row_squares<KS>(r), eps);
#pragma unroll
    for (int s = 0; s < KS / 2; s++)
#pragma unroll
        for (int e = 0; e < 2; e++) {
            const int c = 8 * s + 2 * g + e;
            const float4_t cs = tab(c), sn = tab(kHalf + c), wa = w(c), wb = w(kHalf + c);
#pragma unroll
            for (int i = 0; i < 4; i++) {
                float ra, rb;
                dfl_rope_pair(r[s][4 * e + i] * by * wa[i], r[s + KS / 2][4 * e + i] * by * wb[i], sn[i], cs[i], ra, rb);
                put(s, 4 * e + i, ra);
                put(s + KS / 2, 4 * e + i, rb);
            }
        }
}
// The wave that makes the block's keys (values: VALUES) of one KV head: row: this lane's row of that head, table and weights in memory;
// tiles: the ring; cache: key 0 of the split (null: another workgroup writes it).  Keeps the other waves' barriers.
template <int HD, bool VALUES>
__device__ __forceinline__ void attn_new_rows(const float *__restrict__ row, const float *__restrict__ table, const float *__restrict__ w, float eps,
                                              int n_rows, int first_new, int n_keys, int n_steps, half8_t *ring, _Float16 *cache, int64_t stride) {
    constexpr int KS = HD / 32, CH = HD / 8, kKPieces = 32 * CH;
    const int lane = threadIdx.x & 63, n = lane & 15, g = lane >> 4;
    float r[KS][8];
#pragma unroll
    for (int s = 0; s < KS; s++)
#pragma unroll
        for (int e = 0; e < 2; e++) {
            const float4_t x = *reinterpret_cast<const float4_t *>(row + 32 * s + 8 * g + 4 * e);
#pragma unroll
            for (int i = 0; i < 4; i++) r[s][4 * e + i] = x[i];
        }
    __builtin_amdgcn_s_barrier();  // (the others': what they asked for ahead of the stages is there)
    half8_t out[KS];
    if constexpr (VALUES) {
#pragma unroll
        for (int s = 0; s < KS; s++)
#pragma unroll
            for (int j = 0; j < 8; j++) out[s][j] = static_cast<_Float16>(r[s][j]);
    } else {
        // (asked for along with the row, in one trip to memory)
        const float4_t *t = reinterpret_cast<const float4_t *>(table) + min(n, n_rows - 1) * (HD / 4), *wt = reinterpret_cast<const float4_t *>(w);
        float4_t tv[2 * KS], wv[2 * KS];
#pragma unroll
        for (int i = 0; i < 2 * KS; i++) tv[i] = t[8 * (i >> 1) + 2 * g + (i & 1)];
#pragma unroll
        for (int i = 0; i < 2 * KS; i++) wv[i] = wt[8 * (i >> 1) + 2 * g + (i & 1)];
#pragma unroll
        for (int i = 0; i < 2 * KS; i++) asm volatile("" : "+v"(tv[i]), "+v"(wv[i]));
        attn_rotate<KS>(r, g, eps, [&](int c) { return tv[(c - 2 * g) / 8 * 2 + (c - 2 * g) % 8]; },
                        [&](int c) { return wv[(c - 2 * g) / 8 * 2 + (c - 2 * g) % 8]; }, [&](int s, int j, float v) { out[s][j] = static_cast<_Float16>(v); });
    }
    const int at = first_new + n;  // this row's key
    const bool mine = n < n_rows && at >= 0 && at < n_keys;
    for (int st = 0; st < n_steps; st++) {
        __builtin_amdgcn_s_barrier();
        if (32 * st + 31 < first_new) continue;
        asm volatile("" ::: "memory");
        half8_t *kt = ring + (st % kAttnBufs) * (2 * kKPieces);
        const int key = at - 32 * st;
        if (mine && key >= 0 && key < 32) {
#pragma unroll
            for (int s = 0; s < KS; s++) {
                if constexpr (VALUES) {
                    _Float16 *vt = reinterpret_cast<_Float16 *>(kt + kKPieces);
#pragma unroll
                    for (int j = 0; j < 8; j++) {
                        const int d = 32 * s + 8 * g + j;
                        vt[(d * 4 + ((key >> 3) ^ attn_swz_v(d))) * 8 + (key & 7)] = out[s][j];
                    }
                } else {
                    kt[key * CH + ((4 * s + g) ^ attn_swz<CH>(key))] = out[s];
                }
            }
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
    }
    if (cache && mine) {
#pragma unroll
        for (int s = 0; s < KS; s++) {
            if constexpr (VALUES) {
#pragma unroll
                for (int j = 0; j < 8; j++) cache[(32 * s + 8 * g + j) * stride + at] = out[s][j];
            } else {
                *reinterpret_cast<half8_t *>(cache + at * stride + 32 * s + 8 * g) = out[s];
            }
        }
    }
}

// One workgroup = one KV head x one contiguous chunk of keys; wave w = query head w of the GQA
// group.  Stage = 32 keys: the K tile [32 keys][HD] and the V^T tile [HD dims][32 keys] are copied
// global -> LDS with direct-to-LDS loads into a ring of kAttnBufs buffers, so the whole group
// shares one copy and the loads of the next stages are in flight while one is consumed.
// MAXW = most waves a workgroup may have; it sets the register budget.
// MAXL: most loads a wave issues per stage (2 HD / 16 / waves, rounded up to a power of two).
// What bounds it is a stage's chain, not its bytes: loads landed, barrier, K fragments, two chains of MFMAs, the
// maximum over the row's lanes, the exponentials, the second product.  So the scores of stage t + 1 are computed ahead
// of the softmax of stage t (the matrix cores work under the exponentials), V fragments are asked for ahead of
// them, the maximum crosses the lanes without LDS, the last stage's special cases stand outside of the others' code, and
// a load's address is made of one lane part and one uniform part: 16 rows x 100 k keys, 48 / 8 heads of 128, with the
// merge: 105.9 -> 98.3 us, both trees in turn (4.2 TB/s of keys and values; a copy reaches 5.03).
// MERGE: the workgroup takes all of its rows' keys, split by split, and merges the splits as it goes (see
// attn_rows_kernel); else one split, whose partial result it writes.
template <int HD, typename TQ, int MAXW, int MAXL, bool MERGE, bool ROPE>
__device__ __forceinline__ void attn_body(const TQ *__restrict__ q, const _Float16 *__restrict__ k_cache,
                                          const _Float16 *__restrict__ vt_cache, float *__restrict__ part_o, float *__restrict__ part_ml,
                                          int64_t ctx_len, const int32_t *__restrict__ ctx_len_dev, int n_rows_total, int n_kv, int group, int n_waves,
                                          int64_t vt_stride, int want, int min_chunk, float scale, int full_block, int64_t window,
                                          int split_stride, int64_t part_slots, int block, float *__restrict__ out, void *__restrict__ out_xf,
                                          int out_xf_kind, size_t xf_stride, AttnRope rope = {}) {
    static_assert(!(MERGE && ROPE) && (!ROPE || sizeof(TQ) == 4), "a lone block's f32 rows");
    const int n_q = n_kv * group;
    // block: which block of sixteen query rows (a prefill group hands over many: block b's rows follow block
    // b - 1's in q and in the cache, its partial tiles sit part_slots slots further on)
    const int n_rows = min(16, n_rows_total - 16 * block);
    q += static_cast<int64_t>(block) * 16 * n_q * HD;
    constexpr int KS = HD / 32;       // k-steps of the score product
    constexpr int DT = HD / 16;       // 16-dim tiles of the output
    constexpr int CH = HD / 8;        // 16-byte chunks per key row
    constexpr int kKPieces = 32 * CH; // pieces of the K tile; the V^T tile has as many
    constexpr int kWaveLoads = 2 * kKPieces / 64;
    static_assert(HD < 256 || MAXW <= 8, "sixteen waves leave a wave 128 registers");
    extern __shared__ half8_t lds[];  // kAttnBufs x (K tile, V^T tile)
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int n = lane & 15, g = lane >> 4;
    const int kvh = blockIdx.y;
    // blockIdx.x = split + split_stride * (part of the GQA group this workgroup serves); split_stride is a multiple
    // of 8, so the workgroups that read one chunk of keys are dispatched to the same XCD and share its L2 copy
    const int split = MERGE ? 0 : blockIdx.x % split_stride;
    if constexpr (ROPE) {
        if (wave >= n_waves) {
            const int64_t from = split * static_cast<int64_t>(min_chunk), to = min(ctx_len + n_rows, from + min_chunk);
            if (to <= ctx_len || from >= to) return;
            const bool values = wave > n_waves;
            const float *row = reinterpret_cast<const float *>(q) + (static_cast<int64_t>(min(n, n_rows - 1)) * (n_q + 2 * n_kv) + n_q + (values ? n_kv : 0) + kvh) * HD;
            const int first = static_cast<int>(ctx_len - from), keys = static_cast<int>(to - from), steps = (keys + 31) / 32;
            const bool writes = static_cast<int>(blockIdx.x) < split_stride;
            if (values)
                attn_new_rows<HD, true>(row, nullptr, nullptr, 0.0f, n_rows, first, keys, steps, lds,
                                        writes ? const_cast<_Float16 *>(vt_cache) + static_cast<int64_t>(kvh) * HD * vt_stride + from : nullptr, vt_stride);
            else
                attn_new_rows<HD, false>(row, rope.table, rope.k_w, rope.eps, n_rows, first, keys, steps, lds,
                                         writes ? const_cast<_Float16 *>(k_cache) + (from * n_kv + kvh) * HD : nullptr, static_cast<int64_t>(n_kv) * HD);
            return;
        }
    }
    const int head = kvh * group + (MERGE ? blockIdx.x : blockIdx.x / split_stride) * n_waves + wave;  // this wave's query head
    // Q^T fragments: lane (row n, g) holds Q[n][head][32 s + 8 g ..+8]
    // (rows at or past n_rows repeat the last row: they are never stored)
    AttnQ8<TQ> q_raw[KS];
    const int64_t q_heads = ROPE ? n_q + 2 * n_kv : n_q;  // heads from one row to the next
    const TQ *qrow = q + (static_cast<int64_t>(min(n, n_rows - 1)) * q_heads + head) * HD + 8 * g;
    attn_load_q<0, KS>(q_raw, qrow);
    if (ctx_len < 0) ctx_len = *ctx_len_dev;
    ctx_len += 16 * static_cast<int64_t>(block);
    const int64_t n_pos = ctx_len + n_rows;
    const int64_t chunk = want ? attn_chunk(n_pos, want, min_chunk) : min_chunk;
    if (!MERGE && split * chunk >= n_pos) return;  // the grid is sized for the longest context
    const int64_t c0 = MERGE ? 0 : split * chunk;
    const int64_t c1 = MERGE ? n_pos : min(n_pos, c0 + chunk);
    const int n_steps = static_cast<int>((c1 - c0 + 31) / 32);
    const int64_t kv_dim = static_cast<int64_t>(n_kv) * HD;
    const int per_wave = (kWaveLoads + n_waves - 1) / n_waves;  // loads each wave issues per stage
    ATT_TR(0);

    // Stage `st` (keys c0 + 32 st ..) into ring buffer st % kAttnBufs: wave-load qd covers LDS pieces
    // 64 qd ..; this wave takes qd = j n_waves + wave, and loads past the end repeat earlier ones
    // (same bytes to the same place) so that every wave issues per_wave loads.  Key rows at or past
    // n_pos are never dereferenced: the last stage of the cache re-reads row n_pos - 1 instead (its
    // scores are masked and its V columns zeroed below).
    const uint8_t *ksrc = reinterpret_cast<const uint8_t *>(k_cache + static_cast<int64_t>(kvh) * HD) + c0 * kv_dim * 2;
    const uint8_t *vsrc = reinterpret_cast<const uint8_t *>(vt_cache + static_cast<int64_t>(kvh) * HD * vt_stride) + c0 * 2;
    // A wave-load is 64 / CH key rows or sixteen dims of V^T: the first row is the uniform part of its address, and the
    // lane's part is the same for every load but for the swizzle, whose bits of the first row are one more xor.
    constexpr int kRowsPerLoad = 64 / CH;
    const int sub = lane / CH;
    const uint32_t k_row = static_cast<uint32_t>(sub) * static_cast<uint32_t>(kv_dim) * 2, k_chunk = ((lane % CH) ^ attn_swz<CH>(sub)) * 16;
    const uint32_t v_off = static_cast<uint32_t>(lane >> 2) * static_cast<uint32_t>(vt_stride) * 2 + 16 * ((lane & 3) ^ attn_swz_v(lane >> 2));
    int issued = 0;
    auto issue_stage = [&]() {
        half8_t *buf = lds + (issued % kAttnBufs) * (2 * kKPieces);
        const int rows_left = static_cast<int>(min(n_pos - c0 - 32ll * issued, static_cast<int64_t>(32)));
        int qd = wave;
        if constexpr (MAXL > 8) asm volatile("" : "+s"(qd));  // (so many addresses are made anew per stage, not kept in registers)
#pragma unroll
        for (int j = 0; j < MAXL; j++) {
            if (j >= per_wave) break;
            if (qd >= kWaveLoads) qd -= kWaveLoads;
            const uint8_t *src;
            if (qd * 64 < kKPieces) {
                const int row0 = qd * kRowsPerLoad;
                uint32_t o = k_row + (k_chunk ^ static_cast<uint32_t>(attn_swz<CH>(row0) * 16));
                if (rows_left < 32) o -= static_cast<uint32_t>(max(row0 + sub - (rows_left - 1), 0)) * static_cast<uint32_t>(kv_dim) * 2;
                src = ksrc + static_cast<int64_t>(row0) * kv_dim * 2 + static_cast<int32_t>(o);
            } else {
                src = vsrc + static_cast<int64_t>((qd * 64 - kKPieces) >> 2) * vt_stride * 2 + v_off;
            }
            __builtin_amdgcn_global_load_lds((gptr_t)(src), (lptr_t)(buf + qd * 64), 16, 0, 0);
            qd += n_waves;
        }
        ksrc += 64 * kv_dim;
        vsrc += 64;
        issued++;
    };

    // ROPE: the norm's weights (a KB) and the table in the place of the last buffer.  The table's 16-byte chunk c of row r sits at c ^ r:
    // sixteen lanes read the sixteen rows' at once.
    constexpr int RP = HD / 4;  // chunks of a row of the table
    static_assert(!ROPE || 64 + 16 * RP <= 2 * kKPieces, "the ring's last buffer holds the table");
    half8_t *const raw_w = lds + (kAttnBufs - 1) * (2 * kKPieces), *const raw_tab = raw_w + 64;
    const bool has_rows = ROPE && c1 > ctx_len;
    const int first_new = ROPE ? static_cast<int>(min(ctx_len - c0, static_cast<int64_t>(0x3fffffff))) : 0;  // where the block's first key lies, relative to c0
    if constexpr (ROPE) {
        const int row_loads = (n_rows * RP + 63) / 64;
        for (int i = wave; i < row_loads + 1; i += n_waves) {
            const int p = 64 * i + lane, r = min(p / RP, n_rows - 1);
            const float *src = i < row_loads ? rope.table + r * HD + 4 * ((p % RP) ^ r) : rope.q_w + 4 * (lane % RP);
            __builtin_amdgcn_global_load_lds((gptr_t)(src), (lptr_t)(i < row_loads ? raw_tab + 64 * i : raw_w), 16, 0, 0);
        }
    }

    // prologue: kAttnBufs - 1 stages in flight
#pragma unroll
    for (int st = 0; st < kAttnBufs - 1; st++)
        if (issued < n_steps) issue_stage();
    if constexpr (!MERGE) {
        dfl_have(scale, full_block, window, part_o, part_ml);
        if (block) {
            part_o += static_cast<int64_t>(block) * part_slots * HD;
            part_ml += static_cast<int64_t>(block) * part_slots * 2;
        }
    }

    ATT_TR(1);
    half8_t qf[KS];  // Q^T, times scale * log2(e)
    {
        const float mult = scale * kLog2e;
        attn_wait(per_wave * issued);
        if constexpr (!ROPE) {
#pragma unroll
            for (int s = 0; s < KS; s++) {
                q_raw[s].arrived();
#pragma unroll
                for (int i = 0; i < 8; i++) qf[s][i] = static_cast<_Float16>(q_raw[s].get(i) * mult);
            }
        } else {
            float r[KS][8];
#pragma unroll
            for (int s = 0; s < KS; s++) {
                q_raw[s].arrived();
#pragma unroll
                for (int i = 0; i < 8; i++) r[s][i] = q_raw[s].get(i);
            }
            asm volatile("" ::: "memory");
            __builtin_amdgcn_s_barrier();  // what all waves asked for is there
            asm volatile("" ::: "memory");
            const int row = min(n, n_rows - 1);
            const float4_t *tab = reinterpret_cast<const float4_t *>(raw_tab) + row * RP, *wt = reinterpret_cast<const float4_t *>(raw_w);
            attn_rotate<KS>(r, g, rope.eps, [&](int c) { return tab[c ^ row]; }, [&](int c) { return wt[c]; },
                            [&](int s, int j, float v) { qf[s][j] = static_cast<_Float16>(v * mult); });
        }
    }

    ATT_TR(2);
    float4_t acc[DT];
#pragma unroll
    for (int t = 0; t < DT; t++) acc[t] = float4_t{0, 0, 0, 0};
    float m_run = -INFINITY, l_run = 0.0f;  // running maximum of row n (base-2 logits, shared by its four lanes); this lane's share of the row sum
    // visible keys of row n, relative to c0: [lo, hi].  Block-causal: everything up to the row's own
    // position; full_block (drafter, non-causal): the whole block; a window keeps |distance| < window.
    auto row_range = [&](int row, int &lo, int &hi) {
        const int64_t row_pos = ctx_len + row;
        int64_t hi64 = full_block ? n_pos - 1 : row_pos;
        int64_t lo64 = 0;
        if (window > 0) {
            lo64 = row_pos - window + 1;
            hi64 = min(hi64, row_pos + window - 1);
        }
        hi64 = min(hi64, c1 - 1);
        hi = static_cast<int>(max(min(hi64 - c0, static_cast<int64_t>(0x3fffffff)), static_cast<int64_t>(-1)));
        lo = static_cast<int>(max(min(lo64 - c0, static_cast<int64_t>(0x3fffffff)), static_cast<int64_t>(0)));
    };
    int row_lo, row_hi, all_lo, all_hi, unused;
    row_range(n, row_lo, row_hi);
    // steps whose 32 keys are visible to every row need no masking: [all_lo, all_hi] in keys (both bounds grow with the row)
    row_range(0, unused, all_hi);
    row_range(15, all_lo, unused);

    const int rk0 = 8 * (n >> 2) + (n & 3);  // key row of S^T tile 0 this lane's A operand reads
    auto scores = [&](int st, float4_t (&sc)[2]) {
        const half8_t *kt = lds + (st % kAttnBufs) * (2 * kKPieces);
#pragma unroll
        for (int T = 0; T < 2; T++) {
            const int r = rk0 + 4 * T, sw = attn_swz<CH>(r);
            sc[T] = float4_t{0, 0, 0, 0};
#pragma unroll
            for (int s = 0; s < KS; s++) sc[T] = __builtin_amdgcn_mfma_f32_16x16x32_f16(kt[r * CH + ((4 * s + g) ^ sw)], qf[s], sc[T], 0, 0, 0);
        }
    };
    // stage `st` is in LDS for everyone; every wave is done with stage st - 2
    auto landed = [&](int st) {
        attn_wait(per_wave * (issued - 1 - st));
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        if constexpr (ROPE) {
            if (!has_rows || 32 * st + 31 < first_new) return;
            __builtin_amdgcn_s_barrier();  // the block's own rows are over what the cache still holds there
            asm volatile("" ::: "memory");
        }
    };
    // MERGE: what the splits so far come to; the split at hand ends ahead of stage split_end
    float4_t tot[MERGE ? DT : 1];
    float m_tot = -INFINITY, l_tot = 0.0f;
    const int chunk_steps = static_cast<int>(min(chunk / 32, static_cast<int64_t>(0x3fffffff)));
    int split_end = chunk_steps;
    bool split_begins = true;
    if constexpr (MERGE)
#pragma unroll
        for (int t = 0; t < DT; t++) tot[t] = float4_t{0, 0, 0, 0};
    float4_t sc[2], sc_next[2];
    landed(0);
    scores(0, sc);
    for (int st = 0; st < n_steps; st++) {
        const half8_t *vt = lds + (st % kAttnBufs) * (2 * kKPieces) + kKPieces;
        const int key0 = 32 * st;  // relative to c0
        if (st + 1 < n_steps) {
            landed(st + 1);
            if (issued < n_steps) issue_stage();  // into the buffer of stage st - 1
            scores(st + 1, sc_next);
        }
        half8_t vf[DT];
#pragma unroll
        for (int t = 0; t < DT; t++) vf[t] = vt[(16 * t + n) * 4 + (g ^ attn_swz_v(n))];
        const bool masked = !(key0 >= all_lo && key0 + 31 <= all_hi);  // uniform: some key of this step is hidden from some row
        float p[8];
#pragma unroll
        for (int i = 0; i < 8; i++) p[i] = (i < 4) ? sc[0][i] : sc[1][i - 4];
        if (masked) {
#pragma unroll
            for (int i = 0; i < 8; i++) {
                const int key = key0 + 8 * g + i;
                p[i] = (key >= row_lo && key <= row_hi) ? p[i] : -INFINITY;
            }
        }
        float mx = fmaxf(fmaxf(fmaxf(p[0], p[1]), fmaxf(p[2], p[3])), fmaxf(fmaxf(p[4], p[5]), fmaxf(p[6], p[7])));
        mx = dfl_max_far(mx);
        const float m_new = fmaxf(m_run, mx);
        // all keys of this step masked for this row and nothing seen before: keep the state
        const float m_safe = (m_new == -INFINITY) ? 0.0f : m_new;
        const float alpha = __builtin_amdgcn_exp2f(m_run - m_safe);  // 0 when m_run = -inf
        float psum = 0.0f;
#pragma unroll
        for (int i = 0; i < 8; i++) {
            p[i] = __builtin_amdgcn_exp2f(p[i] - m_safe);
            psum += p[i];
        }
        l_run = __builtin_fmaf(l_run, alpha, psum);
        if (!(MERGE && split_begins) && __builtin_amdgcn_ballot_w64(alpha != 1.0f) != 0) {
#pragma unroll
            for (int t = 0; t < DT; t++) acc[t] *= alpha;
        }
        m_run = m_new;
        half8_t pf;
#pragma unroll
        for (int i = 0; i < 8; i++) pf[i] = static_cast<_Float16>(p[i]);
        // O^T tile t (dims 16 t ..): A = V^T[dim 16 t + n][keys key0 + 8 g ..+8].  Columns at or past
        // n_pos hold whatever the cache held before (possibly NaN patterns; 0 * NaN would poison
        // the accumulator): zero them in the last stage of the cache
        if (c0 + key0 + 32 > n_pos) {
            const int vkeys = static_cast<int>(n_pos - (c0 + key0)) - 8 * g;  // this lane's columns ahead of n_pos
#pragma unroll
            for (int t = 0; t < DT; t++)
#pragma unroll
                for (int i = 0; i < 8; i++)
                    if (i >= vkeys) vf[t][i] = static_cast<_Float16>(0.0f);
        }
        if (MERGE && split_begins) {  // (as from an accumulator of zeros)
#pragma unroll
            for (int t = 0; t < DT; t++) acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(vf[t], pf, float4_t{0, 0, 0, 0}, 0, 0, 0);
        } else {
#pragma unroll
            for (int t = 0; t < DT; t++) acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(vf[t], pf, acc[t], 0, 0, 0);
        }
        if constexpr (MERGE) {
            split_begins = st + 1 == split_end || st + 1 == n_steps;
            if (split_begins) {
                float l = l_run;
                l += xor_lane(l, 16);
                l += xor_lane(l, 32);
                const AttnMerge w(m_tot, m_run);
                l_tot = w.add(l_tot, l);
                if (__builtin_amdgcn_ballot_w64(w.old != 1.0f) != 0) {
#pragma unroll
                    for (int t = 0; t < DT; t++) tot[t] *= w.old;
                }
#pragma unroll
                for (int t = 0; t < DT; t++)
#pragma unroll
                    for (int i = 0; i < 4; i++) tot[t][i] = __builtin_fmaf(w.next, acc[t][i], tot[t][i]);
                m_tot = w.m;
                m_run = -INFINITY;
                l_run = 0.0f;
                split_end += chunk_steps;
            }
        }
        sc[0] = sc_next[0];
        sc[1] = sc_next[1];
        if (st < 8) ATT_TR(3 + st);
    }
    ATT_TR(12);
    if constexpr (MERGE) {
        float *o = out + ((static_cast<int64_t>(block) * 16 + n) * n_q + head) * HD;
#pragma unroll
        for (int t = 0; t < DT; t++) {
            tot[t] /= l_tot;
            if (n < n_rows) *reinterpret_cast<float4_t *>(o + 16 * t + 4 * g) = tot[t];
        }
        if (out_xf) {
            out_xf = static_cast<uint8_t *>(out_xf) + block * xf_stride;
            attn_store_xf<DT>(tot, out_xf, out_xf_kind, n, g, head * HD, n < n_rows);
        }
        return;
    }
    // row sums over the four lanes of a row; partials: O^T tile t, lane (row n, g) holds dims 16 t + 4 g + i
    float l = l_run;
    l += xor_lane(l, 16);
    l += xor_lane(l, 32);
    if (n < n_rows) {
        const int64_t slot = (static_cast<int64_t>(split) * n_q + head) * 16 + n;
        float *po = part_o + slot * HD;
#pragma unroll
        for (int t = 0; t < DT; t++) *reinterpret_cast<float4_t *>(po + 16 * t + 4 * g) = acc[t];
        if (g == 0) {
            part_ml[slot * 2] = m_run;
            part_ml[slot * 2 + 1] = l;
        }
    }
    ATT_TR(13);
}

template <int HD, typename TQ, int MAXW, int MAXL>
__global__ void __launch_bounds__(64 * MAXW)
    attn_split_kernel(const TQ *__restrict__ q, const _Float16 *__restrict__ k_cache, const _Float16 *__restrict__ vt_cache, int64_t ctx_len,
                      int64_t vt_stride, uint32_t heads, uint32_t split_waves, int n_rows_total, int min_chunk, int want, float scale,
                      float *__restrict__ part_o, float *__restrict__ part_ml, int full_block, int64_t window, int64_t part_slots,
                      const int32_t *__restrict__ ctx_len_dev) {
    // The arguments in the order of their use: the first fourteen words, which the first loads need, come preloaded with the wave.
    // heads = KV heads | group << 20, split_waves = split_stride | waves << 24; ctx_len < 0: it is in device memory; want == 0: min_chunk is the chunk.
    attn_body<HD, TQ, MAXW, MAXL, false, false>(q, k_cache, vt_cache, part_o, part_ml, ctx_len, ctx_len_dev, n_rows_total, heads & 0xfffff, heads >> 20,
                                         split_waves >> 24, vt_stride, want, min_chunk, scale, full_block, window, split_waves & 0xffffff, part_slots,
                                         blockIdx.z, nullptr, nullptr, 0, 0);
}

// A lone block whose rows are as the projections left them: see AttnRope.  heads: the rows, less one | query heads a KV head << 4 | KV heads << 9;
// split_waves: split_stride | heads a workgroup << 11 | the chunk, in stages << 16.  (All the first loads need comes preloaded with the wave.)
template <int HD, int MAXL>
__global__ void __launch_bounds__(HD == 256 ? 512 : 640)
    attn_split_rope_kernel(const float *__restrict__ rows, _Float16 *k_cache, _Float16 *vt_cache, const float *__restrict__ table,
                           const float *__restrict__ q_w, uint32_t heads, uint32_t split_waves, int ctx_len, int vt_stride, const float *__restrict__ k_w, float eps, float scale, float *__restrict__ part_o, float *__restrict__ part_ml, int full_block, int64_t window) {
    attn_body<HD, float, 8, MAXL, false, true>(rows, k_cache, vt_cache, part_o, part_ml, ctx_len, nullptr, (heads & 15) + 1, heads >> 9, heads >> 4 & 31,
                                                  split_waves >> 11 & 31, vt_stride, 0, 32 * (split_waves >> 16), scale, full_block, window, split_waves & 0x7ff, 0, 0, nullptr,
                                                  nullptr, 0, 0, AttnRope{table, q_w, k_w, eps});
}

// Many blocks of rows at once, a prompt's prefill: the blocks are enough workgroups, so one takes all of its block's keys
// and the partial results never leave its registers.  The splits stay (a block's own policy: want and min_chunk of the
// run of blocks it belongs to) as the points where the running result is merged, in the order and with the
// arithmetic of attn_combine_ordered_kernel: the same bits as the block on its own.  Blocks of one launch differ in their
// keys: the longest go first.  Bound by a stage's chain, as the split kernel (1.3 us a stage with two workgroups on a CU):
// 1000 rows of 32 / 8 heads of 128, the first to the last: 153 us as splits and their merges, 42 us here.  (Two blocks per
// workgroup, sharing its keys and values: 50 us; the bytes are not what bounds it.)
constexpr int kAttnRuns = 16;
struct AttnRuns {
    int n, first[kAttnRuns], want[kAttnRuns], min_chunk[kAttnRuns];
};
template <int HD, int MAXL>
__global__ void __launch_bounds__(512)
    attn_rows_kernel(const float *__restrict__ q, const _Float16 *__restrict__ k_cache, const _Float16 *__restrict__ vt_cache, int64_t ctx_len,
                     int n_rows_total, int n_q, int n_kv, int64_t vt_stride, AttnRuns runs, float scale, float *__restrict__ out,
                     void *__restrict__ out_xf, int out_xf_kind, size_t xf_stride) {
    const int block = gridDim.z - 1 - blockIdx.z;
    int want = runs.want[0], min_chunk = runs.min_chunk[0];
    for (int r = 1; r < runs.n && runs.first[r] <= block; r++) {
        want = runs.want[r];
        min_chunk = runs.min_chunk[r];
    }
    attn_body<HD, float, 8, MAXL, true, false>(q, k_cache, vt_cache, nullptr, nullptr, ctx_len, nullptr, n_rows_total, n_kv, n_q / n_kv, blockDim.x >> 6, vt_stride, want, min_chunk,
                                        scale, 0, 0, 1, 0, block, out, out_xf, out_xf_kind, xf_stride);
}

// The same for heads of 256, whose splits are merged by attn_combine_few_kernel: every eighth split after the other, times
// 2^(m_s - m*), then the eight sums in turn.  That order asks for the maximum m* over all splits ahead of the first sum: the keys
// are walked twice, the first time for the scores' maxima alone, the second time split by split in the merge's order.
// Splits are of 64 keys, two stages (the host's rule): both stages' probabilities are there before the first value is
// multiplied, so that a tile of 16 dims goes through its two products, the rescale between them and the merge in four
// registers, and beside the queries a lane keeps one sum.
// LDS: three 64-key tiles of K for the first walk; for the second two splits of K and V, the first of them behind the
// three tiles (it is asked for while the first walk ends), the other in the place of two of them.
// What bounds it: the chain of the longest block.  A wave's products (96 MFMAs a split) and vector work (250 instructions) stand mostly
// one behind the other, 3.4 us a split with eight busy waves, 2.6 to 3.2 with four; without the loads 7 % less, without the first walk's
// products 14 %, without the second walk's 47 %.  So a workgroup has four heads of a long block and of a short one, which
// share keys and values as far as the short one reaches, and the longest are mostly alone on their SIMDs: 2048 rows of 16 / 2 heads, where eight
// heads of one block are a CU's and the longest block's is the last to end, 147 -> 124 us.  As splits they are 425 us (286 MB of partial results
// out and as many back); 300 rows 36 -> 26 us.
// Not kept: the next split's scores under this one's softmax (151 -> 160 us, registers); a quarter of the keys for four heads a wave in the first
// walk, a quarter of its LDS reads, and a tile's second product behind the next tile's first (124 : 124 us).
constexpr int kPairSplit = 64, kPairKeys = 32 * 1024, kPairLds = 5 * kPairKeys;
__global__ void __launch_bounds__(512)
    attn_rows_pair_kernel(const float *__restrict__ q, const _Float16 *__restrict__ k_cache, const _Float16 *__restrict__ vt_cache, int64_t ctx_len,
                          int n_rows_total, int n_q, int n_kv, int64_t vt_stride, float scale, float *__restrict__ out, void *__restrict__ out_xf,
                          int out_xf_kind, size_t xf_stride, int heads) {
    constexpr int HD = 256, KS = HD / 32, DT = HD / 16, CH = HD / 8;
    extern __shared__ half8_t lds[];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), n_waves = blockDim.x >> 6;
    const int n = lane & 15, g = lane >> 4;
    // The longest blocks first.  Twice as many waves as heads: the second half of them has the block as far from the first as
    // this one from the last (none in the middle of an odd number), and goes along with this one's splits as far as its own reach.
    const int far = (n_rows_total + 15) / 16 - 1 - blockIdx.z, near = blockIdx.z;
    const bool second = wave >= heads;
    const int block = second ? near : far;
    const int n_all = static_cast<int>(ctx_len) + min(16 * far + 16, n_rows_total), all_splits = (n_all + kPairSplit - 1) / kPairSplit;
    const int n_rows = min(16, n_rows_total - 16 * block);
    ctx_len += 16 * static_cast<int64_t>(block);
    const int n_pos = static_cast<int>(ctx_len) + n_rows;
    const int kvh = blockIdx.y, head = kvh * (n_q / n_kv) + blockIdx.x * heads + (second ? wave - heads : wave);
    const int n_splits = second && near == far ? 0 : (n_pos + kPairSplit - 1) / kPairSplit;
    const int64_t kv_dim = static_cast<int64_t>(n_kv) * HD;
    const uint8_t *const k_base = reinterpret_cast<const uint8_t *>(k_cache + static_cast<int64_t>(kvh) * HD);
    const uint8_t *const v_base = reinterpret_cast<const uint8_t *>(vt_cache + static_cast<int64_t>(kvh) * HD * vt_stride);
    const uint32_t v_lane = static_cast<uint32_t>(lane >> 2) * static_cast<uint32_t>(vt_stride) * 2 + 16 * ((lane & 3) ^ attn_swz_v(lane >> 2));

    // A wave-load is 1 KB: two key rows, or 16 dims of 32 values.  32 of them are a split's keys, as many again its values; a
    // wave takes every n_waves-th, and where they do not come out even some load what another loads too.  With eight or
    // four waves the loads of a whole split differ by uniform strides and uniform bits of the swizzle.
    const uint32_t k_lane = static_cast<uint32_t>(2 * wave + (lane >> 5)) * static_cast<uint32_t>(kv_dim * 2) +
                            (((lane & 31) ^ attn_swz<CH>(2 * wave + (lane >> 5))) << 4);
    auto load = [&](int split, bool values, uint8_t *dst) {
        const int total = values ? 64 : 32, c0 = split * kPairSplit, last = n_all - 1 - c0;
        auto whole = [&](auto waves) {
            constexpr int NW = decltype(waves)::value;
            const uint8_t *k = k_base + c0 * kv_dim * 2, *v = v_base + static_cast<int64_t>(16 * wave) * vt_stride * 2 + 2 * static_cast<int64_t>(c0);
            uint8_t *to = dst + wave * 1024;
#pragma unroll
            for (int j = 0; j < 32 / NW; j++, to += NW * 1024)
                __builtin_amdgcn_global_load_lds((gptr_t)(k + j * 4 * NW * kv_dim + (k_lane ^ static_cast<uint32_t>(attn_swz<CH>(2 * NW * j & 31) << 4))), (lptr_t)(to),
                                                 16, 0, 0);
            if (values) {
#pragma unroll
                for (int j = 0; j < 32 / NW; j++, to += NW * 1024)
                    __builtin_amdgcn_global_load_lds((gptr_t)(v + (NW * j & 15) * 32 * vt_stride + (NW * j >> 4) * 64 + v_lane), (lptr_t)(to), 16, 0, 0);
            }
        };
        if (n_waves == 8 && last >= kPairSplit - 1) return whole(std::integral_constant<int, 8>());
        if (n_waves == 4 && last >= kPairSplit - 1) return whole(std::integral_constant<int, 4>());
        for (int i = wave; i < (total + n_waves - 1) / n_waves * n_waves; i += n_waves) {
            const int p = i < total ? i : i - total;
            const uint8_t *src;
            if (p < 32) {  // (rows past the last position are never dereferenced: the last one again, its scores are masked)
                const int row = 2 * p + (lane >> 5);
                src = k_base + c0 * kv_dim * 2 + static_cast<uint32_t>(min(row, last)) * static_cast<uint32_t>(kv_dim * 2) + (((lane & 31) ^ attn_swz<CH>(row & 31)) << 4);
            } else {  // (nor is a second stage past the last position: the first one again, its values are zeroed)
                const int stage = (p - 32) >> 4, key = c0 + (32 * stage <= last ? 32 * stage : 0);
                src = v_base + static_cast<int64_t>((p & 15) * 16) * vt_stride * 2 + 2 * static_cast<int64_t>(key) + v_lane;
            }
            __builtin_amdgcn_global_load_lds((gptr_t)(src), (lptr_t)(dst + p * 1024), 16, 0, 0);
        }
    };
    const int per_keys = (32 + n_waves - 1) / n_waves, per_split = (64 + n_waves - 1) / n_waves;
    auto landed = [&](int later) {
        attn_wait(later);
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    uint8_t *const lds_b = reinterpret_cast<uint8_t *>(lds);

    half8_t qf[KS];
    {
        const float mult = scale * kLog2e;
        const float *qrow = q + (static_cast<int64_t>(block) * 16 + min(n, n_rows - 1)) * n_q * HD + static_cast<int64_t>(head) * HD + 8 * g;
        AttnQ8<float> raw[KS];
        load(0, false, lds_b);
        if (all_splits > 1)
            load(1, false, lds_b + kPairKeys);
        else
            load(0, true, lds_b + 3 * kPairKeys);
        attn_load_q<0, KS>(raw, qrow);  // (behind the branches: no asm load is under way where the code branches)
        attn_wait(0);
#pragma unroll
        for (int s = 0; s < KS; s++) {
            raw[s].arrived();
#pragma unroll
            for (int i = 0; i < 8; i++) qf[s][i] = static_cast<_Float16>(raw[s].get(i) * mult);
        }
    }
    // A split's fragments, in the order of their use: K rows of step s of the four score tiles T (4 s + T), then V^T of the
    // two stages of the sixteen tiles of dims (32 + 2 t + st).  Each is read kRing uses ahead, the first of V under the softmax.
    // (K's swizzle permutes a lane's steps four by four: four addresses, the rest is in the offset.)
    constexpr int kRing = 8;
    const uint32_t lds0 = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((lptr_t)lds));
    const uint32_t k_at = lds0 + (8 * (n >> 2) + (n & 3)) * (CH * 16) + (g ^ (n & 3)) * 16, v_at = lds0 + kPairKeys + (4 * n + (g ^ attn_swz_v(n))) * 16;
    const uint32_t k_step[4] = {k_at + (n >> 2) * 64, k_at + ((n >> 2) ^ 1) * 64, k_at + ((n >> 2) ^ 2) * 64, k_at + ((n >> 2) ^ 3) * 64};
    half8_t ring[kRing];
    auto read = [&](auto i, uint32_t buf) {
        constexpr int I = decltype(i)::value;
        if constexpr (I < 4 * KS)
            ring[I % kRing] = lds_read<half8_t, (32 * (I >> 1 & 1) + 4 * (I & 1)) * CH * 16 + (I >> 4) * 256>(k_step[I >> 2 & 3] + buf);
        else
            ring[I % kRing] = lds_read<half8_t, ((I - 4 * KS) >> 1) * 1024 + (I & 1) * 16384>(v_at + buf);
    };
    // The scores of a split's two stages, base-2 logits: p[8 st + i] of key 32 st + 8 g + i.  masked: some are hidden from some row.
    auto scores = [&](auto masked, auto with_values, int split, uint32_t buf, float (&p)[16]) {
        constexpr int N = decltype(with_values)::value ? 4 * KS + 2 * DT : 4 * KS;
        float4_t sc[4];
        static_for<0, kRing>([&](auto i) { read(i, buf); });
        static_for<0, 4 * KS>([&](auto i) {
            constexpr int I = decltype(i)::value, T = I & 3, left = N - 1 - I;
            lds_arrived<(left < kRing - 1 ? left : kRing - 1)>(ring[I % kRing]);
            sc[T] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ring[I % kRing], qf[I >> 2], I < 4 ? float4_t{0, 0, 0, 0} : sc[T], 0, 0, 0);
            if constexpr (I + kRing < N) read(std::integral_constant<int, I + kRing>(), buf);
        });
        const int seen = static_cast<int>(ctx_len) + n - split * kPairSplit - 8 * g;
#pragma unroll
        for (int i = 0; i < 16; i++) {
            p[i] = sc[2 * (i >> 3) + ((i >> 2) & 1)][i & 3];
            if (decltype(masked)::value && 32 * (i >> 3) + (i & 7) > seen) p[i] = -INFINITY;
        }
    };
    // (a split that ends behind the block's first row is the only kind that hides a key from a row)
    auto edge = [&](int split) { return (split + 1) * kPairSplit - 1 > static_cast<int>(ctx_len); };

    // first walk: the maximum over every key a row sees
    float m_star = -INFINITY;
    for (int split = 0, buf = 0; split < all_splits; split++) {
        landed(split + 1 < all_splits ? per_keys : per_split);
        uint8_t *const free_buf = lds_b + (buf == 0 ? 2 : buf - 1) * kPairKeys;
        if (split + 2 < all_splits)
            load(split + 2, false, free_buf);
        else if (split + 2 == all_splits)
            load(0, true, lds_b + 3 * kPairKeys);
        auto maxima = [&](auto masked) {
            float p[16];
            scores(masked, std::false_type(), split, buf * kPairKeys, p);
#pragma unroll
            for (int i = 0; i < 16; i++) m_star = fmaxf(m_star, p[i]);
        };
        if (split < n_splits && edge(split))
            maxima(std::true_type());
        else if (split < n_splits)
            maxima(std::false_type());
        buf = buf == 2 ? 0 : buf + 1;
    }
    m_star = dfl_max_far(m_star);

    // second walk.  Up to eight splits are an eighth each: `sum` is the total.  Else it is an eighth's sum, and the total waits in
    // the block's output rows of this head, seven times there and back (the registers do not hold both): lane by lane, a
    // kilobyte a row, where all sixteen rows are there, else where it belongs.
    float *const o = out + ((static_cast<int64_t>(block) * 16 + n) * n_q + head) * HD + 4 * g;
    const bool live = n < n_rows, held = live || n_rows == 16;
    float *const wait_at = n_rows == 16 ? out + (static_cast<int64_t>(block) * 16 * n_q + head) * HD + 4 * lane : o;
    const int64_t wait_step = n_rows == 16 ? static_cast<int64_t>(n_q) * HD : 16;
    float4_t sum[DT];
#pragma unroll
    for (int t = 0; t < DT; t++) sum[t] = float4_t{0, 0, 0, 0};
    float l_sum = 0.0f, l_tot = 0.0f;
    const bool few = n_splits <= 8;
    for (int split = 0, at = 0, next; at < all_splits; at++, split = next) {
        const bool ends = split + 8 >= n_splits;  // the last of this one's eighth
        next = split + 8 >= all_splits ? (split & 7) + 1 : split + 8;
        landed(0);
        const uint32_t buf = at & 1 ? 0 : 3 * kPairKeys;
        if (at + 1 < all_splits) load(next, true, lds_b + (at & 1 ? 3 * kPairKeys : 0));
        auto merge = [&](auto masked, auto of_few) {
            constexpr bool kFew = decltype(of_few)::value;
            float p[16];
            scores(masked, std::true_type(), split, buf, p);
            // the two stages: running maximum, rescale of the first stage by the second's, row sum
            float mx[2];
#pragma unroll
            for (int st = 0; st < 2; st++) {
                const float *v = p + 8 * st;
                mx[st] = dfl_max_far(fmaxf(fmaxf(fmaxf(v[0], v[1]), fmaxf(v[2], v[3])), fmaxf(fmaxf(v[4], v[5]), fmaxf(v[6], v[7]))));
            }
            const float m1 = mx[0], m2 = fmaxf(m1, mx[1]);
            const float safe[2] = {m1 == -INFINITY ? 0.0f : m1, m2 == -INFINITY ? 0.0f : m2};
            const float alpha = __builtin_amdgcn_exp2f(m1 - safe[1]);
            half8_t pf[2];
            float ps[2] = {0.0f, 0.0f};
#pragma unroll
            for (int st = 0; st < 2; st++)
#pragma unroll
                for (int i = 0; i < 8; i++) {
                    const float e = __builtin_amdgcn_exp2f(p[8 * st + i] - safe[st]);
                    ps[st] += e;
                    pf[st][i] = static_cast<_Float16>(e);
                }
            // (over the row's four lanes: the lane 16 away, then the pair 32 away)
            float l = __builtin_fmaf(ps[0], alpha, ps[1]), l2 = l;
            dfl_swap16(l, l2);
            l += l2;
            l2 = l;
            dfl_swap32(l, l2);
            l += l2;
            const float w = m2 == -INFINITY ? 0.0f : exp2f(m2 - m_star);
            l_sum = kFew ? l_sum + __builtin_fmaf(w, l, 0.0f) : __builtin_fmaf(w, l, l_sum);
            const int left = n_pos - split * kPairSplit - 8 * g;  // this lane's columns ahead of n_pos
            float4_t a[DT];
            static_for<4 * KS, 4 * KS + 2 * DT>([&](auto i) {
                constexpr int I = decltype(i)::value, t = (I - 4 * KS) >> 1, st = I & 1, later = 4 * KS + 2 * DT - 1 - I;
                half8_t &v = ring[I % kRing];
                lds_arrived<(later < kRing - 1 ? later : kRing - 1)>(v);
                if constexpr (decltype(masked)::value) {  // (what the cache holds past n_pos may be NaN patterns)
#pragma unroll
                    for (int k = 0; k < 8; k++)
                        if (32 * st + k >= left) v[k] = static_cast<_Float16>(0.0f);
                }
                if constexpr (st == 0) {
                    a[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(v, pf[0], float4_t{0, 0, 0, 0}, 0, 0, 0);
                    a[t] *= alpha;
                } else {
                    a[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(v, pf[1], a[t], 0, 0, 0);
#pragma unroll
                    for (int k = 0; k < 4; k++) sum[t][k] = kFew ? sum[t][k] + __builtin_fmaf(w, a[t][k], 0.0f) : __builtin_fmaf(w, a[t][k], sum[t][k]);
                }
                if constexpr (I + kRing < 4 * KS + 2 * DT) read(std::integral_constant<int, I + kRing>(), buf);
            });
        };
        if (split >= n_splits) continue;
        if (few && edge(split))
            merge(std::true_type(), std::true_type());
        else if (few)
            merge(std::false_type(), std::true_type());
        else if (edge(split))
            merge(std::true_type(), std::false_type());
        else
            merge(std::false_type(), std::false_type());
        if (ends && !few) {
            l_tot += l_sum;
            float *at_row = wait_at;  // (opaque: sixteen addresses kept across the walk would not fit)
            asm volatile("" : "+v"(at_row));
            if (held && (split & 7) != 0) {
                float4_t v[DT];
                const float *p = at_row;
#pragma unroll
                for (int t = 0; t < DT; t++, p += wait_step) v[t] = *reinterpret_cast<const float4_t *>(p);
#pragma unroll
                for (int t = 0; t < DT; t++) sum[t] = v[t] + sum[t];
            }
            if ((split & 7) != 7) {
                l_sum = 0.0f;
#pragma unroll
                for (int t = 0; t < DT; t++, at_row += wait_step) {
                    if (held) *reinterpret_cast<float4_t *>(at_row) = sum[t];
                    sum[t] = float4_t{0, 0, 0, 0};
                }
            }
        }
    }
    if (n_splits == 0) return;
    if (few) l_tot = l_sum;
#pragma unroll
    for (int t = 0; t < DT; t++) {
        sum[t] /= l_tot;
        if (live) *reinterpret_cast<float4_t *>(o + 16 * t) = sum[t];
    }
    if (out_xf) attn_store_xf<DT>(sum, static_cast<uint8_t *>(out_xf) + block * xf_stride, out_xf_kind, n, g, head * HD, live);
}

#ifdef DFLASH_TRACE
}  // namespace
extern "C" void dflash_dbg_set_attn_trace(uint64_t p) {
    unsigned long long *v = reinterpret_cast<unsigned long long *>(p);
    (void)hipMemcpyToSymbol(HIP_SYMBOL(g_attn_trace), &v, sizeof(v));
}
namespace {
#endif

// out[row][head][:] = sum_s 2^(m_s - m*) O_s / sum_s 2^(m_s - m*) l_s
// One workgroup per (head, row): 256 threads = 8 split lanes x 32 dim lanes; a split lane adds up
// every eighth split (float4 per dim lane, all loads independent), then the eight are summed in LDS.
__global__ void __launch_bounds__(256)
    attn_combine_kernel(const float *__restrict__ part_o, const float *__restrict__ part_ml, float *__restrict__ out,
                        int n_rows_total, int n_q, int hd, int64_t ctx_len, const int32_t *__restrict__ ctx_len_dev, int want,
                        int min_chunk, void *__restrict__ out_xf, int out_xf_kind, int64_t part_slots, size_t xf_stride, int max_splits) {
    // blockIdx.z: which block of sixteen rows (see attn_split_kernel); rows past a short last block leave
    const int n_rows = min(16, n_rows_total - 16 * static_cast<int>(blockIdx.z));
    if (static_cast<int>(blockIdx.y) >= n_rows) return;
    part_o += static_cast<int64_t>(blockIdx.z) * part_slots * hd;
    part_ml += static_cast<int64_t>(blockIdx.z) * part_slots * 2;
    out += static_cast<int64_t>(blockIdx.z) * 16 * n_q * hd;
    if (out_xf) out_xf = static_cast<uint8_t *>(out_xf) + blockIdx.z * xf_stride;
    __shared__ float wgt[1024];          // 2^(m_s - m*) per split (n_splits <= 1024)
    __shared__ float red[8][256 + 4];    // partial outputs per split lane
    __shared__ float red_l[8];
    const int head = blockIdx.x, row = blockIdx.y;
    const int tid = threadIdx.x;
    const int64_t slot0 = static_cast<int64_t>(head) * 16 + row;
    const int64_t slot_stride = static_cast<int64_t>(n_q) * 16;
    // m* = max over splits (a thread keeps the maxima it loaded: n_splits <= 1024 = 4 per thread)
    float m_own[4];
#pragma unroll
    for (int j = 0; j < 4; j++) {
        m_own[j] = -INFINITY;
        if (256 * j >= max_splits) continue;
        const int s = tid + 256 * j;
        m_own[j] = s < max_splits ? part_ml[(slot0 + s * slot_stride) * 2] : -INFINITY;
    }
    // The partial outputs of the first kPre rounds of splits are asked for right behind the maxima, before those are
    // waited for: their addresses do not depend on the weights, so the two trips to memory are in flight together
    // instead of one behind the other across two barriers (the maxima first: loads return in the order of their issue,
    // and the maxima are what the first reduction needs).  The sums below take them in the order of the loop that follows.
    constexpr int kPre = 4;
    const int sl = tid >> 5, dl = tid & 31;  // split lane, dim lane
    const int n_vec = hd / 4;                // float4 per row: 16, 32 or 64
    float4_t pre0[kPre] = {}, pre1[kPre] = {};
    float pre_l[kPre] = {};
#pragma unroll
    for (int i = 0; i < kPre; i++) {
        if (8 * i >= max_splits) continue;  // (uniform; inside a round, lanes past the last split re-read it)
        const int64_t slot = slot0 + min(sl + 8 * i, max_splits - 1) * slot_stride;
        const float4_t *po = reinterpret_cast<const float4_t *>(part_o + slot * hd);
        pre0[i] = po[min(dl, n_vec - 1)];
        if (n_vec > 32) pre1[i] = po[min(dl + 32, n_vec - 1)];
        pre_l[i] = part_ml[slot * 2 + 1];
    }
    // how many splits there are: the context length may have to be read first, and nothing above waits for it
    if (ctx_len_dev) ctx_len = *ctx_len_dev;
    ctx_len += 16 * static_cast<int64_t>(blockIdx.z);
    const int n_splits = attn_splits(ctx_len + n_rows, want, min_chunk);
#pragma unroll
    for (int j = 0; j < 4; j++)
        if (tid + 256 * j >= n_splits) m_own[j] = -INFINITY;
    float m_loc = fmaxf(fmaxf(m_own[0], m_own[1]), fmaxf(m_own[2], m_own[3]));
    for (int off = 32; off > 0; off >>= 1) m_loc = fmaxf(m_loc, __shfl_xor(m_loc, off, 64));
    if ((tid & 63) == 0) red_l[tid >> 6] = m_loc;
    __syncthreads();
    const float m_star = fmaxf(fmaxf(red_l[0], red_l[1]), fmaxf(red_l[2], red_l[3]));
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const int s = tid + 256 * j;
        if (s < n_splits) wgt[s] = (m_own[j] == -INFINITY) ? 0.0f : exp2f(m_own[j] - m_star);
    }
    __syncthreads();  // (also: every thread has read red_l before the split lanes write their sums into it)
    float4_t acc0 = {0, 0, 0, 0}, acc1 = {0, 0, 0, 0};
    float l = 0.0f;
#pragma unroll
    for (int i = 0; i < kPre; i++) {
        const int s = sl + 8 * i;
        if (s < n_splits) {
            const float w = wgt[s];
            if (dl < n_vec) acc0 += w * pre0[i];
            if (dl + 32 < n_vec) acc1 += w * pre1[i];
            if (dl == 0) l += w * pre_l[i];
        }
    }
    for (int s = sl + 8 * kPre; s < n_splits; s += 8) {
        const float w = wgt[s];
        const float4_t *po = reinterpret_cast<const float4_t *>(part_o + (slot0 + s * slot_stride) * hd);
        if (dl < n_vec) acc0 += w * po[dl];
        if (dl + 32 < n_vec) acc1 += w * po[dl + 32];
        if (dl == 0) l += w * part_ml[(slot0 + s * slot_stride) * 2 + 1];
    }
#pragma unroll
    for (int i = 0; i < 4; i++) {
        red[sl][4 * dl + i] = acc0[i];
        red[sl][128 + 4 * dl + i] = acc1[i];
    }
    if (dl == 0) red_l[sl] = l;
    __syncthreads();
    float lsum = 0.0f;
#pragma unroll
    for (int k = 0; k < 8; k++) lsum += red_l[k];
    for (int d = tid; d < hd; d += 256) {
        float o = 0.0f;
#pragma unroll
        for (int k = 0; k < 8; k++) o += red[k][d];
        o /= lsum;
        out[(static_cast<int64_t>(row) * n_q + head) * hd + d] = o;
        if (out_xf) {
            // eight consecutive dims sit in eight consecutive lanes of one wave (hd is a multiple of 64)
            float v[8];
#pragma unroll
            for (int i = 0; i < 8; i++) v[i] = __shfl_down(o, i, 64);
            if ((d & 7) == 0) dfl_xf_store(out_xf, out_xf_kind, row, head * hd + d, v[0], v[1], v[2], v[3], v[4], v[5], v[6], v[7]);
        }
    }
}

// The same for at most 48 splits, with the same sums in the same order (a split lane's every eighth split, then the eight
// in turn).  What bounds it is its chain: a trip to memory for the maxima and the partial outputs, which are in flight
// together, the maximum over the splits, the sums.  Here lane s of every wave keeps split s's maximum and sum, so that the
// weights need no LDS and no barrier (a wave shuffles them to where they are used), and the only barrier stands between
// the split lanes' sums and their total: 5.1 -> 3.6 us inside a verify's graph (24 splits, 32 heads of 128, 16 rows).
// A wave's 64 lanes cover 64 / (HD / 4) split lanes, four dims per lane.
// kEights: eights of splits, by the launch's most.
template <int HD, int kEights>
__global__ void __launch_bounds__(HD == 64 ? 128 : 256)
    attn_combine_few_kernel(const float *__restrict__ part_o, const float *__restrict__ part_ml, int64_t ctx_len, int n_q, int n_rows_total, int max_splits,
                            int min_chunk, int want, float *__restrict__ out, void *__restrict__ out_xf, int out_xf_kind, int64_t part_slots,
                            size_t xf_stride, const int32_t *__restrict__ ctx_len_dev) {
    // (the arguments in the order of their use and with attn_split_kernel's conventions, but want == 0: min_chunk is the number of splits)
    constexpr int kLanes = HD / 4, kPerWave = 64 / kLanes, kWaves = HD == 64 ? 2 : 4, kSteps = 8 / (kPerWave * kWaves);
    const int n_rows = min(16, n_rows_total - 16 * static_cast<int>(blockIdx.z));
    if (static_cast<int>(blockIdx.y) >= n_rows) return;
    const int head = blockIdx.x, row = blockIdx.y, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    __shared__ __attribute__((aligned(16))) float red[8][HD + 4];
    __shared__ float red_l[8];
    const int64_t slot_stride = static_cast<int64_t>(n_q) * 16;
    const int64_t slot0 = (blockIdx.z ? static_cast<int64_t>(blockIdx.z) * part_slots : 0) + head * 16 + row;
    const float2 *ml = reinterpret_cast<const float2 *>(part_ml) + slot0;
    const float *po = part_o + slot0 * HD + 4 * (lane % kLanes);
    const float2 own = ml[min(lane, max_splits - 1) * slot_stride];
    float4_t o[kSteps][kEights];
#pragma unroll
    for (int j = 0; j < kSteps; j++)
#pragma unroll
        for (int i = 0; i < kEights; i++) {  // (a lane past the last split re-reads it)
            const int s = min(wave * kPerWave + lane / kLanes + j * kPerWave * kWaves + 8 * i, max_splits - 1);
            o[j][i] = *reinterpret_cast<const float4_t *>(po + s * slot_stride * HD);
        }
    dfl_have(out, out_xf, out_xf_kind, xf_stride);
    if (ctx_len < 0) ctx_len = *ctx_len_dev;
    const int n_splits = want ? attn_splits(ctx_len + 16 * static_cast<int64_t>(blockIdx.z) + n_rows, want, min_chunk) : min_chunk;
    float m_star = lane < n_splits ? own.x : -INFINITY;
    const float m_own = m_star;
    m_star = dfl_wave_max(m_star);
    const float wgt = m_own == -INFINITY ? 0.0f : exp2f(m_own - m_star);
#pragma unroll
    for (int j = 0; j < kSteps; j++) {
        const int sl = wave * kPerWave + lane / kLanes + j * kPerWave * kWaves;
        float4_t acc = {0, 0, 0, 0};
        float l = 0.0f;
#pragma unroll
        for (int i = 0; i < kEights; i++) {
            const int s = sl + 8 * i;
            float w = __shfl(wgt, s, 64), ls = __shfl(own.y, s, 64);
            asm volatile("" : "+v"(w), "+v"(ls));  // (read on every path)
            if (s < n_splits) {
                acc += w * o[j][i];
                l = __builtin_fmaf(w, ls, l);
            }
        }
        *reinterpret_cast<float4_t *>(&red[sl][4 * (lane % kLanes)]) = acc;
        if (lane % kLanes == 0) red_l[sl] = l;
    }
    __syncthreads();
    float lsum = 0.0f;
#pragma unroll
    for (int k = 0; k < 8; k++) lsum += red_l[k];
    if (tid < kLanes) {
        const int d = 4 * tid;
        float4_t v = {0, 0, 0, 0};
#pragma unroll
        for (int k = 0; k < 8; k++) v += *reinterpret_cast<const float4_t *>(&red[k][d]);
        v /= lsum;
        *reinterpret_cast<float4_t *>(out + ((static_cast<int64_t>(blockIdx.z) * 16 + row) * n_q + head) * HD + d) = v;
        if (out_xf)
            dfl_xf_store_pair(static_cast<uint8_t *>(out_xf) + blockIdx.z * xf_stride, out_xf_kind, row, head * HD + (d & ~7), v[0], v[1], v[2], v[3]);
    }
}

// The partial results merged one after the other, as attn_rows_kernel does (which blocks take this: see attn_policy).
// What bounds it is its chain: a trip to memory for the maxima and the partial outputs, which are in flight together,
// then the merges.  Lane s of every wave keeps split s's maximum and sum and computes its two factors
// (the maximum of the splits before it is a scan over the lanes); a thread adds up one dim, with the factors read from the lane
// they are in: no LDS, no barrier.
constexpr int kOrderedSplits = 32;
template <int HD, int kEights>
__global__ void __launch_bounds__(HD)
    attn_combine_ordered_kernel(const float *__restrict__ part_o, const float *__restrict__ part_ml, int64_t ctx_len, int n_q, int n_rows_total,
                                int max_splits, int min_chunk, int want, float *__restrict__ out, void *__restrict__ out_xf, int out_xf_kind,
                                int64_t part_slots, size_t xf_stride, const int32_t *__restrict__ ctx_len_dev) {
    // (the arguments as attn_combine_few_kernel's)
    const int n_rows = min(16, n_rows_total - 16 * static_cast<int>(blockIdx.z));
    if (static_cast<int>(blockIdx.y) >= n_rows) return;
    const int head = blockIdx.x, row = blockIdx.y, d = threadIdx.x, lane = d & 63;
    const int64_t slot_stride = static_cast<int64_t>(n_q) * 16;
    const int64_t slot0 = (blockIdx.z ? static_cast<int64_t>(blockIdx.z) * part_slots : 0) + head * 16 + row;
    const float2 *ml = reinterpret_cast<const float2 *>(part_ml) + slot0;
    const float *po = part_o + slot0 * HD + d;
    const float2 own = ml[min(lane, max_splits - 1) * slot_stride];
    float o[8 * kEights];
#pragma unroll
    for (int s = 0; s < 8 * kEights; s++) {  // (past the last split it is read again)
        o[s] = po[min(s, max_splits - 1) * slot_stride * HD];
    }
    dfl_have(out, out_xf, out_xf_kind, xf_stride);
    if (ctx_len < 0) ctx_len = *ctx_len_dev;
    const int n_splits = want ? attn_splits(ctx_len + 16 * static_cast<int64_t>(blockIdx.z) + n_rows, want, min_chunk) : min_chunk;
    const float m = lane < n_splits ? own.x : -INFINITY;
    const int none = __builtin_bit_cast(int, -INFINITY);
    float upto = m;
#define DFL_MAX_STEP(ctrl, row_mask) \
    upto = fmaxf(upto, __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(none, __builtin_bit_cast(int, upto), ctrl, row_mask, 0xf, false)))
    DFL_MAX_STEP(0x111, 0xf);  // row_shr:1, 2, 4, 8
    DFL_MAX_STEP(0x112, 0xf);
    DFL_MAX_STEP(0x114, 0xf);
    DFL_MAX_STEP(0x118, 0xf);
    DFL_MAX_STEP(0x142, 0xa);  // row_bcast:15 into rows 1 and 3
    DFL_MAX_STEP(0x143, 0xc);  // row_bcast:31 into rows 2 and 3
#undef DFL_MAX_STEP
    const float before = __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(none, __builtin_bit_cast(int, upto), 0x138, 0xf, 0xf, false));  // wave_shr:1
    const AttnMerge w(before, m);
    auto at = [](float v, int s) { return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), s)); };
    float acc = 0.0f, l = 0.0f;
#pragma unroll
    for (int s = 0; s < 8 * kEights; s++) {
        if (s < n_splits) {
            const float old = at(w.old, s), next = at(w.next, s);
            acc = __builtin_fmaf(next, o[s], old * acc);
            l = __builtin_fmaf(next, at(own.y, s), old * l);
        }
    }
    const float v = acc / l;
    out[((static_cast<int64_t>(blockIdx.z) * 16 + row) * n_q + head) * HD + d] = v;
    if (out_xf) {
        // eight consecutive dims sit in eight consecutive lanes of a row of sixteen
        const float e[8] = {v, dfl_dpp<0x101>(v), dfl_dpp<0x102>(v), dfl_dpp<0x103>(v), dfl_dpp<0x104>(v), dfl_dpp<0x105>(v), dfl_dpp<0x106>(v), dfl_dpp<0x107>(v)};
        if ((d & 7) == 0)
            dfl_xf_store(static_cast<uint8_t *>(out_xf) + blockIdx.z * xf_stride, out_xf_kind, row, head * HD + d, e[0], e[1], e[2], e[3], e[4], e[5], e[6], e[7]);
    }
}

// V [pos][n_kv][hd] -> V^T [n_kv][hd][stride]; one workgroup per (32 positions, kv head)
__global__ void __launch_bounds__(256) transpose_v_kernel(const _Float16 *__restrict__ v, _Float16 *__restrict__ vt,
                                                          int64_t n_pos, int n_kv, int hd, int64_t stride) {
    __shared__ _Float16 tile[32][256 + 2];
    const int64_t p0 = static_cast<int64_t>(blockIdx.x) * 32;
    const int kvh = blockIdx.y;
    for (int e = threadIdx.x; e < 32 * hd; e += blockDim.x) {
        int pl = e / hd, d = e - pl * hd;
        int64_t pos = p0 + pl;
        tile[pl][d] = pos < n_pos ? v[(pos * n_kv + kvh) * hd + d] : static_cast<_Float16>(0.0f);
    }
    __syncthreads();
    for (int e = threadIdx.x; e < 32 * hd; e += blockDim.x) {
        int d = e >> 5, pl = e & 31;
        int64_t pos = p0 + pl;
        if (pos < stride) vt[(static_cast<int64_t>(kvh) * hd + d) * stride + pos] = tile[pl][d];
    }
}

template <int HD, typename TQ>
int32_t launch_split(dflash_ctx *ctx, dim3 grid, int threads, hipStream_t st, const void *q, const _Float16 *k, const _Float16 *vt,
                  float *po, float *pml, int64_t ctx_len, const int32_t *ctx_len_dev, int n_rows, int n_q, int n_kv,
                  int64_t vt_stride, int want, int min_chunk, float scale, int full_block, int64_t window, int split_stride,
                  int64_t part_slots, const dfl_attn_rope *rope) {
    const size_t lds = static_cast<size_t>(kAttnBufs) * 2 * (32 * HD / 8) * sizeof(half8_t);
    constexpr int kWaveLoads = 2 * 32 * (HD / 8) / 64;
    const int n_waves = threads / 64, per_wave = (kWaveLoads + n_waves - 1) / n_waves;
    const uint32_t heads = static_cast<uint32_t>(n_kv) | static_cast<uint32_t>(n_q / n_kv) << 20;  // (a group is at most 16)
    const uint32_t split_waves = static_cast<uint32_t>(split_stride) | static_cast<uint32_t>(n_waves) << 24;
    // a single block whose context length is known here: its chunk is, too
    const int64_t chunk = attn_chunk(ctx_len + n_rows, want, min_chunk);
    if (n_rows <= 16 && !ctx_len_dev && chunk <= 0x7fffffff) {
        want = 0;
        min_chunk = static_cast<int>(chunk);
    }
    const uint32_t rope_heads = static_cast<uint32_t>(n_rows - 1) | static_cast<uint32_t>(n_q / n_kv) << 4 | static_cast<uint32_t>(n_kv) << 9;
    const uint32_t rope_split = static_cast<uint32_t>(split_stride) | static_cast<uint32_t>(n_waves) << 11 | static_cast<uint32_t>(chunk / 32) << 16;
#define DFL_ATTN_LAUNCH(MAXW, MAXL)                                                                                 \
    do {                                                                                                            \
        if constexpr (sizeof(TQ) == 4 && MAXW == 8)                                                                 \
            if (rope) {                                                                                             \
                if (const int32_t rc_ = dfl_raise_lds_limit(ctx, reinterpret_cast<const void *>(attn_split_rope_kernel<HD, MAXL>), lds)) \
                    return rc_;                                                                                     \
                attn_split_rope_kernel<HD, MAXL><<<grid, threads + 128, lds, st>>>(                             \
                    static_cast<const float *>(q), const_cast<_Float16 *>(k), const_cast<_Float16 *>(vt), rope->table, rope->q_w, rope_heads, \
                    rope_split, static_cast<int>(ctx_len), static_cast<int>(vt_stride), rope->k_w, rope->eps, scale, po, pml, full_block, window); \
                break;                                                                                              \
            }                                                                                                       \
        if (const int32_t rc_ = dfl_raise_lds_limit(ctx, reinterpret_cast<const void *>(attn_split_kernel<HD, TQ, MAXW, MAXL>), lds)) \
            return rc_;                                                                                             \
        attn_split_kernel<HD, TQ, MAXW, MAXL><<<grid, threads, lds, st>>>(static_cast<const TQ *>(q), k, vt, ctx_len_dev ? -1 : ctx_len, vt_stride, \
                                                                         heads, split_waves, n_rows, min_chunk, want, scale, po, pml, \
                                                                         full_block, window, part_slots, ctx_len_dev); \
    } while (0)
    // one head per wave: two halve the LDS reads per head but measured slower on MI355X
    // (fewer waves to hide the per-stage dependency chain)
    if constexpr (HD < 256) {
        if (threads > 512) {
            DFL_ATTN_LAUNCH(16, 4);
            return DFLASH_OK;
        }
    }
    if (per_wave <= 4)
        DFL_ATTN_LAUNCH(8, 4);
    else if (per_wave <= 8)
        DFL_ATTN_LAUNCH(8, 8);
    else if (per_wave <= 16)
        DFL_ATTN_LAUNCH(8, 16);
    else
        DFL_ATTN_LAUNCH(8, 32);
#undef DFL_ATTN_LAUNCH
    return DFLASH_OK;
}

template <int HD>
int32_t launch_rows(dflash_ctx *ctx, dim3 grid, int n_waves, hipStream_t st, const float *q, const _Float16 *k, const _Float16 *vt, int64_t ctx_len,
                    int n_rows, int n_q, int n_kv, int64_t vt_stride, const AttnRuns &runs, float scale, float *out, void *out_xf, int out_xf_kind) {
    const size_t lds = static_cast<size_t>(kAttnBufs) * 2 * (32 * HD / 8) * sizeof(half8_t);
    constexpr int kWaveLoads = 2 * 32 * (HD / 8) / 64;
    const int per_wave = (kWaveLoads + n_waves - 1) / n_waves;
    const auto fn = per_wave <= 4 ? attn_rows_kernel<HD, 4> : per_wave <= 8 ? attn_rows_kernel<HD, 8> : attn_rows_kernel<HD, 16>;
    if (const int32_t rc_ = dfl_raise_lds_limit(ctx, reinterpret_cast<const void *>(fn), lds)) return rc_;
    fn<<<grid, 64 * n_waves, lds, st>>>(q, k, vt, ctx_len, n_rows, n_q, n_kv, vt_stride, runs, scale, out, out_xf, out_xf_kind,
                                       dfl_xf_bytes(static_cast<int64_t>(n_q) * HD));
    DFL_HIP_CHECK(ctx, hipGetLastError());
    return DFLASH_OK;
}
int32_t launch_rows_pair(dflash_ctx *ctx, dim3 grid, int n_waves, int heads, hipStream_t st, const float *q, const _Float16 *k, const _Float16 *vt, int64_t ctx_len,
                         int n_rows, int n_q, int n_kv, int64_t vt_stride, float scale, float *out, void *out_xf, int out_xf_kind) {
    if (const int32_t rc_ = dfl_raise_lds_limit(ctx, reinterpret_cast<const void *>(attn_rows_pair_kernel), kPairLds)) return rc_;
    attn_rows_pair_kernel<<<grid, 64 * n_waves, kPairLds, st>>>(q, k, vt, ctx_len, n_rows, n_q, n_kv, vt_stride, scale, out, out_xf, out_xf_kind,
                                                                dfl_xf_bytes(static_cast<int64_t>(n_q) * 256), heads);
    DFL_HIP_CHECK(ctx, hipGetLastError());
    return DFLASH_OK;
}

}  // namespace

extern "C" int32_t dflash_attn_verify_block(dflash_ctx *ctx, const void *q, int32_t q_type, const void *k_cache,
                                            const void *v_cache, int32_t v_layout, int64_t ctx_len, int32_t n_rows,
                                            int32_t n_q, int32_t n_kv, int32_t head_dim, int64_t kv_capacity,
                                            float scale, float *out, dflash_stream_t stream) {
    return dfl_attn_block(ctx, q, q_type, k_cache, v_cache, v_layout, ctx_len, n_rows, n_q, n_kv, head_dim, kv_capacity,
                          scale, out, stream, 0, 0, nullptr);
}

// n_rows_total rows, sixteen to a block (every block in the same bucket of context lengths: the caller's business);
// max_blocks_out: how many blocks the workspace holds partial tiles for (the caller launches the rest in further runs).
static int32_t attn_rows(dflash_ctx *ctx, const void *q, int32_t q_type, const void *k_cache, const void *v_cache,
                         int32_t v_layout, int64_t ctx_len, int32_t n_rows_total, int32_t n_q, int32_t n_kv, int32_t head_dim,
                         int64_t kv_capacity, float scale, float *out, dflash_stream_t stream, int32_t full_block,
                         int64_t window, const int32_t *ctx_len_dev, void *out_xf, int out_xf_kind, int32_t *blocks_done,
                         const dfl_attn_rope *rope = nullptr);

int32_t dfl_attn_block(dflash_ctx *ctx, const void *q, int32_t q_type, const void *k_cache, const void *v_cache,
                       int32_t v_layout, int64_t ctx_len, int32_t n_rows, int32_t n_q, int32_t n_kv, int32_t head_dim,
                       int64_t kv_capacity, float scale, float *out, dflash_stream_t stream, int32_t full_block,
                       int64_t window, const int32_t *ctx_len_dev, void *out_xf, int out_xf_kind, const dfl_attn_rope *rope) {
    if (!ctx) return DFLASH_ERR_INVALID_INPUT;
    if (n_rows < 1 || n_rows > 16) return dfl_fail(ctx, DFLASH_ERR_BAD_SHAPE, "attn_verify: n_rows %d outside 1..16", n_rows);
    if (rope && (q_type != DFLASH_TYPE_F32 || v_layout != 1 || ctx_len_dev ||
                 !dfl_attn_rope_takes(ctx, *rope, q, n_q, n_kv, ctx_len, n_rows, head_dim, kv_capacity)))
        return dfl_fail(ctx, DFLASH_ERR_UNSUPPORTED, "attn_verify: rows as the projections left them are not taken here");
    return attn_rows(ctx, q, q_type, k_cache, v_cache, v_layout, ctx_len, n_rows, n_q, n_kv, head_dim, kv_capacity, scale, out, stream,
                     full_block, window, ctx_len_dev, out_xf, out_xf_kind, nullptr, rope);
}

static int32_t attn_check(dflash_ctx *ctx, const void *q, int32_t q_type, const void *k_cache, const void *v_cache, int32_t v_layout,
                          int64_t ctx_len, int32_t n_rows_total, int32_t n_q, int32_t n_kv, int32_t head_dim, int64_t kv_capacity,
                          const float *out, const int32_t *ctx_len_dev, const void *out_xf, int out_xf_kind) {
    if (n_rows_total > 16 && (v_layout != 1 || ctx_len_dev))
        return dfl_fail(ctx, DFLASH_ERR_UNSUPPORTED, "attn_verify: several blocks need the transposed V cache and a host-side context length");
    if (out_xf && ((n_q * head_dim) % DFL_QK_K || reinterpret_cast<uintptr_t>(out_xf) % 16 ||
                   (out_xf_kind != DFL_XF_Q4K && out_xf_kind != DFL_XF_Q6K)))
        return dfl_fail(ctx, DFLASH_ERR_BAD_SHAPE, "attn_verify: fragment-order output needs n_q * head_dim %% 256 == 0 and a kind");
    if (!q || !k_cache || !v_cache || !out) return dfl_fail(ctx, DFLASH_ERR_INVALID_INPUT, "attn_verify: null pointer");
    if (n_q < 1 || n_kv < 1 || n_q % n_kv || n_q / n_kv > 16)
        return dfl_fail(ctx, DFLASH_ERR_BAD_SHAPE, "attn_verify: %d query heads over %d KV heads (group must be 1..16)",
                        n_q, n_kv);
    if (head_dim != 64 && head_dim != 128 && head_dim != 256)
        return dfl_fail(ctx, DFLASH_ERR_UNSUPPORTED, "attn_verify: head_dim %d (64, 128, 256 supported)", head_dim);
    if (ctx_len < 0 || ctx_len + n_rows_total > kv_capacity)
        return dfl_fail(ctx, DFLASH_ERR_STATE, "attn_verify: context %lld + %d rows exceeds the cache capacity %lld",
                        static_cast<long long>(ctx_len), n_rows_total, static_cast<long long>(kv_capacity));
    if (q_type != DFLASH_TYPE_F32 && q_type != DFLASH_TYPE_F16)
        return dfl_fail(ctx, DFLASH_ERR_UNSUPPORTED, "attn_verify: queries must be f32 or f16");
    if (v_layout != 0 && v_layout != 1) return dfl_fail(ctx, DFLASH_ERR_INVALID_INPUT, "attn_verify: v_layout");
    if (ctx_len_dev && v_layout != 1)
        return dfl_fail(ctx, DFLASH_ERR_UNSUPPORTED, "attn_verify: a device-side context length needs the transposed V cache");
    if (v_layout == 1 && kv_capacity % 32)
        return dfl_fail(ctx, DFLASH_ERR_ALIGNMENT, "attn_verify: transposed V needs a capacity that is a multiple of 32");
    if (reinterpret_cast<uintptr_t>(q) % 16 || reinterpret_cast<uintptr_t>(k_cache) % 16 ||
        reinterpret_cast<uintptr_t>(v_cache) % 16 || reinterpret_cast<uintptr_t>(out) % 16)
        return dfl_fail(ctx, DFLASH_ERR_ALIGNMENT, "attn_verify: Q, K, V and the output must be 16-byte aligned");
    return DFLASH_OK;
}

// How a block's keys are split and its heads shared out, by the bucket of its context length alone.
struct AttnPolicy {
    int want;           // splits asked for
    int64_t min_chunk;  // keys per split at least
    int hw;             // heads per workgroup, a single block
    bool ordered;       // the splits' results are merged in order (attn_combine_ordered_kernel, attn_rows_kernel)
};
static AttnPolicy attn_policy(const dflash_ctx *ctx, int64_t bucket, int n_kv, int group, int head_dim) {
    // KV splits: enough workgroups to cover the chip once or twice, chunks a multiple of 32 keys and at least
    // min_chunk keys long (a split costs a partial tile per head and row).  The policy is a function of the
    // bucket alone.
    // Workgroups per CU the split aims at, in halves.  Short contexts: one (fewer splits, fewer partial tiles to merge).
    // Long contexts: two where two workgroups' LDS rings fit a CU side by side (heads of 64 or 128); with heads of 256 a
    // ring is 128 KB, a CU holds one workgroup, and a second round of them only halves the chunk: a workgroup's partial
    // tiles (16 rows x its heads x head_dim floats) are then as many bytes as the keys and values it read.  Half a
    // workgroup per CU there (16 q / 2 kv heads of 256, 40-layer verify: 5.25 -> 4.79 ms at 16 k of context with chunks
    // of 256 keys instead of 128, 6.21 -> 5.80 ms at 32 k with 512; a quarter measured slower again.  Taken with rings of
    // three buffers, 96 KB, which share a CU as little.)
    const size_t ring_bytes = static_cast<size_t>(kAttnBufs) * 2 * 32 * head_dim * sizeof(_Float16);
    int per_cu_x2 = bucket >= 16384 ? (2 * ring_bytes <= static_cast<size_t>(ctx->lds_bytes) ? 4 : 1) : 2;
    int64_t min_chunk = bucket >= 8192 ? 128 : 64;
    // A workgroup serves hw heads of a GQA group (one wave each).  What a workgroup moves is its chunk of K and V,
    // its heads' queries and their partial outputs, and one CU takes in only 20-30 KB per microsecond: at short
    // contexts, where whole groups would leave most CUs without a workgroup, the group is divided until the chip
    // is covered (the chunk is then read by group / hw workgroups, of one XCD).
    // (Measured on the 16 q / 2 kv head shape of 256, 40-layer verify: covering half the chip is enough - 4 heads per
    // workgroup at 2 k of context, 2 at 1 k: 4.19 against 4.24 ms and 4.35 against 4.57 ms - but eight waves on one chunk
    // are too many - at 4-8 k, 4 heads per workgroup: 4.75 against 4.81 ms, 4.20 against 4.28 ms.)
    static const int env_cover_div = [] { const char *e = getenv("DFLASH_ATTN_COVER_DIV"); return e ? atoi(e) : 0; }();
    const int cover_div = env_cover_div > 0 ? env_cover_div : 2;
    int hw = group;
    if (cover_div > 1 && group % 4 == 0 && group > 4 && bucket < 16384) hw = 4;
    while (hw % 2 == 0 && static_cast<int64_t>(n_kv) * (group / hw) * ((bucket + min_chunk - 1) / min_chunk) < ctx->n_cu / cover_div) hw /= 2;
    // tuning knobs, read once per process
    static const int env_per_cu = [] { const char *e = getenv("DFLASH_ATTN_PER_CU"); return e ? atoi(e) : 0; }();
    static const int env_min_chunk = [] { const char *e = getenv("DFLASH_ATTN_MIN_CHUNK"); return e ? atoi(e) : 0; }();
    static const int env_hw = [] { const char *e = getenv("DFLASH_ATTN_HW"); return e ? atoi(e) : 0; }();
    if (env_per_cu > 0) per_cu_x2 = 2 * env_per_cu;
    if (env_min_chunk > 0) min_chunk = env_min_chunk;
    // A workgroup of one wave asks for a whole stage by itself, with a table's loads ahead of it where the attention rotates (65 loads a
    // split, heads of 256), and none of its SIMD's time is another's: two heads at least, with heads of 128 four, where the rule
    // above divides further.  What covers the chip decides on the split (want) all the same: the same bits.  A call at 330 positions,
    // one, two and four heads a workgroup, 16 rows / one row: 16 / 2 heads of 256 12.4, 10.5, 11.4 / 11.7, 9.3, 9.3 us; 32 / 8 of
    // 128 9.1, 8.4, 8.5 / 8.3, 7.5, 7.2; 16 / 8 of 128 8.6, 7.9 / 8.2, 7.4; 16 / 4 of 64 7.2, 6.5, 6.7 / 7.0, 6.2, 6.3; at
    // 1000 positions by as much.  With the rotation inside, of a layer: 16 / 2 of 256 3.2, 2.5 / 2.7, 3.1 less than with one head, 32 / 8 of 128
    // 1.1, 2.9 / 1.8, 2.6.  (Six heads of 128 keep their one part or two: 48 / 8 at 1500 positions, 13.7 : 12.3 / 8.4 : 8.8.)
    int served = hw;
    const int least = head_dim == 128 ? 4 : 2;
    while (2 * served <= least && group % (2 * served) == 0) served *= 2;
    if (env_hw > 0 && group % env_hw == 0) served = hw = env_hw;
    if (per_cu_x2 < 1) per_cu_x2 = 1;
    if (min_chunk < 32) min_chunk = 32;
    const int n_parts = group / hw;
    int want = static_cast<int>(std::max<int64_t>(
        1, (static_cast<int64_t>(per_cu_x2) * ctx->n_cu + 2 * n_kv * n_parts - 1) / (2 * n_kv * n_parts)));
    // (one workgroup per CU at most: beyond half the chip the chunks stay at 512 to 1024 keys - at 64 k of context 256
    // workgroups of 512 keys took 5.79 ms per 40-layer verify where 128 of 1024 took 6.70)
    static const int env_long_chunk = [] { const char *e = getenv("DFLASH_ATTN_LONG_CHUNK"); return e ? atoi(e) : 0; }();
    // (at most 256 splits, which two workgroups per CU would ask for as well: the partial tiles' share of the workspace stays what it was)
    if (per_cu_x2 == 1)
        want = std::max<int>(want, static_cast<int>(std::min<int64_t>(256, bucket / (env_long_chunk >= 32 ? env_long_chunk : 512))));
    // In order where a prefill's workgroup can then keep a merge in registers beside the split at hand (heads of 256 are
    // two accumulators of 64 a lane, the queries' 32 and the values' 64: one wave per SIMD) and where the merge is no slower
    // for a block alone (16 rows of 32 heads of 128 inside a graph: 17 to 32 splits 4.6 -> 4.2 us; 64 splits, 16 rows x
    // 100 k keys, 101.3 -> 102.7 us with the attention).  By the most splits any context of the bucket can have, not the
    // launch's: the bits must not depend on it.
    const int64_t max_splits = std::min<int64_t>(want, (2 * bucket - 1 + min_chunk - 1) / min_chunk);
    return {want, min_chunk, served, head_dim < 256 && max_splits <= kOrderedSplits};
}

// Loads of rows, table and weights are of 16 bytes; a chunk goes over as sixteen bits of stages.  Beside its heads' waves a workgroup has two more: with
// heads of 256 a wave holds more than a third of a SIMD's registers, so there are eight at most.
bool dfl_attn_rope_takes(const dflash_ctx *ctx, const dfl_attn_rope &r, const void *rows, int32_t n_q, int32_t n_kv, int64_t ctx_len, int32_t n_rows,
                         int32_t head_dim, int64_t kv_capacity) {
    const uintptr_t at = reinterpret_cast<uintptr_t>(rows) | reinterpret_cast<uintptr_t>(r.table) | reinterpret_cast<uintptr_t>(r.q_w) | reinterpret_cast<uintptr_t>(r.k_w);
    if (!r.table || !r.q_w || !r.k_w || !rows || at % 16 || n_rows < 1 || n_rows > 16 || ctx_len < 0 || kv_capacity > 65535 * 32 || n_kv < 1 || n_kv >= 1 << 20 || n_q % n_kv ||
        n_q / n_kv > 16 || (head_dim != 64 && head_dim != 128 && head_dim != 256))
        return false;
    return attn_policy(ctx, dfl_attn_bucket(ctx_len + n_rows), n_kv, n_q / n_kv, head_dim).hw <= (head_dim == 256 ? 6 : 8);
}

int32_t dfl_attn_blocks(dflash_ctx *ctx, const void *q, int32_t q_type, const void *k_cache, const void *vt_cache, int64_t ctx_len,
                        int32_t n_rows_total, int32_t n_q, int32_t n_kv, int32_t head_dim, int64_t kv_capacity, float scale,
                        float *out, dflash_stream_t stream, void *out_xf, int out_xf_kind) {
    if (!ctx) return DFLASH_ERR_INVALID_INPUT;
    if (n_rows_total < 1) return dfl_fail(ctx, DFLASH_ERR_BAD_SHAPE, "attn_verify: %d rows", n_rows_total);
    const size_t q_block = static_cast<size_t>(16) * n_q * head_dim;
    const size_t xf_block = dfl_xf_bytes(static_cast<int64_t>(n_q) * head_dim);
    const size_t q_el = q_type == DFLASH_TYPE_F16 ? 2 : 4;
    int32_t done = 0;
    const int32_t n_blocks = (n_rows_total + 15) / 16;
    if (const int32_t rc_ = attn_check(ctx, q, q_type, k_cache, vt_cache, 1, ctx_len, n_rows_total, n_q, n_kv, head_dim, kv_capacity, out, nullptr,
                                       out_xf, out_xf_kind))
        return rc_;
    const int group = n_q / n_kv;
    auto bucket_of = [&](int32_t b) { return dfl_attn_bucket(ctx_len + 16ll * b + std::min(16, n_rows_total - 16 * b)); };
    {
        // The leading blocks whose splits are merged in order: one launch without partial results, or the splits and their
        // merges.  A workgroup of the one launch takes its stages one after the other, about 1.15 us each: n_steps of them for
        // the last block.  The splits spread them over the chip, but they are two launches for every run of blocks that
        // shares a policy (11 us), and a partial tile (16 rows of a head, 8 KB at 128 dims) goes out and comes back; besides,
        // a stage of a workgroup.  Both sides in us, by least squares over 111 pairs of measured sides: 16 / 8, 32 / 8, 48 / 8
        // and 20 / 4 heads of 128, 32 / 4 of 64, 33 - 1024 rows behind 0 - 3900 positions (one layer, splits against one
        // launch: 32 / 8 heads 143 : 46 us for 1024 rows behind none, 87 : 78 for 256 behind 1900, 56 : 134 for 128 behind
        // 3900; 32 / 4 of 64 80 : 36, 55 : 66, 32 : 115).  The better side, or within 6 % of it, in all but one (1.24).
        AttnRuns runs = {};
        int32_t taken = 0;
        int64_t partials = 0;  // partial tiles of 128 dims
        for (int64_t last = -1; taken < n_blocks && q_type == DFLASH_TYPE_F32; taken++) {
            const int64_t n_pos = ctx_len + std::min(16 * (taken + 1), n_rows_total), bucket = dfl_attn_bucket(n_pos);
            if (bucket != last) {
                const AttnPolicy p = attn_policy(ctx, bucket, n_kv, group, head_dim);
                if ((!p.ordered && head_dim != 256) || runs.n == kAttnRuns) break;
                last = bucket;
                runs.first[runs.n] = taken;
                runs.want[runs.n] = p.want;
                runs.min_chunk[runs.n++] = static_cast<int>(p.min_chunk);
            }
            const int64_t chunk = attn_chunk(n_pos, runs.want[runs.n - 1], runs.min_chunk[runs.n - 1]);
            if (head_dim == 256 && (chunk != kPairSplit || n_pos > 0x3fffffff)) break;
            partials += (n_pos + chunk - 1) / chunk * n_q * head_dim / 128;
        }
        int hw = std::min(group, 8);
        while (group % hw) hw--;
        const int32_t rows = std::min(n_rows_total, 16 * taken);
        // Heads of 256: four heads of a block where those workgroups fit the chip side by side, 2.6 us a split (with eight heads 3.4:
        // 16 / 2 heads, 1024 rows 85 -> 67 us); beyond, four heads of two blocks, a long one and a short one, as
        // attn_rows_pair_kernel has them: 3.2 us for a split of the longest (1536 rows 117 -> 94 us, 2048 rows 147 -> 124).
        const bool fours = head_dim == 256 && hw % 4 == 0, two = fours && static_cast<int64_t>(taken) * n_kv * (group / 4) > ctx->n_cu;
        if (fours) hw = 4;
        const int32_t units = two ? (taken + 1) / 2 : taken;
        const int64_t wgs = static_cast<int64_t>(units) * n_kv * (group / hw), n_steps = (ctx_len + rows + 31) / 32;
        const int64_t stages = wgs * (ctx_len + rows / 2) / 32;
        const double as_splits = (head_dim == 256 ? 20.0 : 11.0) * runs.n + (0.5 * stages + 1.1 * partials) / ctx->n_cu;
        double one_launch = 5.5 + 1.15 * n_steps;
        // Heads of 256 walk the keys twice: 14 us and 2.6, 3.2 or (workgroups of another number of heads than four) 4.2 us for a split of
        // two stages, 8 us more where the total goes out and back; the two launches of a run 20 us.  Both sides in us, the last layer's worth of 95 measured
        // pairs (splits : one launch): 16 / 2 heads 452 : 154 for 2048 rows behind none, 60 : 36 for 512, 155 : 111 for 512 behind
        // 1520, 71 : 98 for 256 behind 1520, 38 : 149 for 64 behind 3040; 8 / 1 heads 74 : 107 and 161 : 129 for 512 and 1024
        // behind 1520; 32 / 4 heads 43 : 25 for 256 behind none; 5 / 1 heads 191 : 193 for 2048 behind none.
        if (head_dim == 256)
            one_launch = (n_steps > 16 ? 22.0 : 14.0) + (two ? 3.2 : fours ? 2.6 : 4.2) * std::max(0.5 * n_steps, 0.65 * stages / ctx->n_cu);
        if (taken > 1 && one_launch <= as_splits) {
            hipStream_t st = static_cast<hipStream_t>(stream);
            dfl_timed timer(ctx, st, DFL_T_ATTN);
            if (head_dim == 256) {
                if (const int32_t rc_ = launch_rows_pair(ctx, dim3(group / hw, n_kv, units), two ? 8 : hw, hw, st, static_cast<const float *>(q),
                                                         static_cast<const _Float16 *>(k_cache), static_cast<const _Float16 *>(vt_cache), ctx_len, rows, n_q,
                                                         n_kv, kv_capacity, scale, out, out_xf, out_xf_kind))
                    return rc_;
            } else if (const int32_t rc_ = (head_dim == 64 ? launch_rows<64> : launch_rows<128>)(ctx, dim3(group / hw, n_kv, taken), hw, st, static_cast<const float *>(q), static_cast<const _Float16 *>(k_cache),
                                           static_cast<const _Float16 *>(vt_cache), ctx_len, rows, n_q, n_kv, kv_capacity, runs, scale, out, out_xf,
                                           out_xf_kind))
                return rc_;
            done = taken;
        }
    }
    while (done < n_blocks) {
        // a run: the blocks from `done` on that share its bucket (the split policy is a function of the bucket)
        const int64_t len0 = ctx_len + 16ll * done;
        int32_t run = 1;
        while (done + run < n_blocks && bucket_of(done + run) == bucket_of(done)) run++;
        const int32_t rows = std::min(n_rows_total - 16 * done, 16 * run);
        int32_t taken = 0;
        const int32_t rc = attn_rows(ctx, static_cast<const uint8_t *>(q) + done * q_block * q_el, q_type, k_cache, vt_cache, 1, len0, rows,
                                     n_q, n_kv, head_dim, kv_capacity, scale, out + done * q_block, stream, 0, 0, nullptr,
                                     out_xf ? static_cast<uint8_t *>(out_xf) + done * xf_block : nullptr, out_xf_kind, &taken);
        if (rc) return rc;
        done += taken;
    }
    return DFLASH_OK;
}

static int32_t attn_rows(dflash_ctx *ctx, const void *q, int32_t q_type, const void *k_cache, const void *v_cache,
                         int32_t v_layout, int64_t ctx_len, int32_t n_rows_total, int32_t n_q, int32_t n_kv, int32_t head_dim,
                         int64_t kv_capacity, float scale, float *out, dflash_stream_t stream, int32_t full_block,
                         int64_t window, const int32_t *ctx_len_dev, void *out_xf, int out_xf_kind, int32_t *blocks_done,
                         const dfl_attn_rope *rope) {
    int32_t n_blocks = (n_rows_total + 15) / 16;
    const int32_t n_rows = std::min(16, n_rows_total);  // rows of the first block: what the split policy looks at
    if (const int32_t rc_ = attn_check(ctx, q, q_type, k_cache, v_cache, v_layout, ctx_len, n_rows_total, n_q, n_kv, head_dim, kv_capacity, out,
                                       ctx_len_dev, out_xf, out_xf_kind))
        return rc_;

    hipStream_t st = static_cast<hipStream_t>(stream);
    const int group = n_q / n_kv;
    // with ctx_len_dev the context length is read on the device: everything sized here is then sized for the
    // largest context of the bucket
    const int64_t bucket = dfl_attn_bucket(ctx_len + n_rows);
    int64_t n_pos = ctx_len_dev ? std::min<int64_t>(kv_capacity, 2 * bucket - 1) : ctx_len + n_rows_total;

    const AttnPolicy policy = attn_policy(ctx, bucket, n_kv, group, head_dim);
    const int want = policy.want;
    const int64_t min_chunk = policy.min_chunk;
    int hw = policy.hw, n_parts = group / hw;  // workgroups per (chunk, KV head)
    // Several blocks in one launch cover the chip between them: a workgroup then serves the whole GQA group, so a chunk
    // of keys is staged once instead of group / hw times (a workgroup's LDS ring leaves no room for a second one on
    // its CU, whatever its size).  The split of the keys (want, min_chunk) stays the single block's, and a head is one
    // wave's work either way: the same bits.
    if (n_blocks > 1) {
        hw = group;
        n_parts = 1;
    }
    // heads of 256: eight waves at most (registers); again the split of the keys stays
    while (head_dim == 256 && hw > 8) {
        int d = hw - 1;
        while (group % d) d--;
        hw = d;
        n_parts = group / hw;
    }
    // The most splits that any of the blocks has, or, with ctx_len_dev, that any context up to n_pos can have.  Not always the
    // last block's: where a split's share of the keys passes a whole stage, all splits grow by one and there are fewer of them
    // (6 splits asked for: 384 keys are 6 of 64, 385 are 5 of 96).
    auto splits_for = [&](int32_t blocks) {
        if (ctx_len_dev) return static_cast<int>(std::min<int64_t>(want, (n_pos + min_chunk - 1) / min_chunk));
        int most = 1;
        for (int32_t b = 0; b < blocks; b++) most = std::max(most, attn_splits(ctx_len + std::min(16 * (b + 1), n_rows_total), want, min_chunk));
        return most;
    };
    int n_splits = splits_for(n_blocks);
    // several blocks: as many as the workspace has room for partial tiles of (the caller comes back for the rest)
    const size_t slot_bytes = static_cast<size_t>(n_q) * 16 * (head_dim + 2) * sizeof(float);
    if (n_blocks > 1) {
        const size_t room = ctx->workspace_bytes > 4096 ? ctx->workspace_bytes - 4096 : 0;
        while (n_blocks > 1 && static_cast<size_t>(n_blocks) * n_splits * slot_bytes > room) {
            n_blocks--;
            n_rows_total = 16 * n_blocks;
            n_pos = ctx_len + n_rows_total;
            n_splits = splits_for(n_blocks);
        }
    }
    if (blocks_done) *blocks_done = n_blocks;
    const int64_t part_slots = static_cast<int64_t>(n_splits) * n_q * 16;

    size_t off = 0;
    float *part_o = dfl_ws_take<float>(ctx, &off, static_cast<size_t>(n_blocks) * part_slots * head_dim * sizeof(float));
    float *part_ml = dfl_ws_take<float>(ctx, &off, static_cast<size_t>(n_blocks) * part_slots * 2 * sizeof(float));
    const _Float16 *vt = static_cast<const _Float16 *>(v_cache);
    int64_t vt_stride = kv_capacity;
    if (v_layout == 0) {
        vt_stride = (n_pos + 31) / 32 * 32;
        _Float16 *vt_ws = dfl_ws_take<_Float16>(ctx, &off, static_cast<size_t>(n_kv) * head_dim * vt_stride * 2);
        if (!vt_ws)
            return dfl_fail(ctx, DFLASH_ERR_WORKSPACE,
                            "attn_verify: transposing V needs %zu workspace bytes; pass the transposed cache instead",
                            static_cast<size_t>(n_kv) * head_dim * vt_stride * 2);
        transpose_v_kernel<<<dim3(static_cast<unsigned>(vt_stride / 32), n_kv), 256, 0, st>>>(
            static_cast<const _Float16 *>(v_cache), vt_ws, n_pos, n_kv, head_dim, vt_stride);
        vt = vt_ws;
    }
    if (!part_o || !part_ml) return dfl_fail(ctx, DFLASH_ERR_WORKSPACE, "attn_verify: workspace too small");

    if (n_splits > 1024) return dfl_fail(ctx, DFLASH_ERR_UNSUPPORTED, "attn_verify: %d KV splits", n_splits);
    const int split_stride = (n_splits + 7) / 8 * 8;
    const dim3 grid(split_stride * n_parts, n_kv, n_blocks);
    const int threads = 64 * hw;
    const _Float16 *k = static_cast<const _Float16 *>(k_cache);
    int32_t rc = DFLASH_OK;
    {
        dfl_timed timer(ctx, st, DFL_T_ATTN);
#define DFL_ATTN(HD)                                                                                              \
    if (q_type == DFLASH_TYPE_F32)                                                                                \
        rc = launch_split<HD, float>(ctx, grid, threads, st, q, k, vt, part_o, part_ml, ctx_len, ctx_len_dev, n_rows_total, n_q, n_kv, \
                                     vt_stride, want, static_cast<int>(min_chunk), scale, full_block, window,     \
                                     split_stride, part_slots, rope);                                             \
    else                                                                                                          \
        rc = launch_split<HD, _Float16>(ctx, grid, threads, st, q, k, vt, part_o, part_ml, ctx_len, ctx_len_dev, n_rows_total, n_q, \
                                        n_kv, vt_stride, want, static_cast<int>(min_chunk), scale, full_block, window, \
                                        split_stride, part_slots, nullptr)
        if (head_dim == 64) {
            DFL_ATTN(64);
        } else if (head_dim == 128) {
            DFL_ATTN(128);
        } else {
            DFL_ATTN(256);
        }
#undef DFL_ATTN
    }
    if (rc) return rc;
    const bool known = n_blocks == 1 && !ctx_len_dev;  // (the number of splits: the one block's)
    if (policy.ordered) {
        typedef decltype(&attn_combine_ordered_kernel<64, 1>) fn_t;
        static const fn_t fns[2][4] = {
            {attn_combine_ordered_kernel<64, 1>, attn_combine_ordered_kernel<64, 2>, attn_combine_ordered_kernel<64, 3>, attn_combine_ordered_kernel<64, 4>},
            {attn_combine_ordered_kernel<128, 1>, attn_combine_ordered_kernel<128, 2>, attn_combine_ordered_kernel<128, 3>, attn_combine_ordered_kernel<128, 4>}};
        static_assert(kOrderedSplits == 32, "as many eights");
        const fn_t fn = fns[head_dim == 128][(n_splits - 1) / 8];
        fn<<<dim3(n_q, n_rows, n_blocks), head_dim, 0, st>>>(part_o, part_ml, ctx_len_dev ? -1 : ctx_len, n_q, n_rows_total, n_splits, known ? n_splits : static_cast<int>(min_chunk),
                                                            known ? 0 : want, out, out_xf, out_xf_kind, part_slots,
                                                            dfl_xf_bytes(static_cast<int64_t>(n_q) * head_dim), ctx_len_dev);
        DFL_HIP_CHECK(ctx, hipGetLastError());
        return DFLASH_OK;
    }
    // (more splits than that and the shuffles of the weights cost more than the barriers they replace)
    if (n_splits <= 48) {
        typedef decltype(&attn_combine_few_kernel<64, 1>) fn_t;
#define DFL_FEW(HD)                                                                                                       \
    {attn_combine_few_kernel<HD, 1>, attn_combine_few_kernel<HD, 2>, attn_combine_few_kernel<HD, 3>, attn_combine_few_kernel<HD, 4>, \
     attn_combine_few_kernel<HD, 5>, attn_combine_few_kernel<HD, 6>}
        static const fn_t fns[3][6] = {DFL_FEW(64), DFL_FEW(128), DFL_FEW(256)};
#undef DFL_FEW
        const fn_t fn = fns[head_dim / 128][(n_splits - 1) / 8];
        fn<<<dim3(n_q, n_rows, n_blocks), head_dim == 64 ? 128 : 256, 0, st>>>(part_o, part_ml, ctx_len_dev ? -1 : ctx_len, n_q, n_rows_total, n_splits,
                                                                              known ? n_splits : static_cast<int>(min_chunk), known ? 0 : want, out, out_xf,
                                                                              out_xf_kind, part_slots, dfl_xf_bytes(static_cast<int64_t>(n_q) * head_dim),
                                                                              ctx_len_dev);
        DFL_HIP_CHECK(ctx, hipGetLastError());
        return DFLASH_OK;
    }
    attn_combine_kernel<<<dim3(n_q, n_rows, n_blocks), 256, 0, st>>>(part_o, part_ml, out, n_rows_total, n_q, head_dim, ctx_len, ctx_len_dev,
                                                                    want, static_cast<int>(min_chunk), out_xf, out_xf_kind, part_slots,
                                                                    dfl_xf_bytes(static_cast<int64_t>(n_q) * head_dim), n_splits);
    DFL_HIP_CHECK(ctx, hipGetLastError());
    return DFLASH_OK;
}
