// DFlash-2 extras of the block drafter: the two-tap dynamic depthwise convolution
// (kernel_dflash2_conv_f32, kernels/dflash2.metal:40-69) and the greedy selector walk over the
// predecessor / successor codebooks (select_draft_path, metal_dflash.rs:17176-17251; codebook rows
// DFlash2Codebook::dequant_row, :3275-3343) with its sampled form (draft_block_sampled,
// :17268-17415).  The per-row top-16 that feeds the walk is dflash_top16.
#include "common.h"
#include "device_quant.h"
#include "sampler_chain.h"

#include <algorithm>

// The walk's scores follow the reference's scalar loop: every product and every addition is
// rounded on its own: plain operators with contraction switched off (the __f*_rn intrinsics do not
// stop the compiler from fusing them).
#pragma clang fp contract(off)

namespace {

// y[t][c] = sum_tap (base[side][tap][c] + dyn[t][side][tap][c / group_size]) * x[t - tap][c]; rows
// before the block count as zeros; taps accumulate in order with a fused multiply-add, as the
// reference kernel does.  One thread per element.
// What bounds it: one trip to memory.  So the index arithmetic has no divisions (by_group: ceil(2^32 / group_size), or 0 where that
// is not exact for every channel), two taps' values travel together, and what the first loads need comes preloaded with the wave.
__global__ void __launch_bounds__(256)
    dflash2_conv_kernel(const float *__restrict__ x, const float *__restrict__ dyn, const float *__restrict__ base, int h, int kernel_size,
                        int n_groups, uint32_t by_group, int side, int group_size, float *__restrict__ y, void *__restrict__ y_xf, int y_xf_kind) {
    const int t = blockIdx.x, c = blockIdx.y * 256 + threadIdx.x;
    if (c >= h) return;
    const int g = by_group ? static_cast<int>(__umulhi(c, by_group)) : c / group_size;
    const float *dyn_t = dyn + (static_cast<size_t>(t) * 2 + side) * kernel_size * n_groups + g;
    const float *base_c = base + static_cast<size_t>(side) * kernel_size * h + c, *x_c = x + c;
    float acc = 0.0f;
    for (int tap = 0; tap < kernel_size && tap <= t; tap += 2) {
        const bool two = tap + 1 < kernel_size && tap + 1 <= t;
        const int tp = two ? tap + 1 : tap;
        const float b0 = base_c[static_cast<size_t>(tap) * h], b1 = base_c[static_cast<size_t>(tp) * h];
        const float d0 = dyn_t[static_cast<size_t>(tap) * n_groups], d1 = dyn_t[static_cast<size_t>(tp) * n_groups];
        const float x0 = x_c[static_cast<size_t>(t - tap) * h], x1 = x_c[static_cast<size_t>(t - tp) * h];
        if (tap == 0) dfl_have(y, y_xf, y_xf_kind);
        acc = __builtin_fmaf(b0 + d0, x0, acc);
        if (two) acc = __builtin_fmaf(b1 + d1, x1, acc);
    }
    y[static_cast<size_t>(t) * h + c] = acc;
    if (y_xf) {
        // (h a multiple of 256: the grid has no ragged end and eight consecutive lanes hold eight consecutive channels of a row)
        float v[8];
#pragma unroll
        for (int i = 0; i < 8; i++) v[i] = __shfl_down(acc, i, 64);
        if ((c & 7) == 0) dfl_xf_store(y_xf, y_xf_kind, t, c, v[0], v[1], v[2], v[3], v[4], v[5], v[6], v[7]);
    }
}

struct Codebook {
    int type;
    int rank;
    int64_t n_rows;
    const uint8_t *data;
    size_t row_bytes;
};

// element r of row `row`
__device__ __forceinline__ float codebook_elem(const Codebook &cb, int64_t row, int r) {
    const uint8_t *p = cb.data + static_cast<size_t>(row) * cb.row_bytes;
    if (cb.type == DFLASH_TYPE_F16) return __half2float(reinterpret_cast<const __half *>(p)[r]);
    return dfl_dequant_elem(cb.type, p, r);
}

constexpr int kSelThreads = 256;
constexpr int kSelMaxTopK = 16;
constexpr int kSelMaxRank = 1024;

// What the sampled walk reports besides the tokens.
struct SampledOut {
    int32_t status;      // 0, 1 = predecessor row out of range, else a DFLASH_ERR_* of the sampler
    int32_t err_pos;     // position of that error
    int32_t n_sampled;   // positions whose draw was made (the proposal sampler advances by this)
    int32_t pad;
    int32_t counts[16];                          // candidates with positive weight per position (index pos - 1)
    dflash_weighted_candidate cands[15 * 16];    // [pos - 1][top_k], distribution order
};

// where the raw rows sit in the scores kernel's LDS, behind the decoded ones (bytes)
__host__ __device__ inline size_t sel_raw_pred_bytes(size_t row_bytes) { return (row_bytes + 15) / 16 * 16; }
__host__ __device__ inline size_t sel_raw_succ_stride(size_t row_bytes) { return (row_bytes + 3) / 4 * 4; }
// floats in front of them: gate[rank], products[top_k][sel_prod_stride(rank)], rounded up to a 16-byte boundary
// (a row of products every stride: the sixteen scoring threads read four of sixteen rows at once, and rows a multiple of 64
// floats apart would all sit in one bank)
__host__ __device__ inline int sel_prod_stride(int rank) { return (rank + 3) / 4 * 4 + 4; }
__host__ __device__ inline size_t sel_gate_floats(int rank) { return (static_cast<size_t>(rank) + 3) / 4 * 4; }
__host__ __device__ inline size_t sel_decoded_floats(int top_k, int rank) { return sel_gate_floats(rank) + static_cast<size_t>(top_k) * sel_prod_stride(rank); }

// The walk's scores do not have to wait for the walk: the predecessor of position pos is one of the top_k candidates
// of position pos - 1 (the carry token for pos = 1), so score(pos, a, b) for every candidate a of the previous position
// and every candidate b of this one is known work up front: (n - 1) x top_k workgroups, all at once, each with the
// reference's arithmetic for its sixteen scores.  Workgroup (a, pos): the predecessor row of candidate a gives gate = pred *
// sel_h[pos] in LDS, the successor rows of position pos's candidates the products gate[r] * succ_b[r], all elements at once;
// thread b then adds up candidate b's products as the reference's scalar loop does (products and additions rounded
// separately, rank order): table[pos - 1][a][b] = vals[pos][b] + sum_r gate[r] * succ_b[r], NaN for a candidate without a
// successor row.  A previous candidate without a predecessor row gets no scores: the walk stops when it picks one.
// What bounds it: two trips to memory (the candidates, then their rows) and the sum's chain of `rank` additions.  So a wave
// takes whole rows, whose bytes it asks for together (an index that is divided into row and word, and the candidate looked up again
// per word, were 15.7 us a launch; now 6.5), and in Q4_K a thread decodes sixteen elements of two sub-blocks' scales.
constexpr int kScoreThreads = 512;
__global__ void __launch_bounds__(kScoreThreads)
    dflash2_scores_kernel(const int32_t *__restrict__ ids, const uint8_t *__restrict__ pred_rows, const uint8_t *__restrict__ succ_rows,
                          const float *__restrict__ sel_h, int carry, int top_k, int rank, uint32_t n_pred, uint32_t n_succ, int pred_bytes,
                          int succ_bytes, int pred_type, int succ_type, const float *__restrict__ vals, float *__restrict__ table) {
    extern __shared__ float lds[];  // gate, products, then the raw rows: predecessor, top_k successors
    constexpr int kWaves = kScoreThreads / 64, kRows = kSelMaxTopK / kWaves;  // rows a wave has at most
    float *gate = lds, *prod = lds + sel_gate_floats(rank);
    const int ps = sel_prod_stride(rank);
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int a = blockIdx.x, pos = 1 + blockIdx.y;
    if (pos == 1 && a != 0) return;  // (one predecessor only: the carry token)
    const int32_t cands = ids[pos * top_k + min(lane, top_k - 1)];  // lane b: candidate b
    const int32_t prev = pos == 1 ? carry : ids[(pos - 1) * top_k + a];
    const float *hrow = sel_h + static_cast<size_t>(pos) * rank;
    float h[kSelMaxRank / kScoreThreads];
#pragma unroll
    for (int i = 0; i < kSelMaxRank / kScoreThreads; i++) h[i] = hrow[min(tid + kScoreThreads * i, rank - 1)];
    dfl_have(vals, table);
    if (static_cast<uint32_t>(prev) >= n_pred) return;  // (a negative one, too)
    // The rows' bytes come in with coalesced loads first (decoding element by element straight from memory cost a cold
    // trip per field of every element).  Rows of every codebook type are a whole number of 2-byte words and start on
    // one; in LDS the predecessor row sits first and the successor rows follow, each on a 4-byte boundary.
    uint8_t *raw = reinterpret_cast<uint8_t *>(lds + sel_decoded_floats(top_k, rank));
    const int pw = pred_bytes / 2, sw = succ_bytes / 2;
    const size_t succ_at = sel_raw_pred_bytes(pred_bytes), succ_stride = sel_raw_succ_stride(succ_bytes);
    bool live[kRows];
    const uint16_t *src[kRows];
#pragma unroll
    for (int i = 0; i < kRows; i++) {
        const int b = wave + kWaves * i;
        const int32_t cand = __builtin_amdgcn_readlane(cands, b);
        live[i] = b < top_k && static_cast<uint32_t>(cand) < n_succ;
        src[i] = reinterpret_cast<const uint16_t *>(succ_rows + static_cast<size_t>(live[i] ? cand : 0) * succ_bytes);
    }
    const uint16_t *psrc = reinterpret_cast<const uint16_t *>(pred_rows + static_cast<size_t>(prev) * pred_bytes);
    uint16_t p0 = psrc[min(tid, pw - 1)];
    constexpr int kWords = 3;  // of a lane at once: rows of 384 bytes
    for (int at = 0; at < sw; at += 64 * kWords) {
        uint16_t v[kRows][kWords];
#pragma unroll
        for (int i = 0; i < kRows; i++)
#pragma unroll
            for (int k = 0; k < kWords; k++) v[i][k] = src[i][min(at + lane + 64 * k, sw - 1)];
#pragma unroll
        for (int i = 0; i < kRows; i++)
#pragma unroll
            for (int k = 0; k < kWords; k++)
                if (live[i] && at + lane + 64 * k < sw)
                    reinterpret_cast<uint16_t *>(raw + succ_at + (wave + kWaves * i) * succ_stride)[at + lane + 64 * k] = v[i][k];
    }
    if (tid < pw) reinterpret_cast<uint16_t *>(raw)[tid] = p0;
    for (int i = tid + kScoreThreads; i < pw; i += kScoreThreads) reinterpret_cast<uint16_t *>(raw)[i] = psrc[i];
    __syncthreads();
    Codebook pred_l = {pred_type, rank, 1, raw, static_cast<size_t>(pred_bytes)}, succ_l = {succ_type, rank, top_k, raw + succ_at, succ_stride};
#pragma unroll
    for (int i = 0; i < kSelMaxRank / kScoreThreads; i++)
        if (tid + kScoreThreads * i < rank) gate[tid + kScoreThreads * i] = codebook_elem(pred_l, 0, tid + kScoreThreads * i) * h[i];
    __syncthreads();
    if (succ_type == DFLASH_TYPE_Q4_K) {
        // eight bytes of quants a thread: eight elements of sub-block 2 p, eight of 2 p + 1 (dfl_dequant_elem's arithmetic)
        const int per_row = rank / 16;  // (a multiple of sixteen)
#pragma unroll
        for (int i = 0; i < kRows; i++) {
            if (!live[i]) continue;
            const int b = wave + kWaves * i;
            for (int c = lane; c < per_row; c += 64) {
                const int sb = c >> 4, p = (c >> 2) & 3, l0 = (c & 3) * 8;
                const uint8_t *blk = raw + succ_at + b * succ_stride + sb * DFL_Q4_K_BYTES;
                const uint2 q = *reinterpret_cast<const uint2 *>(blk + 16 + 32 * p + l0);
                float d1[2], m1[2];
#pragma unroll
                for (int u = 0; u < 2; u++) {
                    int sc, m;
                    dfl_q4k_scale_min(blk + 4, 2 * p + u, &sc, &m);
                    d1[u] = __fmul_rn(dfl_h2f(blk), static_cast<float>(sc));
                    m1[u] = __fmul_rn(dfl_h2f(blk + 2), static_cast<float>(m));
                }
                const int r0 = 256 * sb + 64 * p + l0;
#pragma unroll
                for (int u = 0; u < 2; u++)
#pragma unroll
                    for (int k = 0; k < 8; k++) {
                        const uint32_t word = k < 4 ? q.x : q.y;
                        const float e = __fsub_rn(__fmul_rn(d1[u], static_cast<float>((word >> (8 * (k & 3) + 4 * u)) & 15)), m1[u]);
                        prod[b * ps + r0 + 32 * u + k] = gate[r0 + 32 * u + k] * e;
                    }
            }
        }
    } else {
#pragma unroll
        for (int i = 0; i < kRows; i++) {
            if (!live[i]) continue;
            const int b = wave + kWaves * i;
            for (int r = lane; r < rank; r += 64) prod[b * ps + r] = gate[r] * codebook_elem(succ_l, b, r);
        }
    }
    __syncthreads();
    if (tid < top_k) {
        float sc = __builtin_nanf("");  // skipped candidates never compare greater
        if (static_cast<uint32_t>(cands) < n_succ) {
            float dot = 0.0f;
            const float *pr = prod + tid * ps;
            int r = 0;
#pragma unroll 8
            for (; r + 4 <= rank; r += 4) {  // (every product and every sum rounded on its own: contraction is off in this file)
                const float4 v = *reinterpret_cast<const float4 *>(pr + r);
                dot += v.x;
                dot += v.y;
                dot += v.z;
                dot += v.w;
            }
            for (; r < rank; r++) dot += pr[r];
            sc = vals[pos * top_k + tid] + dot;
        }
        table[(static_cast<size_t>(pos - 1) * top_k + a) * top_k + tid] = sc;
    }
}

// The walk over the table, one workgroup: the table and the candidates go to LDS, thread 0 then follows the picks.
// Per position it keeps the first strict maximum of the previous pick's row of scores (greedy) or samples from
// softmax(score / T) with the sampler chain and the position's pre-drawn uniform (SAMPLED).  status: 0, or 1 when a
// picked token has no predecessor row (the walk stops there).
template <bool SAMPLED>
__global__ void __launch_bounds__(kSelThreads)
    dflash2_select_kernel(int64_t n_pred_rows, int64_t n_succ_rows, int top_k, int carry, int n, const int32_t *__restrict__ ids,
                          const float *__restrict__ table, int32_t *__restrict__ out, int32_t *__restrict__ status,
                          float temperature, const double *__restrict__ uniforms, SampledOut *__restrict__ sampled, int32_t *page) {
    // page (may be null): where the tokens go as well, a host page; a place the walk does not reach gets what out holds there
    __shared__ float table_s[15 * kSelMaxTopK * kSelMaxTopK];
    __shared__ int32_t ids_s[16 * kSelMaxTopK];
    __shared__ __attribute__((aligned(16))) uint8_t next_s[16][16];
    __shared__ RowDist dist;
    const int tid = threadIdx.x;
    if (tid == 0) {
        out[0] = ids[0];
        *status = 0;
        if (SAMPLED) {
            sampled->status = 0;
            sampled->err_pos = 0;
            sampled->n_sampled = 0;
            for (int p = 1; p < n; p++) out[p] = ids[0];  // the reference pre-fills every slot with the anchor's top-1
        }
    }
    if (n < 2 || carry < 0 || carry >= n_pred_rows) {
        if (n >= 2 && tid == 0) *status = 1;
        if (page && tid < n) page[tid] = tid == 0 ? ids[0] : out[tid];
        return;
    }
    {
        const int n_table = (n - 1) * top_k * top_k;
        float t[15];
#pragma unroll
        for (int i = 0; i < 15; i++) t[i] = table[min(tid + kSelThreads * i, n_table - 1)];
        const int32_t id = ids[min(tid, n * top_k - 1)];
#pragma unroll
        for (int i = 0; i < 15; i++)
            if (tid + kSelThreads * i < n_table) table_s[tid + kSelThreads * i] = t[i];
        if (tid < n * top_k) ids_s[tid] = id;
    }
    __syncthreads();
    if (!SAMPLED) {
        // greedy.  Which candidate follows candidate a of the position before is known for every (position, a) without the walk: the
        // first strict maximum over the candidates with a successor row, as the scalar loop `if (score[b] > best)` from best =
        // -inf keeps it (a NaN or -inf score is never greater: with none greater, candidate 0 stands).  Sixteen lanes a
        // previous candidate find it for all positions (the maximum crosses them by DPP moves), and the walk itself
        // is a look-up per position out of scalar registers.  (A maximum over shuffles per position, one after the other: 9.7 us
        // a launch; now 6.1.)
        const int b = tid & 15, a = tid >> 4;  // (256 threads: sixteen previous candidates)
        for (int pos = 1; pos < n; pos++) {
            const int32_t cand = b < top_k ? ids_s[pos * top_k + b] : -1;
            const float v = b < top_k && a < top_k ? table_s[(static_cast<size_t>(pos - 1) * top_k + a) * top_k + b] : -INFINITY;
            const float sc = cand >= 0 && cand < n_succ_rows && v > -INFINITY ? v : -INFINITY;
            float best = sc;
            best = fmaxf(best, dfl_dpp<0x128>(best));  // row_ror:8, 4, 2, 1
            best = fmaxf(best, dfl_dpp<0x124>(best));
            best = fmaxf(best, dfl_dpp<0x122>(best));
            best = fmaxf(best, dfl_dpp<0x121>(best));
            const unsigned long long at = __ballot(sc == best && best > -INFINITY);
            const uint32_t mine = static_cast<uint32_t>(at >> (16 * (a & 3))) & 0xffffu;
            if (b == 0) next_s[pos][a] = static_cast<uint8_t>(mine ? __builtin_ctz(mine) : 0);
        }
        __syncthreads();
        if (tid >= 64) return;
        const uint4 next = *reinterpret_cast<const uint4 *>(next_s[min(tid, 15)]);  // lane pos: the sixteen of a position
        int picked = 0, prev_a = 0;  // lane pos: its pick
        for (int pos = 1; pos < n; pos++) {
            const uint32_t w = prev_a < 8 ? (prev_a < 4 ? __builtin_amdgcn_readlane(next.x, pos) : __builtin_amdgcn_readlane(next.y, pos))
                                          : (prev_a < 12 ? __builtin_amdgcn_readlane(next.z, pos) : __builtin_amdgcn_readlane(next.w, pos));
            prev_a = w >> (8 * (prev_a & 3)) & 255;
            picked = tid == pos ? prev_a : picked;
        }
        // the walk ends behind the first pick without a predecessor row
        const int32_t chosen = tid >= 1 && tid < n ? ids_s[tid * top_k + picked] : 0;
        const unsigned long long bad = __ballot(tid >= 1 && tid < n && (chosen < 0 || chosen >= n_pred_rows));
        const int last = bad ? __builtin_ctzll(bad) : n - 1;
        if (page && tid < n) page[tid] = tid == 0 ? ids_s[0] : tid <= last ? chosen : out[tid];
        if (tid >= 1 && tid <= last) out[tid] = chosen;
        if (bad && tid == 0) *status = 1;
        return;
    }
    if (tid != 0) return;
    int prev_a = 0;  // which candidate of the previous position was picked (the carry token's scores sit in row 0)
    for (int pos = 1; pos < n; pos++) {
        const float *score = table_s + (static_cast<size_t>(pos - 1) * top_k + prev_a) * top_k;
        const int32_t *cands = ids_s + pos * top_k;
        int best_b = 0;
        {
            // scores of skipped candidates are -inf; the "tokens" of the distribution are candidate indices
            uint64_t keys[kSelMaxTopK];
            int nan_at = -1;
            for (int b = 0; b < top_k; b++) {
                const int32_t cand = cands[b];
                const float sc = (cand < 0 || cand >= n_succ_rows) ? -INFINITY : score[b];
                if (sc != sc && nan_at < 0) nan_at = b;
                const uint64_t key = cand_key(static_cast<uint32_t>(b), sc);
                int j = b;  // insertion sort, ascending keys = best first
                while (j > 0 && keys[j - 1] > key) {
                    keys[j] = keys[j - 1];
                    j--;
                }
                keys[j] = key;
            }
            dist.err = 0;
            if (nan_at >= 0) {
                dist.err = DFLASH_ERR_NAN_LOGIT;
            } else {
                ChainCfg cc = {};
                cc.temperature = temperature;
                cc.top_p = 1.0f;
                cc.min_p = 0.0f;
                cc.k = top_k;
                run_chain(keys, top_k, cc, &dist);
            }
            if (dist.err) {
                sampled->status = dist.err;
                sampled->err_pos = pos;
                *status = dist.err;
                return;  // sampler error: the walk stops
            }
            const int idx = pick_index(dist.weights, dist.n_keep, uniforms[pos - 1] * dist.total);
            best_b = dist.tokens[idx];
            sampled->n_sampled = pos;
            int cnt = 0;
            for (int i = 0; i < dist.n_keep; i++) {
                if (!(dist.weights[i] > 0.0)) continue;
                dflash_weighted_candidate &wc = sampled->cands[(pos - 1) * top_k + cnt++];
                wc.token = cands[dist.tokens[i]];
                wc.weight = dist.weights[i];
            }
            sampled->counts[pos - 1] = cnt;
        }
        const int32_t chosen = cands[best_b];
        out[pos] = chosen;
        if (chosen < 0 || chosen >= n_pred_rows) {
            *status = 1;
            if (SAMPLED) {
                sampled->status = 1;
                sampled->err_pos = pos;
            }
            return;
        }
        prev_a = best_b;
    }
}

// Both launches of a walk: the score table ((n - 1) x top_k x top_k floats of context workspace behind *ws_off), then
// the walk itself.
template <bool SAMPLED>
int32_t launch_walk(dflash_ctx *ctx, size_t *ws_off, const Codebook &pc, const Codebook &sc, int top_k, int rank, int carry, int n,
                    const int32_t *ids, const float *vals, const float *sel_h, int32_t *out, int32_t *status, float temperature,
                    const double *uniforms, SampledOut *sampled, hipStream_t st, int32_t *page = nullptr) {
    float *table = dfl_ws_take<float>(ctx, ws_off, static_cast<size_t>(15) * kSelMaxTopK * kSelMaxTopK * sizeof(float));
    if (!table) return dfl_fail(ctx, DFLASH_ERR_WORKSPACE, "select_draft_path: workspace too small");
    if (n > 1) {
        // (decoded rows as floats + the same rows' bytes)
        const size_t lds = sel_decoded_floats(top_k, rank) * sizeof(float) + sel_raw_pred_bytes(pc.row_bytes) +
                           static_cast<size_t>(top_k) * sel_raw_succ_stride(sc.row_bytes);
        if (pc.row_bytes % 2 || sc.row_bytes % 2 || reinterpret_cast<uintptr_t>(pc.data) % 2 || reinterpret_cast<uintptr_t>(sc.data) % 2)
            return dfl_fail(ctx, DFLASH_ERR_ALIGNMENT, "select_draft_path: codebook rows must start on 2-byte boundaries");
        if (lds > 48 * 1024) {
            if (const int32_t rc_ = dfl_raise_lds_limit(ctx, reinterpret_cast<const void *>(dflash2_scores_kernel), lds)) return rc_;
        }
        auto rows = [](int64_t n_rows) { return static_cast<uint32_t>(std::min<int64_t>(n_rows, int64_t(1) << 31)); };  // (tokens are below 2^31)
        dflash2_scores_kernel<<<dim3(top_k, n - 1), kScoreThreads, lds, st>>>(ids, pc.data, sc.data, sel_h, carry, top_k, rank, rows(pc.n_rows),
                                                                             rows(sc.n_rows), static_cast<int>(pc.row_bytes),
                                                                             static_cast<int>(sc.row_bytes), pc.type, sc.type, vals, table);
    }
    dflash2_select_kernel<SAMPLED><<<1, kSelThreads, 0, st>>>(pc.n_rows, sc.n_rows, top_k, carry, n, ids, table, out, status, temperature,
                                                               uniforms, sampled, page);
    DFL_HIP_CHECK(ctx, hipGetLastError());
    return DFLASH_OK;
}

int32_t check_codebook(dflash_ctx *ctx, const dflash_codebook *cb, int rank, Codebook *out, const char *what) {
    if (!cb || !cb->data || cb->n_rows < 1) return dfl_fail(ctx, DFLASH_ERR_INVALID_INPUT, "select_draft_path: %s codebook", what);
    size_t rb = 0;
    switch (cb->type) {
    case DFLASH_TYPE_F32: rb = static_cast<size_t>(rank) * 4; break;
    case DFLASH_TYPE_F16: rb = static_cast<size_t>(rank) * 2; break;
    case DFLASH_TYPE_Q8_0:
    case DFLASH_TYPE_Q4_K: rb = dflash_row_bytes(cb->type, rank); break;
    default: break;
    }
    if (rb == 0)
        return dfl_fail(ctx, DFLASH_ERR_UNSUPPORTED, "select_draft_path: %s codebook type %d with rank %d", what, cb->type, rank);
    *out = Codebook{cb->type, rank, cb->n_rows, static_cast<const uint8_t *>(cb->data), rb};
    return DFLASH_OK;
}

}  // namespace

extern "C" int32_t dflash_dflash2_conv(dflash_ctx *ctx, const float *x, const float *dyn, const float *base, float *y,
                                       int32_t n_tokens, int32_t h, int32_t kernel_size, int32_t group_size, int32_t side,
                                       dflash_stream_t stream) {
    return dfl_dflash2_conv(ctx, x, dyn, base, y, n_tokens, h, kernel_size, group_size, side, stream, nullptr, DFL_XF_NONE);
}

int32_t dfl_dflash2_conv(dflash_ctx *ctx, const float *x, const float *dyn, const float *base, float *y, int32_t n_tokens, int32_t h,
                         int32_t kernel_size, int32_t group_size, int32_t side, dflash_stream_t stream, void *y_xf, int y_xf_kind) {
    if (!ctx) return DFLASH_ERR_INVALID_INPUT;
    if (y_xf && (h % DFL_QK_K || n_tokens > 16 || (y_xf_kind != DFL_XF_Q4K && y_xf_kind != DFL_XF_Q6K)))
        return dfl_fail(ctx, DFLASH_ERR_BAD_SHAPE, "dflash2_conv: fragment-order output needs h %% 256 == 0, at most 16 rows and a kind");
    if (!x || !dyn || !base || !y) return dfl_fail(ctx, DFLASH_ERR_INVALID_INPUT, "dflash2_conv: null pointer");
    if (n_tokens < 1 || h < 1 || kernel_size < 1 || group_size < 1 || h % group_size || (side != 0 && side != 1))
        return dfl_fail(ctx, DFLASH_ERR_BAD_SHAPE, "dflash2_conv: n_tokens %d h %d kernel %d group %d side %d", n_tokens, h,
                        kernel_size, group_size, side);
    const size_t bytes = static_cast<size_t>(n_tokens) * h * sizeof(float);
    if (dfl_ranges_overlap(y, bytes, x, bytes))
        return dfl_fail(ctx, DFLASH_ERR_ALIAS, "dflash2_conv: y aliases x (taps read neighbouring rows)");
    // c * ceil(2^32 / g) >> 32 is c / g while c * g stays below 2^32
    const uint32_t by_group = group_size > 1 && static_cast<int64_t>(h) * group_size < (1ll << 32)
                                  ? static_cast<uint32_t>(((1ull << 32) + group_size - 1) / group_size) : 0;
    dflash2_conv_kernel<<<dim3(n_tokens, (h + 255) / 256), 256, 0, static_cast<hipStream_t>(stream)>>>(
        x, dyn, base, h, kernel_size, h / group_size, by_group, side, group_size, y, y_xf, y_xf_kind);
    DFL_HIP_CHECK(ctx, hipGetLastError());
    return DFLASH_OK;
}

extern "C" int32_t dflash_select_draft_path(dflash_ctx *ctx, const dflash_codebook *predecessor,
                                            const dflash_codebook *successor, int32_t rank, int32_t top_k, int32_t carry_token,
                                            int32_t n, const int32_t *topk_ids, const float *topk_vals, const float *sel_h,
                                            int32_t *out_tokens, int32_t *out_tokens_host, dflash_stream_t stream) {
    return dfl_select_draft_path(ctx, predecessor, successor, rank, top_k, carry_token, n, topk_ids, topk_vals, sel_h, out_tokens, out_tokens_host,
                                 nullptr, stream);
}

int32_t dfl_select_draft_path(dflash_ctx *ctx, const dflash_codebook *predecessor, const dflash_codebook *successor, int32_t rank, int32_t top_k,
                              int32_t carry_token, int32_t n, const int32_t *topk_ids, const float *topk_vals, const float *sel_h, int32_t *out_tokens,
                              int32_t *out_tokens_host, int32_t *page, dflash_stream_t stream) {
    if (!ctx) return DFLASH_ERR_INVALID_INPUT;
    if (!topk_ids || !topk_vals || !sel_h || !out_tokens)
        return dfl_fail(ctx, DFLASH_ERR_INVALID_INPUT, "select_draft_path: null pointer");
    if (n < 1 || n > 16 || top_k < 1 || top_k > kSelMaxTopK || rank < 1 || rank > kSelMaxRank)
        return dfl_fail(ctx, DFLASH_ERR_BAD_SHAPE, "select_draft_path: n %d top_k %d rank %d", n, top_k, rank);
    Codebook pc, sc;
    int32_t rc;
    if ((rc = check_codebook(ctx, predecessor, rank, &pc, "predecessor"))) return rc;
    if ((rc = check_codebook(ctx, successor, rank, &sc, "successor"))) return rc;
    size_t off = 0;
    int32_t *status = dfl_ws_take<int32_t>(ctx, &off, sizeof(int32_t));
    if (!status) return dfl_fail(ctx, DFLASH_ERR_WORKSPACE, "select_draft_path: workspace too small");
    hipStream_t st = static_cast<hipStream_t>(stream);
    if ((rc = launch_walk<false>(ctx, &off, pc, sc, top_k, rank, carry_token, n, topk_ids, topk_vals, sel_h, out_tokens, status, 0.0f,
                                 nullptr, nullptr, st, page)))
        return rc;
    if (out_tokens_host) {
        // the blocking form also reports an invalid predecessor row, as the reference's CPU walk does
        int32_t status_host = 0;
        DFL_HIP_CHECK(ctx, hipMemcpyAsync(out_tokens_host, out_tokens, n * sizeof(int32_t), hipMemcpyDeviceToHost, st));
        DFL_HIP_CHECK(ctx, hipMemcpyAsync(&status_host, status, sizeof(int32_t), hipMemcpyDeviceToHost, st));
        DFL_HIP_CHECK(ctx, hipStreamSynchronize(st));
        if (status_host) return dfl_fail(ctx, DFLASH_ERR_INVALID_TOKEN, "select_draft_path: selector codebook row out of range");
    }
    return DFLASH_OK;
}

extern "C" int32_t dflash_select_draft_path_sampled(dflash_ctx *ctx, const dflash_codebook *predecessor,
                                                    const dflash_codebook *successor, int32_t rank, int32_t top_k,
                                                    int32_t carry_token, int32_t n, const int32_t *topk_ids,
                                                    const float *topk_vals, const float *sel_h,
                                                    dflash_sampler *proposal_sampler, int32_t *out_tokens_host,
                                                    int32_t *prop_counts_host, dflash_weighted_candidate *prop_cands_host,
                                                    dflash_stream_t stream) {
    if (!ctx) return DFLASH_ERR_INVALID_INPUT;
    if (!topk_ids || !topk_vals || !sel_h || !proposal_sampler || !out_tokens_host || !prop_counts_host || !prop_cands_host)
        return dfl_fail(ctx, DFLASH_ERR_INVALID_INPUT, "select_draft_path_sampled: null pointer");
    if (n < 1 || n > 16 || top_k < 1 || top_k > kSelMaxTopK || rank < 1 || rank > kSelMaxRank)
        return dfl_fail(ctx, DFLASH_ERR_BAD_SHAPE, "select_draft_path_sampled: n %d top_k %d rank %d", n, top_k, rank);
    const dflash_sampling_config &pc_cfg = proposal_sampler->cfg;
    if (!(pc_cfg.temperature > 0.0f) || pc_cfg.top_k != 0 || pc_cfg.top_p != 1.0f || pc_cfg.min_p != 0.0f)
        return dfl_fail(ctx, DFLASH_ERR_INVALID_INPUT,
                        "select_draft_path_sampled: the proposal sampler must use temperature without target filters");
    Codebook pc, sc;
    int32_t rc;
    if ((rc = check_codebook(ctx, predecessor, rank, &pc, "predecessor"))) return rc;
    if ((rc = check_codebook(ctx, successor, rank, &sc, "successor"))) return rc;
    size_t off = 0;
    int32_t *status = dfl_ws_take<int32_t>(ctx, &off, sizeof(int32_t));
    int32_t *out_dev = dfl_ws_take<int32_t>(ctx, &off, 16 * sizeof(int32_t));
    double *uniforms = dfl_ws_take<double>(ctx, &off, 16 * sizeof(double));
    SampledOut *sampled = dfl_ws_take<SampledOut>(ctx, &off, sizeof(SampledOut));
    if (!status || !out_dev || !uniforms || !sampled)
        return dfl_fail(ctx, DFLASH_ERR_WORKSPACE, "select_draft_path_sampled: workspace too small");
    hipStream_t st = static_cast<hipStream_t>(stream);
    // one uniform per position, drawn ahead; the sampler is advanced afterwards by the draws actually made
    double u_host[16] = {0};
    if (n > 1) dflash_sampler_peek(proposal_sampler, n - 1, u_host);
    DFL_HIP_CHECK(ctx, hipMemcpyAsync(uniforms, u_host, sizeof(u_host), hipMemcpyHostToDevice, st));
    if ((rc = launch_walk<true>(ctx, &off, pc, sc, top_k, rank, carry_token, n, topk_ids, topk_vals, sel_h, out_dev, status,
                                pc_cfg.temperature, uniforms, sampled, st)))
        return rc;
    static_assert(sizeof(SampledOut) <= DFL_PINNED_BYTES, "the walk's result is read back through the context's pinned page");
    const SampledOut &host = *static_cast<const SampledOut *>(ctx->pinned);
    DFL_HIP_CHECK(ctx, hipMemcpyAsync(ctx->pinned, sampled, sizeof(SampledOut), hipMemcpyDeviceToHost, st));
    DFL_HIP_CHECK(ctx, hipMemcpyAsync(out_tokens_host, out_dev, n * sizeof(int32_t), hipMemcpyDeviceToHost, st));
    DFL_HIP_CHECK(ctx, hipStreamSynchronize(st));
    // every completed position consumed one draw, as each sample_with_distribution call commits its own
    dflash_sampler_advance(proposal_sampler, static_cast<uint64_t>(host.n_sampled));
    if (host.status == 1)
        return dfl_fail(ctx, DFLASH_ERR_INVALID_TOKEN, "select_draft_path_sampled: selector codebook row out of range at position %d",
                        host.err_pos);
    if (host.status) return dfl_fail(ctx, host.status, "select_draft_path_sampled: sampler error at position %d", host.err_pos);
    for (int p = 0; p + 1 < n; p++) {
        prop_counts_host[p] = host.counts[p];
        for (int i = 0; i < host.counts[p]; i++) prop_cands_host[p * top_k + i] = host.cands[p * top_k + i];
    }
    return DFLASH_OK;
}
