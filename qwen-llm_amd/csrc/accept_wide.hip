// Sampler chain for wide candidate sets: top_k = 0 (the whole vocabulary) or top_k above the 64
// candidates the selection kernels of accept.hip keep per row.
//
// Reference: sampling.rs:1198-1214 and 1273-1296 (full order: stable radix sort of the logit half of
// the (descending logit bits, token) keys; top_k < len: the top_k smallest keys, sorted), chain
// sampling.rs:1541-1615.
//
// Two ways.  A set of at most kPickMax candidates (the chat preset's 200) is selected, not sorted: a workgroup per
// 8192 tokens finds its own k smallest keys, a workgroup per row the k smallest of those, ranks them by counting and
// runs the chain with a candidate per thread.  Two launches that read the logits once, each bound
// by its chain of barriers and LDS round trips (the logits take 2 us): 16 rows x 151936 tokens, k = 200: 8.4 + 9.4 us
// where the sort, its 17 clears and its chain take 316; the whole call 334 -> 38 us.
// (Of a vocabulary that a mask has left one token in a thousand of, most words are alike: 13.8 + 15.8 us.)
// Anything larger (the whole vocabulary) is ordered by ONE device-wide radix sort: a key is
//   row << 60 | descending_logit_bits << 28 | token          (token < 2^28, row < 16)
// and ascending key order is (row, descending logit in f32 total order, ascending token id): row r's
// candidates end up, best first, at [r * vocab, (r + 1) * vocab).  All 64 bits are sorted (tokens are
// unique, so this is the reference's stable sort of the logit half; the library's sort over a sub-range of
// bits returned unsorted output for inputs of 4 k to 100 k keys on ROCm 7.2, checked against a host sort,
// while the full-width sort is correct at every size).  The sort itself is
// rocPRIM's radix_sort_keys (a plain library routine on a cold path; the streaming kernels of the hot
// path are in accept.hip).  The chain then runs per row on one workgroup: what is order-free (the
// min-p / +inf prefix lengths, the exponentials) is done by all threads, every sum that is compared
// with a uniform draw is the reference's sequential f64 fold, fed through LDS a tile at a time so
// that the one adding thread never waits on memory.
#include "common.h"
#include "sampler_chain.h"

#include <algorithm>
#include <cstring>

#include <rocprim/device/device_radix_sort.hpp>

#include "accept_select.h"
#include "accept_wide.h"

namespace {

constexpr int kWideThreads = 1024;
constexpr int kWideTile = 4096;  // doubles staged in LDS per step of a sequential fold
constexpr int kNoNanW = 0x7fffffff;

__device__ __forceinline__ float wide_key_logit(uint64_t key) {
    const uint32_t asc = ~static_cast<uint32_t>(key >> kWideTokenBits);
    const uint32_t bits = (asc & 0x80000000u) ? (asc & 0x7fffffffu) : ~asc;
    return __uint_as_float(bits);
}

__global__ void __launch_bounds__(256)
    wide_keys_kernel(const float *__restrict__ logits, int64_t vocab, int64_t stride, uint64_t *__restrict__ keys,
                     int32_t *__restrict__ nan_first) {
    const int row = blockIdx.y;
    const int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
    if (i >= vocab) return;
    const float v = logits[row * stride + i];
    if (v != v) atomicMin(nan_first + row, static_cast<int32_t>(i));
    keys[row * vocab + i] = (static_cast<uint64_t>(row) << 60) |
                            (static_cast<uint64_t>(desc_bits(__float_as_uint(v))) << kWideTokenBits) | static_cast<uint64_t>(i);
}

// ------------------------------------------------------------------------------------------
// selection of up to kPickMax candidates
// ------------------------------------------------------------------------------------------
constexpr int kPickThreads = 512;
constexpr int kPickChunk = 8192;  // tokens per workgroup: 16 rows of 151936 are 304 workgroups, one round of two per CU
constexpr int kPickMax = 1024;    // threads of the row kernel: a candidate each
constexpr int kPickSlots = 16 * kPickMax;  // chunk winners of a row that its workgroup holds in registers

// The largest key of a row with at most this ordering word.
__device__ __forceinline__ uint64_t wide_bound(int row, uint32_t word) {
    const uint64_t bound = (static_cast<uint64_t>(row) << 60) | (static_cast<uint64_t>(word) << kWideTokenBits) | kWideTokenMask;
    return bound < kNoKey ? bound : kNoKey - 1;
}

template <int PER>
__device__ __forceinline__ uint64_t first_key(const uint64_t (&key)[PER]) {
    uint64_t first = kNoKey;
#pragma unroll
    for (int j = 0; j < PER; j++) first = key[j] < first ? key[j] : first;
    return first;
}

// A chunk's winners, the k best keys and at most cap >= k, in no order, at out[(row * n_chunks + chunk) * cap], filled up
// with kNoKey; the chunk's lowest NaN token.  The k-th best of the per-thread best words bounds every winner, and what is
// below it usually fits the slots (k = 200: about 250 keys); only where it does not, the threads' best keys bound them, and only where
// that does not do either, as many of all as fit are looked for.
__global__ void __launch_bounds__(kPickThreads)
    pick_chunk_kernel(const float *__restrict__ logits, int64_t vocab, int64_t stride, int k, int cap, uint64_t *__restrict__ out,
                      int32_t *__restrict__ nan_first) {
    constexpr int kPer = kPickChunk / kPickThreads;
    __shared__ KthShared<kPickThreads> sh;
    __shared__ int cnt[2], nan_sh;
    const int row = blockIdx.y, tid = threadIdx.x;
    const float *x = logits + row * stride;
    const int64_t base = static_cast<int64_t>(blockIdx.x) * kPickChunk + tid;
    float v[kPer];
#pragma unroll
    for (int j = 0; j < kPer; j++) v[j] = x[base + j * kPickThreads < vocab ? base + j * kPickThreads : vocab - 1];
    if (tid == 0) {
        cnt[0] = cnt[1] = 0;
        nan_sh = kNoNanW;
    }
    __syncthreads();
    uint64_t key[kPer];
    uint32_t best = 0xffffffffu;
#pragma unroll
    for (int j = 0; j < kPer; j++) {
        const int64_t i = base + j * kPickThreads;
        const bool nan = v[j] != v[j];
        if (i < vocab && nan) atomicMin(&nan_sh, static_cast<int32_t>(i));
        key[j] = i < vocab && !nan ? (static_cast<uint64_t>(row) << 60) |
                                         (static_cast<uint64_t>(desc_bits(__float_as_uint(v[j]))) << kWideTokenBits) | static_cast<uint64_t>(i)
                                   : kNoKey;
        best = min(best, static_cast<uint32_t>(key[j] >> kWideTokenBits));
    }
    const uint32_t word = block_kth_word(best, k, k + k / 8, sh);
    uint64_t bound = wide_bound(row, word);
    const int64_t at = static_cast<int64_t>(row) * gridDim.x + blockIdx.x;
    uint64_t *o = out + at * cap;
    compact_keys(key, bound, o, cap, &cnt[0]);
    __syncthreads();
    int n = cnt[0];
    if (n > cap) {
        bound = block_kth_first(first_key(key), best, word, bound, k, sh);
        __syncthreads();  // (the counters have been read)
        bound = block_kth<kPer>(key, bound, k, cap, sh);
        compact_keys(key, bound, o, cap, &cnt[1]);
        __syncthreads();
        n = cnt[1];
    }
    for (int i = n + tid; i < cap; i += kPickThreads) o[i] = kNoKey;
    if (tid == 0) nan_first[at] = nan_sh;
}

// One row: the k best of its chunks' winners (n_chunks * cap <= PER * kPickMax slots), ranked by counting, then
// wide_chain_kernel's chain with a candidate per thread.  The kept candidates go to keys_out / weights [row * k ..].
template <int PER>
__global__ void __launch_bounds__(kPickMax)
    pick_row_kernel(const uint64_t *__restrict__ chunk_keys, const int32_t *__restrict__ chunk_nan, int n_chunks, int cap, ChainCfg cfg,
                    BlockWalk walk, RowDist *__restrict__ rows, uint64_t *__restrict__ keys_out, double *__restrict__ weights) {
    constexpr int kFold = 16;  // additions per round of the sum
    __shared__ KthShared<kPickMax> sh;
    __shared__ uint64_t cand[kPickMax], sorted[kPickMax];
    __shared__ alignas(16) double w_sh[kPickMax + kFold], upto[kPickMax];
    __shared__ int rank_sh[kPickMax];
    __shared__ int cnt[2], nan_sh;
    const int row = blockIdx.x, tid = threadIdx.x, k = cfg.k, n_in = n_chunks * cap;
    RowDist *d = rows + row;
    uint64_t key[PER];
    uint32_t best = 0xffffffffu;
#pragma unroll
    for (int j = 0; j < PER; j++) {
        const int i = j * kPickMax + tid;
        const uint64_t got = chunk_keys[static_cast<int64_t>(row) * n_in + (i < n_in ? i : 0)];
        key[j] = i < n_in ? got : kNoKey;
        best = min(best, static_cast<uint32_t>(key[j] >> kWideTokenBits));
    }
    const int nan = tid < n_chunks ? chunk_nan[row * n_chunks + tid] : kNoNanW;  // (n_chunks <= kPickSlots / k < kPickMax)
    rank_sh[tid] = 0;
    if (tid == 0) {
        cnt[0] = cnt[1] = 0;
        nan_sh = kNoNanW;
    }
    __syncthreads();
    if (nan != kNoNanW) atomicMin(&nan_sh, nan);
    const uint32_t word = block_kth_word(best, k, k + k / 8, sh);  // (its barriers are behind the minimum)
    uint64_t bound = wide_bound(row, word);
    auto finish = [&](int32_t err, int64_t err_index, int n_keep, double total, int32_t pick, double draft_weight) {
        if (tid == 0) {
            d->n_keep = n_keep;
            d->err = err;
            d->err_index = err_index;
            d->total = total;
            d->pick = pick;
            d->draft_weight = draft_weight;
            d->d_err = 0;
            d->d_err_index = -1;
        }
    };
    if (nan_sh != kNoNanW) return finish(DFLASH_ERR_NAN_LOGIT, nan_sh, 0, 0.0, 0, -0.0);
    compact_keys(key, bound, cand, kPickMax, &cnt[0]);
    __syncthreads();
    int n = cnt[0];
    if (n > kPickMax) {
        bound = block_kth_first(first_key(key), best, word, bound, k, sh);
        __syncthreads();  // (the counters have been read)
        bound = block_kth<PER>(key, bound, k, kPickMax, sh);
        compact_keys(key, bound, cand, kPickMax, &cnt[1]);
        __syncthreads();
        n = cnt[1];
    }
    {
        // A wave takes a sixteenth of the list and counts, for four candidates a lane, those of it that are below them: an element is
        // read from LDS once for 256 candidates (each thread with one candidate and a longer slice: 2.2 us for 228 of them, 1.1 now).
        const int lane = tid & 63, per = (n + kPickMax / 64 - 1) / (kPickMax / 64), j0 = (tid >> 6) * per, j1 = min(n, j0 + per);
        for (int i0 = 0; i0 < n; i0 += 256) {
            uint64_t x[4];
            int c[4] = {0, 0, 0, 0};
#pragma unroll
            for (int u = 0; u < 4; u++) x[u] = cand[min(i0 + 64 * u + lane, n - 1)];
#pragma unroll 4
            for (int j = j0; j < j1; j++) {
                const uint64_t y = cand[j];
#pragma unroll
                for (int u = 0; u < 4; u++) c[u] += y < x[u];
            }
#pragma unroll
            for (int u = 0; u < 4; u++)
                if (c[u] && i0 + 64 * u + lane < n) atomicAdd(&rank_sh[i0 + 64 * u + lane], c[u]);
        }
    }
    __syncthreads();
    if (tid < n && rank_sh[tid] < k) sorted[rank_sh[tid]] = cand[tid];
    __syncthreads();
    n = min(n, k);
    const uint64_t mine = tid < n ? sorted[tid] : 0;
    const double l = tid < n ? static_cast<double>(wide_key_logit(mine)) : 0.0, l0 = static_cast<double>(wide_key_logit(sorted[0]));
    int len = n;
    if (cfg.min_p > 0.0f && isfinite(l0)) len = __syncthreads_count(tid < len && l >= l0 + cfg.ln_min_p);  // a prefix of the order
    if (len == 0) return finish(DFLASH_ERR_NO_CANDIDATES, -1, 0, 0.0, 0, -0.0);
    double w = 0.0;
    if (l0 == INFINITY) {
        len = __syncthreads_count(tid < len && l == INFINITY);
        w = tid < len ? 1.0 : 0.0;
    } else {
        const double temperature = static_cast<double>(cfg.temperature), max_logit = l0 / temperature;
        if (max_logit == -INFINITY) return finish(DFLASH_ERR_NO_CANDIDATES, -1, 0, 0.0, 0, -0.0);
        if (tid < len) w = exp(l / temperature - max_logit);  // (no logit is above the first, which is finite: at most 1)
    }
    w_sh[tid] = w;
    if (tid < len) {
        keys_out[static_cast<int64_t>(row) * k + tid] = mine;
        weights[static_cast<int64_t>(row) * k + tid] = w;
    }
    __syncthreads();
    if (tid >= 64) return;
    // Every sum of the chain is a prefix of one: the weights added in order, one after the other (from +0 or -0 is the
    // same, no weight is below +0), a round's elements asked for ahead of the round before it.
    {
        double acc = 0.0, r[kFold];
#pragma unroll
        for (int j = 0; j < kFold; j++) r[j] = w_sh[j];
        for (int base = 0; base < len; base += kFold) {
            double next[kFold];
#pragma unroll
            for (int j = 0; j < kFold; j++) next[j] = w_sh[base + kFold + j];
#pragma unroll
            for (int j = 0; j < kFold; j++) {
                acc += r[j];
                r[j] = acc;
            }
            if (tid == 0) {
#pragma unroll
                for (int j = 0; j < kFold; j++) upto[base + j] = r[j];
            }
#pragma unroll
            for (int j = 0; j < kFold; j++) r[j] = next[j];
        }
    }
    __builtin_amdgcn_s_waitcnt(0);
    __builtin_amdgcn_wave_barrier();
    auto first = [&](auto reached) {  // the first of [0, len) whose running sum does, or len - 1
        for (int base = 0; base < len; base += 64) {
            const uint64_t m = __builtin_amdgcn_ballot_w64(base + tid < len && reached(upto[base + tid < len ? base + tid : 0]));
            if (m) return base + static_cast<int>(__builtin_ctzll(m));
        }
        return len - 1;
    };
    if (cfg.top_p < 1.0f) {
        const double target = upto[len - 1] * static_cast<double>(cfg.top_p);
        len = first([&](double s) { return s >= target; }) + 1;
    }
    const double total = upto[len - 1];
    if (!(isfinite(total) && total > 0.0)) return finish(DFLASH_ERR_NO_CANDIDATES, -1, 0, 0.0, 0, -0.0);
    const double drawn = walk.uniforms[row] * total;
    const int at = first([&](double s) { return drawn < s; });
    double draft_weight = -0.0;
    for (int base = 0; base < len; base += 64) {  // (tokens are distinct: at most one is the draft)
        const uint64_t m = __builtin_amdgcn_ballot_w64(base + tid < len && row + 1 < walk.n_tokens &&
                                                       static_cast<int32_t>(sorted[base + tid] & kWideTokenMask) == walk.verified[row + 1]);
        if (m) draft_weight = w_sh[base + __builtin_ctzll(m)];
    }
    finish(0, -1, len, total, static_cast<int32_t>(sorted[at] & kWideTokenMask), draft_weight);
}

// ------------------------------------------------------------------------------------------
// the full order
// ------------------------------------------------------------------------------------------
__global__ void wide_init_kernel(int32_t *nan_first, int n) {
    if (static_cast<int>(threadIdx.x) < n) nan_first[threadIdx.x] = kNoNanW;
}

// workgroup-wide integer sum, result to every thread
__device__ int64_t block_sum_i64(int64_t v, int64_t *sh) {
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    __syncthreads();
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = v;
    __syncthreads();
    int64_t r = 0;
    for (int w = 0; w < static_cast<int>(blockDim.x >> 6); w++) r += sh[w];
    return r;
}

// The reference's `acc = start; for w in weights[..n] { acc += w }` by thread 0, weights staged through LDS.
// With use_stop the fold stops after the first element that brings the sum to >= stop_at (top-p; strict: above it, the
// categorical pick); *count is the number of elements added.  Returns the sum (to every thread).
__device__ double sequential_fold(const double *__restrict__ w, int64_t n, double start, bool use_stop, bool strict, double stop_at,
                                  int64_t *count, double *tile, double *bcast, int64_t *bcast_n, int *done) {
    if (threadIdx.x == 0) {
        *bcast = start;
        *bcast_n = 0;
        *done = 0;
    }
    __syncthreads();
    for (int64_t base = 0; base < n; base += kWideTile) {
        const int m = static_cast<int>(n - base < kWideTile ? n - base : kWideTile);
        for (int i = threadIdx.x; i < m; i += blockDim.x) tile[i] = w[base + i];
        __syncthreads();
        if (threadIdx.x == 0) {
            double acc = *bcast;
            int i = 0;
            for (; i < m; i++) {
                acc += tile[i];
                if (use_stop && (strict ? stop_at < acc : acc >= stop_at)) {
                    i++;
                    *done = 1;
                    break;
                }
            }
            *bcast = acc;
            *bcast_n += i;
        }
        __syncthreads();
        if (*done) break;
    }
    const double result = *bcast;
    if (count) *count = *bcast_n;
    __syncthreads();  // everyone has read the result before the next fold resets it
    return result;
}

// sampling.rs:1541-1615 on the ordered candidates of one row; weights[row * vocab + i] receives candidate i's weight
__global__ void __launch_bounds__(kWideThreads)
    wide_chain_kernel(const uint64_t *__restrict__ keys_sorted, int64_t vocab, ChainCfg cfg, BlockWalk walk,
                      const int32_t *__restrict__ nan_first, RowDist *__restrict__ rows, double *__restrict__ weights) {
    __shared__ double tile[kWideTile];
    __shared__ int64_t red[kWideThreads / 64];
    __shared__ double bcast;
    __shared__ int64_t bcast_n;
    __shared__ int done;
    const int row = blockIdx.x, tid = threadIdx.x;
    const uint64_t *keys = keys_sorted + static_cast<int64_t>(row) * vocab;
    double *w = weights + static_cast<int64_t>(row) * vocab;
    RowDist *d = rows + row;
    auto finish = [&](int32_t err, int64_t err_index, int64_t n_keep, double total) {
        if (tid == 0) {
            d->n_keep = static_cast<int32_t>(n_keep);
            d->err = err;
            d->err_index = err_index;
            d->total = total;
            d->d_err = 0;
            d->d_err_index = -1;
            d->pick = 0;
            d->draft_weight = -0.0;
        }
    };
    if (nan_first[row] != kNoNanW) return finish(DFLASH_ERR_NAN_LOGIT, nan_first[row], 0, 0.0);
    int64_t len = cfg.k < vocab ? cfg.k : vocab;  // top-k
    const double l0 = static_cast<double>(wide_key_logit(keys[0]));
    if (cfg.min_p > 0.0f && isfinite(l0)) {  // min-p, before the temperature: a prefix of the descending order
        const double threshold = l0 + cfg.ln_min_p;
        int64_t c = 0;
        for (int64_t i = tid; i < len; i += kWideThreads) c += static_cast<double>(wide_key_logit(keys[i])) >= threshold;
        len = block_sum_i64(c, red);
    }
    if (len == 0) return finish(DFLASH_ERR_NO_CANDIDATES, -1, 0, 0.0);
    bool all_inf = false;
    if (l0 == INFINITY) {  // only the +inf logits stay, with weight one each
        int64_t c = 0;
        for (int64_t i = tid; i < len; i += kWideThreads) c += wide_key_logit(keys[i]) == INFINITY;
        len = block_sum_i64(c, red);
        all_inf = true;
    }
    const double temperature = static_cast<double>(cfg.temperature);
    if (all_inf) {
        for (int64_t i = tid; i < len; i += kWideThreads) w[i] = 1.0;
    } else {
        const double max_logit = l0 / temperature;
        if (max_logit == -INFINITY) return finish(DFLASH_ERR_NO_CANDIDATES, -1, 0, 0.0);
        int64_t bad = 0;
        for (int64_t i = tid; i < len; i += kWideThreads) {
            const double wi = exp(static_cast<double>(wide_key_logit(keys[i])) / temperature - max_logit);
            bad += !isfinite(wi);
            w[i] = wi;
        }
        if (block_sum_i64(bad, red) != 0) return finish(DFLASH_ERR_NO_CANDIDATES, -1, 0, 0.0);
    }
    __syncthreads();  // the weights are read back by other threads below
    if (cfg.top_p < 1.0f) {
        const double total = sequential_fold(w, len, -0.0, false, false, 0.0, nullptr, tile, &bcast, &bcast_n, &done);
        const double target = total * static_cast<double>(cfg.top_p);
        int64_t keep = 0;
        sequential_fold(w, len, 0.0, true, false, target, &keep, tile, &bcast, &bcast_n, &done);
        len = keep < 1 ? 1 : keep;
    }
    const double total_weight = sequential_fold(w, len, -0.0, false, false, 0.0, nullptr, tile, &bcast, &bcast_n, &done);
    if (!(isfinite(total_weight) && total_weight > 0.0)) return finish(DFLASH_ERR_NO_CANDIDATES, -1, 0, 0.0);
    // what the decision takes from the row's order: the token its draw falls on, and the weight of its draft
    int64_t upto = 0;
    const double drawn = walk.uniforms[row] * total_weight;
    const double sum = sequential_fold(w, len, 0.0, true, true, drawn, &upto, tile, &bcast, &bcast_n, &done);
    finish(0, -1, len, total_weight);
    __syncthreads();  // (thread 0 has cleared the draft's weight)
    if (tid == 0) d->pick = static_cast<int32_t>(keys[(drawn < sum ? upto : len) - 1] & kWideTokenMask);
    if (row + 1 < walk.n_tokens)  // (tokens are distinct: at most one is the draft)
        for (int64_t i = tid; i < len; i += kWideThreads)
            if (static_cast<int32_t>(keys[i] & kWideTokenMask) == walk.verified[row + 1]) d->draft_weight = w[i];
}

}  // namespace

int32_t dfl_accept_wide_rows(dflash_ctx *ctx, const float *logits, int32_t n_rows, int64_t vocab, int64_t stride, const ChainCfg &cfg,
                             const BlockWalk &walk, RowDist *rows, size_t *ws_off, const uint64_t **keys_out, const double **weights_out,
                             int64_t *out_stride, hipStream_t st) {
    if (n_rows > 16 || vocab >= (int64_t(1) << kWideTokenBits))
        return dfl_fail(ctx, DFLASH_ERR_UNSUPPORTED, "accept_prefix: wide top-k needs <= 16 rows and a vocabulary below 2^28");
    // Selection where a thread can hold each candidate and a workgroup the winners of all of a row's chunks (k <= 862 at
    // 151936 tokens); the sort is the only one that has no such bound.
    const int64_t n_chunks = (vocab + kPickChunk - 1) / kPickChunk;
    if (cfg.k <= kPickMax && n_chunks * cfg.k <= kPickSlots) {
        const int cap = static_cast<int>(std::min<int64_t>(2 * cfg.k, kPickSlots / n_chunks));
        const size_t slots = static_cast<size_t>(n_chunks) * cap, kept = static_cast<size_t>(n_rows) * cfg.k;
        uint64_t *winners = dfl_ws_take<uint64_t>(ctx, ws_off, n_rows * slots * sizeof(uint64_t));
        int32_t *nans = dfl_ws_take<int32_t>(ctx, ws_off, n_rows * n_chunks * sizeof(int32_t));
        uint64_t *keys = dfl_ws_take<uint64_t>(ctx, ws_off, kept * sizeof(uint64_t));
        double *weights = dfl_ws_take<double>(ctx, ws_off, kept * sizeof(double));
        if (!winners || !nans || !keys || !weights)
            return dfl_fail(ctx, DFLASH_ERR_WORKSPACE,
                            "accept_prefix: top_k %lld over a vocabulary of %lld needs about %zu KB of context workspace",
                            static_cast<long long>(cfg.k), static_cast<long long>(vocab), (n_rows * slots + 2 * kept) * 8 >> 10);
        const int nc = static_cast<int>(n_chunks);
        pick_chunk_kernel<<<dim3(nc, n_rows), kPickThreads, 0, st>>>(logits, vocab, stride, cfg.k, cap, winners, nans);
        if (slots <= 8 * kPickMax)
            pick_row_kernel<8><<<n_rows, kPickMax, 0, st>>>(winners, nans, nc, cap, cfg, walk, rows, keys, weights);
        else
            pick_row_kernel<16><<<n_rows, kPickMax, 0, st>>>(winners, nans, nc, cap, cfg, walk, rows, keys, weights);
        DFL_HIP_CHECK(ctx, hipGetLastError());
        *keys_out = keys;
        *weights_out = weights;
        *out_stride = cfg.k;
        return DFLASH_OK;
    }
    const size_t n = static_cast<size_t>(n_rows) * static_cast<size_t>(vocab);
    uint64_t *keys_a = dfl_ws_take<uint64_t>(ctx, ws_off, n * sizeof(uint64_t));
    uint64_t *keys_b = dfl_ws_take<uint64_t>(ctx, ws_off, n * sizeof(uint64_t));
    double *weights = dfl_ws_take<double>(ctx, ws_off, n * sizeof(double));
    int32_t *nan_first = dfl_ws_take<int32_t>(ctx, ws_off, 16 * sizeof(int32_t));
    size_t tmp_bytes = 0;
    if (rocprim::radix_sort_keys(nullptr, tmp_bytes, keys_a, keys_b, n, 0, 64, st, false) != hipSuccess)
        return dfl_fail(ctx, DFLASH_ERR_HIP, "accept_prefix: radix sort size query failed");
    void *tmp = dfl_ws_take<char>(ctx, ws_off, tmp_bytes ? tmp_bytes : 1);
    if (!keys_a || !keys_b || !weights || !nan_first || !tmp)
        return dfl_fail(ctx, DFLASH_ERR_WORKSPACE,
                        "accept_prefix: top_k %lld over a vocabulary of %lld needs about %zu MB of context workspace",
                        static_cast<long long>(cfg.k), static_cast<long long>(vocab), (3 * n * 8 + tmp_bytes) >> 20);
    wide_init_kernel<<<1, 64, 0, st>>>(nan_first, n_rows);
    wide_keys_kernel<<<dim3(static_cast<unsigned>((vocab + 255) / 256), n_rows), 256, 0, st>>>(logits, vocab, stride, keys_a, nan_first);
    DFL_HIP_CHECK(ctx, rocprim::radix_sort_keys(tmp, tmp_bytes, keys_a, keys_b, n, 0, 64, st, false));
    wide_chain_kernel<<<n_rows, kWideThreads, 0, st>>>(keys_b, vocab, cfg, walk, nan_first, rows, weights);
    DFL_HIP_CHECK(ctx, hipGetLastError());
    *keys_out = keys_b;
    *weights_out = weights;
    *out_stride = vocab;
    return DFLASH_OK;
}
