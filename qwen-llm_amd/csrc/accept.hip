// Acceptance: row-wise argmax / top-k over logits, the sampler-v1 filter chain and the
// speculative couplings, and the accept-prefix block decision, on the GPU.
//
// Reference: kernels/elementwise.metal:1153-1359 (argmax family), kernels/dflash2.metal:73-170
// (top-16), crates/qwen-llm/src/sampling.rs (chain :1541-1615, couplings :692-790, ordering keys
// :1206-1235, RNG :1621-1670), crates/qwen-llm/src/metal_dflash/accept.rs:76-183 (block decision,
// CPU-only in the reference).
//
// Everything here is HBM-bound streaming over [rows][vocab] f32 plus O(top_k) arithmetic, and, at one block per
// call, a chain of latencies (a dependent launch, a trip to memory for what another XCD wrote, an LDS read) rather
// than a volume of work:
//  * a row is cut into chunks (8192 tokens for the argmax, 16384 for the top-k selection) so that rows x chunks
//    workgroups cover the chip in one round; each workgroup streams its chunk once with coalesced loads;
//  * order decisions use the reference's integer keys (descending f32 total order above ascending
//    token id), so the selected candidates and their order are exact, not approximately sorted;
//  * top-k of a chunk: a bound per wave on its share of the winners, the largest of those on all of them; only what is
//    below it is ranked, by counting (keys are distinct), not by sorting networks in LDS, whose every step is a workgroup barrier;
//  * everything that feeds a comparison with a uniform draw is f64 and added in the order of the reference's
//    loops; what is independent per candidate (conversions, exponentials) is done a candidate per lane;
//  * a block with dense draft proposals is three launches: selection of both logit tensors, the rows' chains with their
//    draws and draft weights together with the draft rows' tile sums, the decision (written straight to pinned host memory): 7.2 + 9.3 +
//    5.3 us at 16 rows of 151936 and k = 20 (14.3 + 13.1 + 13.2 with a digit search per chunk, a barrier per tree level and the
//    walk's scans in one wave; the whole call 57 -> 39 us).
#include "common.h"
#include "sampler_chain.h"
#include "accept_select.h"
#include "accept_wide.h"

#include <cmath>
#include <cstring>

namespace {

constexpr int kChunk = 8192;       // tokens per workgroup of the argmax / top-2 kernel
// Tokens per workgroup of the top-k selection.  A 16-row block with dense draft proposals is 31 rows: at 8192 tokens
// per workgroup that is 589 workgroups of 1024 threads, more than the chip holds at once (two per CU), and the kernel
// takes two rounds of a workgroup whose time is mostly latency; at 16384 it is 310 and one round.
constexpr int kSelChunk = 16384;
constexpr int kSelThreads = 1024;  // 16 tokens per thread
constexpr int kMaxRows = 16;
constexpr int kNoNan = 0x7fffffff;

// ------------------------------------------------------------------------------------------
// argmax_top2: IEEE comparisons, lowest index on ties, second value counts duplicates
// ------------------------------------------------------------------------------------------
struct Top2 {
    float v1;
    uint32_t i1;
    float v2;
};

__device__ __forceinline__ Top2 top2_merge(Top2 a, Top2 b) {
    if (b.v1 > a.v1 || (b.v1 == a.v1 && b.i1 < a.i1)) {
        Top2 t = a;
        a = b;
        b = t;
    }
    if (b.v1 > a.v2) a.v2 = b.v1;
    if (b.v2 > a.v2) a.v2 = b.v2;
    return a;
}

__device__ __forceinline__ Top2 top2_wave(Top2 t) {  // over a wave, in every lane
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        Top2 o;
        o.v1 = __shfl_xor(t.v1, off, 64);
        o.i1 = static_cast<uint32_t>(__shfl_xor(static_cast<int>(t.i1), off, 64));
        o.v2 = __shfl_xor(t.v2, off, 64);
        t = top2_merge(t, o);
    }
    return t;
}
// What bounds it and the launch that follows it: their chains (the merges are of maxima and of the lowest token among equals, so any order
// gives the same).  All of a thread's tokens are asked for at once, waves merge by lane moves; the last launch has a chunk a lane.
// With a tree through LDS and one thread a row behind it : this, medians of traces: a 16 x 151936 block by itself 6.0 + 4.6 : 6.5 + 2.6 us, one row
// 5.0 + 3.4 : 4.9 + 1.8; at the end of a verify of 16 rows 6.5 + 4.8 : 6.8 + 4.2.
__global__ void __launch_bounds__(kSelThreads)
    top2_chunk_kernel(const float *__restrict__ logits, int64_t vocab, int64_t stride, Top2 *__restrict__ part) {
    __shared__ Top2 sh[kSelThreads / 64];
    const int row = blockIdx.y, chunk = blockIdx.x;
    const float *x = logits + row * stride;
    const int64_t base = static_cast<int64_t>(chunk) * kChunk + threadIdx.x;
    float v[kChunk / kSelThreads];
#pragma unroll
    for (int j = 0; j < kChunk / kSelThreads; j++) v[j] = x[min(base + j * kSelThreads, vocab - 1)];
    Top2 t = {-INFINITY, 0xffffffffu, -INFINITY};
#pragma unroll
    for (int j = 0; j < kChunk / kSelThreads; j++) {
        const int64_t i = base + j * kSelThreads;  // (a thread's tokens ascend: among equals the first stands)
        if (i < vocab) {
            if (v[j] > t.v1 || (v[j] == t.v1 && t.i1 == 0xffffffffu)) {
                t.v2 = t.v1;
                t.v1 = v[j];
                t.i1 = static_cast<uint32_t>(i);
            } else if (v[j] > t.v2) {
                t.v2 = v[j];
            }
        }
    }
    t = top2_wave(t);
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = t;
    __syncthreads();
    if (threadIdx.x >= 64) return;
    t = top2_wave(threadIdx.x < kSelThreads / 64 ? sh[threadIdx.x] : Top2{-INFINITY, 0xffffffffu, -INFINITY});
    if (threadIdx.x == 0) part[row * gridDim.x + chunk] = t;
}

__global__ void __launch_bounds__(64) top2_final_kernel(const Top2 *__restrict__ part, int n_chunks, int32_t *__restrict__ idx, float *__restrict__ gap,
                                                        int32_t *page, const int32_t *__restrict__ also) {
    const int row = blockIdx.x, lane = threadIdx.x;
    Top2 t = {-INFINITY, 0xffffffffu, -INFINITY};
    for (int c = lane; c < n_chunks; c += 64) t = top2_merge(t, part[row * n_chunks + c]);
    t = top2_wave(t);
    if (lane != 0) return;
    const float d = t.v1 - t.v2;
    idx[row] = static_cast<int32_t>(t.i1);
    gap[row] = d;
    if (page) {
        page[row] = static_cast<int32_t>(t.i1);
        if (also) page[16 + row] = also[row];
        page[32 + row] = __float_as_int(d);
    }
}

// ------------------------------------------------------------------------------------------
// chunk selection: best K keys of a chunk (sorted), lowest NaN index, optional second row set
// ------------------------------------------------------------------------------------------
// A chunk's list is k keys, ascending, at out[(row * n_chunks + chunk) * k], filled up with kNoKey.  A chunk with a NaN has
// the lowest NaN's token id, with nothing above it, as its first key: that is below every candidate's key (only a NaN's
// bits order as 0), so the least key of a row says whether it holds a NaN and which.
__device__ __forceinline__ bool key_is_nan(uint64_t key) { return (key >> 32) == 0; }

// min over the workgroup of a key, result in the first wave
__device__ __forceinline__ uint64_t block_min_u64(uint64_t v, uint64_t *sh) {
    const int lane = threadIdx.x & 63, n_waves = blockDim.x >> 6;
    v = wave_min_u64(v);
    if (lane == 0) sh[threadIdx.x >> 6] = v;
    __syncthreads();
    return threadIdx.x < 64 ? wave_min_u64(lane < n_waves ? sh[lane] : kNoKey) : kNoKey;
}

// A chunk's tokens j * kSelThreads + tid, all asked for at once (past the vocabulary: its last token again).
constexpr int kSelPer = kSelChunk / kSelThreads;
__device__ __forceinline__ void load_chunk(const float *__restrict__ x, int vocab, int base, float (&v)[kSelPer]) {
#pragma unroll
    for (int j = 0; j < kSelPer; j++) v[j] = x[min(base + j * kSelThreads, vocab - 1)];
}

// the best key alone: greedy targets, and the largest logit of a draft row
__device__ __forceinline__ void best_of_chunk(const float *__restrict__ x, int vocab, uint64_t *__restrict__ out) {
    __shared__ uint64_t red[kSelThreads / 64];
    const int base = blockIdx.x * kSelChunk + threadIdx.x;
    float v[kSelPer];
    load_chunk(x, vocab, base, v);
    uint64_t best = kNoKey;
#pragma unroll
    for (int j = 0; j < kSelPer; j++) {
        const int i = base + j * kSelThreads;  // (a repeated last token is passed over: its key would be another token's)
        const uint64_t key = v[j] != v[j] ? static_cast<uint64_t>(i) : cand_key(static_cast<uint32_t>(i), v[j]);
        best = i < vocab && key < best ? key : best;
    }
    best = block_min_u64(best, red);
    if (threadIdx.x == 0) *out = best;
}

// The k best, without a sort and without finding the k-th: of every wave's 64 per-thread bests the m-th least ordering word,
// m = ceil(k / waves), bounds m of them, so the largest of the waves' bounds bounds at least k keys of the chunk, and few more
// than that (k = 20: about a hundred).  What is below it is ranked by counting the candidates below each, and the candidate of
// rank r < k is output r.  Keys are distinct (the token id is in the low bits), so ranks are too.  (The k-th of the threads' best keys
// digit by digit in every chunk was 4.7 of its workgroup's 11.3 us, the collecting of what it bounds another 1.8.)
// Where many tokens are below the bound (a vocabulary of which a mask has left a few; logits ordered by token, or alike), the
// k-th best of the threads' best keys is what bounds them, and with the winners no more than the kSelPer tokens of k threads.  From 512 on the
// ranking costs more than that search (logits that fall from token to token, k = 20, 960 below the bound: a call of 62 us, now 41).
// (16 rows of 151936, k = 20, one token in a thousand left: 14.8 us, 7.3 unmasked; a digit search over all of the tokens: about 110.)
__device__ __forceinline__ void select_chunk_body(const float *__restrict__ x, int vocab, int k, uint64_t *__restrict__ out,
                                                  bool nan_is_candidate) {
    __shared__ uint64_t cand[kSelThreads];
    __shared__ KthShared<kSelThreads> kth;
    __shared__ int rank_sh[kSelThreads];
    __shared__ uint32_t bounds[kSelThreads / 64];
    __shared__ int cnt[2];
    __shared__ int nan_sh;
    constexpr int kWaves = kSelThreads / 64;
    static_assert(kSelPer * kMaxK <= kSelThreads, "the tokens of k threads are candidates of a thread each");
    const int tid = threadIdx.x, lane = tid & 63, base = blockIdx.x * kSelChunk + tid;
    float v[kSelPer];
    load_chunk(x, vocab, base, v);
    rank_sh[tid] = 0;
    if (tid == 0) {
        cnt[0] = cnt[1] = 0;
        nan_sh = kNoNan;
    }
    // (a token that is no candidate orders last; so does one NaN, which is why the collecting asks for the token, too)
    uint32_t d[kSelPer], best = 0xffffffffu;
    int nan_first = kNoNan;
#pragma unroll
    for (int j = 0; j < kSelPer; j++) {
        const int i = base + j * kSelThreads;
        const bool nan = v[j] != v[j];
        d[j] = i < vocab && (nan_is_candidate || !nan) ? desc_bits(__float_as_uint(v[j])) : 0xffffffffu;
        nan_first = nan && i < vocab ? min(nan_first, i) : nan_first;
        best = min(best, d[j]);
    }
    {
        uint32_t left = best, least = 0xffffffffu;
        for (int m = 0; m < k; m = kWaves * __popcll(__builtin_amdgcn_ballot_w64(best <= least))) {
            least = wave_min_u32(left);
            left = left == least ? 0xffffffffu : left;
        }
        if (lane == 0) bounds[tid >> 6] = least;
    }
    __syncthreads();
    if (!nan_is_candidate && nan_first != kNoNan) atomicMin(&nan_sh, nan_first);
    const uint32_t bound = wave_max_u32(lane < kWaves ? bounds[lane] : 0);
    // a thread with candidates asks for their slots at once (a bound above every number: all that are tokens)
    auto collect = [&](auto is_candidate) {
        int n = 0;
#pragma unroll
        for (int j = 0; j < kSelPer; j++) n += is_candidate(j);
        int at = n ? atomicAdd(&cnt[0], n) : 0;
#pragma unroll
        for (int j = 0; j < kSelPer; j++) {
            if (is_candidate(j)) {
                if (at < kSelThreads) cand[at] = (static_cast<uint64_t>(d[j]) << 32) | static_cast<uint32_t>(base + j * kSelThreads);
                at++;
            }
        }
    };
    if (bound == 0xffffffffu)
        collect([&](int j) { return base + j * kSelThreads < vocab; });
    else if (best <= bound)
        collect([&](int j) { return d[j] <= bound; });
    __syncthreads();
    int n_cand = cnt[0];
    if (n_cand > kSelThreads / 2) {
        uint64_t keys[kSelPer], first = kNoKey;
#pragma unroll
        for (int j = 0; j < kSelPer; j++) {
            const int i = base + j * kSelThreads;
            keys[j] = i < vocab ? (static_cast<uint64_t>(d[j]) << 32) | static_cast<uint32_t>(i) : kNoKey;
            first = keys[j] < first ? keys[j] : first;
        }
        const uint64_t limit = bound < 0xffffffffu ? (static_cast<uint64_t>(bound) << 32) | 0xffffffffu : kNoKey - 1;
        const uint64_t kth_key = block_kth_first(first, best, bound, limit, k, kth);
        compact_keys(keys, kth_key, cand, kSelThreads, &cnt[1]);
        __syncthreads();
        n_cand = cnt[1];
    }
    const bool nan_row = nan_sh != kNoNan;
    {
        // candidate i = tid % 2^log_n, 2^log_n >= n_cand, counts the candidates below it in slice tid / 2^log_n of the list
        const int log_n = n_cand > 1 ? 32 - __clz(n_cand - 1) : 0, log_slices = 10 - log_n, i = tid & ((1 << log_n) - 1);
        if (i < n_cand) {
            const int per = (n_cand + (1 << log_slices) - 1) >> log_slices, j0 = (tid >> log_n) * per, j1 = min(n_cand, j0 + per);
            const uint64_t key = cand[i];
            int c = 0;
#pragma unroll 4
            for (int j = j0; j < j1; j++) c += cand[j] < key;
            if (c) atomicAdd(&rank_sh[i], c);
        }
    }
    __syncthreads();
    if (tid < n_cand && rank_sh[tid] < k && !(nan_row && rank_sh[tid] == 0)) out[rank_sh[tid]] = cand[tid];
    if (tid < k && tid >= n_cand) out[tid] = kNoKey;
    if (tid == 0 && nan_row) out[0] = static_cast<uint64_t>(nan_sh);
}

__global__ void __launch_bounds__(kSelThreads, 8)
    select_chunk_kernel(const float *__restrict__ logits, int64_t stride, uint64_t *__restrict__ out, int vocab, int k, bool nan_is_candidate) {
    const int row = blockIdx.y;
    out += static_cast<int64_t>(row) * gridDim.x * k + blockIdx.x * k;
    if (k == 1)
        best_of_chunk(logits + row * stride, vocab, out);
    else
        select_chunk_body(logits + row * stride, vocab, k, out, nan_is_candidate);
}

// Two row sets in one launch: rows [0, n_a) of a (best k_a keys of every chunk), then the rows of b (best key).
__global__ void __launch_bounds__(kSelThreads, 8)
    select_pair_kernel(const float *__restrict__ a, const float *__restrict__ b, int64_t stride, uint64_t *__restrict__ out_a,
                       uint64_t *__restrict__ out_b, int vocab, int n_a, int k_a) {
    const int row = blockIdx.y;
    if (row >= n_a)
        best_of_chunk(b + (row - n_a) * stride, vocab, out_b + static_cast<int64_t>(row - n_a) * gridDim.x + blockIdx.x);
    else if (k_a == 1)
        best_of_chunk(a + row * stride, vocab, out_a + static_cast<int64_t>(row) * gridDim.x + blockIdx.x);
    else
        select_chunk_body(a + row * stride, vocab, k_a, out_a + (static_cast<int64_t>(row) * gridDim.x + blockIdx.x) * k_a, false);
}

// Number of keys below x in the ascending list of 1 <= n keys; step0 = the largest power of two <= n.
__device__ __forceinline__ int count_below(const uint64_t *list, int n, int step0, uint64_t x) {
    int below = 0;
    for (int step = step0; step >= 1; step >>= 1) {
        const int probe = below + step;
        const uint64_t v = list[min(probe, n) - 1];
        below = probe <= n && v < x ? probe : below;
    }
    return below;
}

// A lane's share of a draft row's chunk minima, and from the wave's lanes the row's largest logit, scaled; NaN where the row
// holds one, its token in *nan_token.
__device__ __forceinline__ uint64_t draft_best_of(const uint64_t *__restrict__ draft_best, int n_chunks, int row) {
    uint64_t best = kNoKey;
    for (int c = threadIdx.x & 63; c < n_chunks; c += 64) {
        const uint64_t key = draft_best[static_cast<int64_t>(row) * n_chunks + c];
        best = key < best ? key : best;
    }
    return best;
}
__device__ __forceinline__ double draft_max_scaled(uint64_t best, float draft_temperature, int *nan_token) {
    best = wave_min_u64(best);
    *nan_token = key_is_nan(best) ? key_token(best) : -1;
    return static_cast<double>(key_logit(best)) / static_cast<double>(draft_temperature);
}

// One workgroup per row: merge the chunk lists, order the best k, run the chain (wave 0, a candidate per lane).  With dense
// proposals the second wave takes the draft row's side (its maximum, its errors, the draft's own weight) and the first one, behind
// the chain, the draft row's weights of the kept candidates: what of the decision is independent per row and does not
// need the draft row's sum.
__device__ __forceinline__ void row_merge_body(const uint64_t *__restrict__ chunks, int n_chunks, const uint64_t *__restrict__ draft_best,
                                               const float *__restrict__ draft, int64_t draft_stride, int k, int n_tokens, const ChainCfg &cfg,
                                               const BlockWalk &walk, RowDist *__restrict__ rows, int32_t *__restrict__ greedy_out,
                                               bool draft_only, int row) {
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    RowDist *d = rows + row;
    const bool drafted = row + 1 < n_tokens, dense = draft_best && drafted;
    const int32_t draft_token = drafted ? walk.verified[row + 1] : -1;
    // the draft row's own side, by one wave: asked for ahead of the lists, worked out behind their merge
    const int draft_wave = draft_only ? 0 : 1;
    float draft_token_logit = 0.0f;
    uint64_t best_draft = kNoKey;
    auto draft_side = [&]() {
        int nan_token;
        const double mx = draft_max_scaled(best_draft, cfg.draft_temperature, &nan_token);
        const double q = exp(static_cast<double>(draft_token_logit) / static_cast<double>(cfg.draft_temperature) - mx);
        if (lane == 0) {
            d->d_err = nan_token >= 0 ? DFLASH_ERR_NAN_LOGIT : isfinite(mx) ? 0 : DFLASH_ERR_NO_CANDIDATES;
            d->d_err_index = nan_token;
            d->d_max_scaled = mx;
            d->q_draft = q;
        }
    };
    const int n_in = n_chunks * k;  // <= 2048, checked on the host
    uint64_t in0 = kNoKey, in1 = kNoKey;
    if (!draft_only) {
        const uint64_t *mine = chunks + static_cast<int64_t>(row) * n_in;
        in0 = mine[min(tid, n_in - 1)];
        in1 = mine[min(tid + kSelThreads, n_in - 1)];
    }
    if (dense && wave < 2) {
        if (wave == draft_wave) draft_token_logit = draft[row * draft_stride + draft_token];
        best_draft = draft_best_of(draft_best, n_chunks, row);
    }
    if (draft_only) {  // the target side of these rows was filled by the wide chain
        if (dense && wave == 0) draft_side();
        return;
    }
    // The chunks' lists are ascending: the rank of a key among all of them is the sum, over the lists, of the keys
    // below it (binary searches); the keys of rank < k, in rank order, are the row's candidates, best first.  Only keys up to the
    // largest of the full lists' m-th, m = ceil(k / lists), can be among them: those lists hold k keys up to there.
    // (Ranking all of the lists' keys: 3.2 us of the row's 6.8 at ten lists of 20.)
    __shared__ uint64_t sk[kMaxK];
    __shared__ uint64_t lists[2 * kSelThreads], cand[2 * kSelThreads];
    __shared__ int rank_sh[2 * kSelThreads];
    __shared__ uint64_t red[kSelThreads / 64];
    __shared__ int cnt;
    if (k == 1) {
        const uint64_t best = block_min_u64(min(in0, in1), red);
        if (tid == 0) sk[0] = best;
    } else {
        lists[tid] = in0;
        lists[tid + kSelThreads] = in1;
        rank_sh[tid] = rank_sh[tid + kSelThreads] = 0;
        if (tid < kMaxK) sk[tid] = kNoKey;
        if (tid == 0) cnt = 0;
        __syncthreads();
        const int n_full = n_chunks - (lists[n_in - 1] == kNoKey);
        uint32_t top = n_full ? 0 : 0xffffffffu;
        if (n_full) {
            const int m = (k + n_full - 1) / n_full;
            for (int c = lane; c < n_full; c += 64) top = max(top, static_cast<uint32_t>(lists[c * k + m - 1] >> 32));
            top = wave_max_u32(top);
        }
#pragma unroll
        for (int u = 0; u < 2; u++) {
            const int i = tid + u * kSelThreads;
            const uint64_t key = u ? in1 : in0;
            if (i < n_in && key != kNoKey && static_cast<uint32_t>(key >> 32) <= top) cand[atomicAdd(&cnt, 1)] = key;
        }
        __syncthreads();
        // (key, list) pairs: neighbouring threads take a key's lists
        const int n_cand = cnt, step0 = 1 << (31 - __clz(k)), log_c = n_chunks > 1 ? 32 - __clz(n_chunks - 1) : 0;  // n_chunks <= 2^log_c <= kSelThreads
        const int c = tid & ((1 << log_c) - 1);
        for (int i = tid >> log_c; i < n_cand && c < n_chunks; i += kSelThreads >> log_c) {
            const int below = count_below(lists + c * k, k, step0, cand[i]);
            if (below) atomicAdd(&rank_sh[i], below);
        }
        __syncthreads();
        for (int i = tid; i < n_cand; i += kSelThreads)
            if (rank_sh[i] < k) sk[rank_sh[i]] = cand[i];
    }
    __syncthreads();
    if (dense && wave == 1) draft_side();
    if (wave > 0) return;
    const uint64_t first = sk[0];
    const int nan_token = key_is_nan(first) ? key_token(first) : -1;
    if (greedy_out) {  // (the greedy argmax wants nothing else of the row)
        if (tid == 0) greedy_out[row] = nan_token >= 0 ? ~nan_token : key_token(first);
        return;
    }
    const uint64_t key = tid < k ? sk[tid < kMaxK ? tid : 0] : kNoKey;
    const int n_keys = __popcll(__builtin_amdgcn_ballot_w64(key != kNoKey));  // (missing keys sort last)
    const int32_t token = key != kNoKey ? key_token(key) : 0;
    float draft_logit = 0.0f;
    if (dense && nan_token < 0) draft_logit = draft[row * draft_stride + token];  // (used behind the chain)
    WaveChain ch = {0, 0.0, 0.0, 0.0};
    int32_t pick = 0;
    double draft_weight = -0.0;
    if (nan_token < 0) {
        if (cfg.temperature == 0.0f) {  // greedy target: one-hot on the total-order argmax (sampling.rs:391-400)
            ch = {1, 1.0, 1.0, 1.0};
            pick = key_token(first);
        } else {
            ch = run_chain_wave(key_logit(key), n_keys, cfg);
            if (ch.len) {
                const double drawn = walk.uniforms[row] * ch.total;
                pick = __builtin_amdgcn_readlane(token, wave_first(drawn < ch.upto, ch.len));
            }
        }
        const uint64_t at = __builtin_amdgcn_ballot_w64(drafted && lane < ch.len && token == draft_token);  // (tokens are distinct)
        if (at) draft_weight = chain_bcast(ch.w, static_cast<int>(__builtin_ctzll(at)));
    }
    if (dense && ch.len) {
        int none;
        const double mx = draft_max_scaled(best_draft, cfg.draft_temperature, &none);
        const double q = exp(static_cast<double>(draft_logit) / static_cast<double>(cfg.draft_temperature) - mx);
        if (lane < ch.len) d->q[lane] = q;
    }
    if (lane < ch.len) {
        d->tokens[lane] = token;
        d->weights[lane] = ch.w;
    }
    if (lane == 0) {
        d->n_keep = ch.len;
        d->err = nan_token >= 0 ? DFLASH_ERR_NAN_LOGIT : ch.len ? 0 : DFLASH_ERR_NO_CANDIDATES;
        d->err_index = nan_token;
        d->total = ch.total;
        d->pick = pick;
        d->draft_weight = draft_weight;
        if (!dense) {
            d->d_err = 0;
            d->d_err_index = -1;
        }
    }
}

__global__ void __launch_bounds__(kSelThreads)
    row_merge_kernel(const uint64_t *__restrict__ chunks, RowDist *__restrict__ rows, int32_t *__restrict__ greedy_out, int n_chunks, int k,
                     ChainCfg cfg, BlockWalk walk) {
    row_merge_body(chunks, n_chunks, nullptr, nullptr, 0, k, walk.n_tokens, cfg, walk, rows, greedy_out, false, blockIdx.x);
}

// top-16 output from the merged order
__global__ void __launch_bounds__(kSelThreads)
    top16_merge_kernel(const uint64_t *__restrict__ chunks, int n_chunks, int32_t *__restrict__ ids,
                       float *__restrict__ vals) {
    __shared__ uint64_t lists[2 * kSelThreads], sk[16];
    const int row = blockIdx.x, tid = threadIdx.x;
    const int n_in = n_chunks * 16;  // <= 2048, checked on the host
    for (int i = tid; i < n_in; i += kSelThreads) lists[i] = chunks[static_cast<int64_t>(row) * n_in + i];
    if (tid < 16) sk[tid] = kNoKey;
    __syncthreads();
    // a key's rank by counting the keys below it, sixteen lanes a key: a chunk's list each, sixteen chunks a round
    for (int i0 = 0; i0 < n_in; i0 += kSelThreads / 16) {
        const int i = i0 + (tid >> 4);
        const uint64_t key = i < n_in ? lists[i] : 0;
        int below = 0;
        for (int c = tid & 15; c < n_chunks; c += 16) {
#pragma unroll
            for (int j = 0; j < 16; j++) below += lists[16 * c + j] < key;
        }
        for (int off = 8; off > 0; off >>= 1) below += __shfl_xor(below, off, 64);
        if (i < n_in && (tid & 15) == 0 && key != kNoKey && below < 16) sk[below] = key;
    }
    __syncthreads();
    if (tid < 16) {
        uint64_t key = sk[tid];
        ids[row * 16 + tid] = key == kNoKey ? -1 : key_token(key);
        vals[row * 16 + tid] = key == kNoKey ? -INFINITY : key_logit(key);
    }
}

// The rows' chains and the dense proposal's tile sums in one launch (neither needs the other; both need only the
// chunk selection): of a row's workgroups the first is row_merge_kernel's, the rest take four 1024-token tiles each of its
// draft row.  A tile sum is the sum of exp(d/T - max/T) in a fixed shape: slot t of
// a tile holds ((e[4t]+e[4t+1])+e[4t+2])+e[4t+3], then a halving tree over the 256 slots; max is the row's largest
// draft logit, which every wave takes from the chunk minima itself, with its logits on their way.  The tree's two widest levels
// are one trip through LDS, the rest a wave's.  (A barrier per level and tile, and the logits asked for behind the maximum: 8.8 us of
// a workgroup.)
struct __attribute__((packed, aligned(4))) Logits4 {  // (rows start wherever the vocabulary puts them)
    float v[4];
};
__global__ void __launch_bounds__(kSelThreads)
    rows_and_tiles_kernel(const uint64_t *__restrict__ chunks, const float *__restrict__ draft, const uint64_t *__restrict__ draft_best,
                          double *__restrict__ tile_sums, int vocab, int n_chunks, int k, int n_tokens, float draft_temperature, int n_tiles,
                          RowDist *__restrict__ rows, bool draft_only, ChainCfg cfg, BlockWalk walk) {
    const int row = blockIdx.x;
    if (blockIdx.y == 0) {
        row_merge_body(chunks, n_chunks, draft_best, draft, vocab, k, n_tokens, cfg, walk, rows, nullptr, draft_only, row);
        return;
    }
    if (row == n_tokens - 1) return;  // (the last row has no draft)
    __shared__ double slot[4][256];
    const int tid = threadIdx.x, q = tid >> 8, t = tid & 255, tile0 = (blockIdx.y - 1) * 4, i = (tile0 + q) * 1024 + 4 * t;
    const float *x = draft + static_cast<int64_t>(row) * vocab;
    Logits4 in;
    if (i + 3 < vocab)
        in = *reinterpret_cast<const Logits4 *>(x + i);
    else
#pragma unroll
        for (int e = 0; e < 4; e++) in.v[e] = x[min(i + e, vocab - 1)];
    int nan_token;
    const double mx = draft_max_scaled(draft_best_of(draft_best, n_chunks, row), draft_temperature, &nan_token);
    // x / T as x * (1 / T) and one correction by the exact remainder: T and x have 24 bits, so the quotient is no closer than 2^-78
    // of itself to a value where rounding turns, and the corrected one is within 2^-104 of it before its own rounding.
    // (An infinite x has no remainder and stays as it is.)
    const double T = static_cast<double>(draft_temperature), inv_T = 1.0 / T;
    double acc = 0.0;
#pragma unroll
    for (int e = 0; e < 4; e++) {
        const double xe = static_cast<double>(in.v[e]), q0 = xe * inv_T, rem = __builtin_fma(-q0, T, xe);
        const double scaled = rem == rem ? __builtin_fma(rem, inv_T, q0) : q0;
        const double v = i + e < vocab ? exp(scaled - mx) : 0.0;
        acc = (e == 0) ? v : acc + v;
    }
    slot[q][t] = acc;
    __syncthreads();
    const int tile = tid >> 6, lane = tid & 63;  // a wave per tile
    if (tile >= 4) return;
    double sum = (slot[tile][lane] + slot[tile][lane + 128]) + (slot[tile][lane + 64] + slot[tile][lane + 192]);
#pragma unroll
    for (int s = 32; s >= 1; s >>= 1) sum += __shfl_xor(sum, s, 64);
    if (lane == 0 && tile0 + tile < n_tiles) tile_sums[row * n_tiles + tile0 + tile] = sum;
}

struct DecideArgs {
    int32_t n_stop;
    int64_t budget;
    // The block's small host inputs travel by value, in the kernel arguments: a pageable host-to-device copy
    // of a few bytes costs several microseconds of idle GPU each.
    BlockWalk walk;
    int32_t prop_offsets[kMaxRows], prop_counts[kMaxRows];  // sparse proposals: row r's candidates in prop_cands
    const int32_t *stop_ids;   // [n_stop]
    const dflash_weighted_candidate *prop_cands;
    // dense proposals
    const float *draft;
    int64_t draft_stride;
    float temperature, draft_temperature;
    // wide candidate sets (effective top-k above kMaxK): row r's kept candidates are the first n_keep ordered keys
    // / weights at r * wide_stride of these arrays instead of the arrays inside RowDist; null otherwise
    const uint64_t *wide_keys;
    const double *wide_w;
    int64_t wide_stride;
};

// What one row of the walk comes to, given that every row before it accepted.
struct RowOutcome {
    int32_t acc;         // the draft is accepted (draft rows only)
    int32_t stop;        // the draft is a stop id (draft rows only)
    int32_t token;       // correction token (rejected draft row) or bonus token (last row)
    int32_t draws;       // random draws this row consumes
    int32_t err;         // DFLASH_ERR_* of this row, 0 if none
    // wide sets: a rejected row's correction token is still to be drawn from the residual distribution
    // (residual_pick, for the one row the walk stops at)
    int32_t need_residual;
    int64_t err_index;
    double prop_total, u_residual;  // u_residual: the draw the pick uses
};

// One row of accept.rs:147-183 with the couplings of sampling.rs:692-790, by one whole wave.  A row that is reached has seen
// only accepting rows before it, and an accepting row consumes exactly one draw (none when greedy): row r therefore
// starts at draw r whatever the rows before it held, which is what lets every row be evaluated at once.
// rd: the row; token / p / q: lane i's candidate, its probability and its draft weight; target_probability: the draft's;
// u, u_residual: the row's draw and the one behind it; dense_total: the draft row's sum.
__device__ __forceinline__ RowOutcome decide_row(const DecideArgs &a, int mode, const RowDist &rd, int row, int32_t token, double p, double q,
                                                 double target_probability, double u, double u_residual, double dense_total) {
    RowOutcome o = {0, 0, 0, 0, 0, 0, -1, 0.0, 0.0};
    const int lane = threadIdx.x & 63, n_drafts = a.walk.n_tokens - 1;
    const bool greedy = a.temperature == 0.0f;
    if (row == n_drafts || mode == 0) {
        // bonus = sample(last reached row); deterministic coupling: draw the target token, accept iff it is the draft
        o.err = rd.err;
        o.err_index = rd.err_index;
        if (o.err) return o;
        o.token = rd.pick;
        o.draws = !greedy || a.wide_keys;
        o.acc = row < n_drafts && o.token == a.walk.verified[row + 1];
        return o;
    }
    const int32_t draft = a.walk.verified[row + 1];
    // proposal probability q(draft) and, per target candidate, q(candidate)
    double prop_total = 0.0, prop_tok_w = 0.0;
    const dflash_weighted_candidate *pc = a.prop_cands + a.prop_offsets[row];
    const int n_pc = a.prop_counts[row];
    if (mode == 1) {
        if (n_pc == 0) o.err = DFLASH_ERR_NO_CANDIDATES;
        for (int base = 0; base < n_pc && !o.err; base += 64) {
            const int m = min(64, n_pc - base);
            const int32_t t = lane < m ? pc[base + lane].token : -1;
            const double w = lane < m ? pc[base + lane].weight : 0.0;
            const uint64_t bad = __builtin_amdgcn_ballot_w64(!isfinite(w) || w < 0.0);
            if (bad) {
                o.err = DFLASH_ERR_INVALID_PROPOSAL_WEIGHT;
                o.err_index = __builtin_amdgcn_readlane(t, static_cast<int>(__builtin_ctzll(bad)));
                break;
            }
            prop_total = chain_bcast(wave_running_sum(prop_total, w, m), m - 1);
            for (uint64_t at = __builtin_amdgcn_ballot_w64(lane < m && t == draft); at; at &= at - 1)
                prop_tok_w += chain_bcast(w, static_cast<int>(__builtin_ctzll(at)));
        }
    } else {
        o.err = rd.d_err;
        o.err_index = rd.d_err_index;
        prop_total = dense_total;
        prop_tok_w = rd.q_draft;
    }
    if (!o.err && !(isfinite(prop_total) && prop_total > 0.0)) o.err = DFLASH_ERR_NO_CANDIDATES;
    if (!o.err && !(isfinite(prop_tok_w) && prop_tok_w > 0.0)) {
        o.err = DFLASH_ERR_MISSING_PROPOSAL_TOKEN;
        o.err_index = draft;
    }
    if (!o.err && rd.err) {
        o.err = rd.err;
        o.err_index = rd.err_index;
    }
    if (o.err) return o;
    const double proposal_probability = prop_tok_w / prop_total;
    const double acceptance = fmin(target_probability / proposal_probability, 1.0);
    if (u < acceptance) {
        o.acc = 1;
        o.draws = 1;
        return o;
    }
    // The correction token comes from the residual distribution: weights max(p_i - q_i, 0) in the target's order
    // (sampling.rs:752-790), and one more draw.  A candidate per lane; their running sums give the total and the pick.
    o.draws = 2;
    o.u_residual = u_residual;
    o.prop_total = prop_total;
    if (a.wide_keys) {
        o.need_residual = 1;
        return o;
    }
    if (mode == 1) {
        q = -0.0;
        for (int base = 0; base < n_pc; base += 64) {
            const int m = min(64, n_pc - base);
            const int32_t t = lane < m ? pc[base + lane].token : -1;
            const double w = lane < m ? pc[base + lane].weight : 0.0;
            for (int j = 0; j < m; j++) {
                const double wj = chain_bcast(w, j);
                if (__builtin_amdgcn_readlane(t, j) == token) q += wj;
            }
        }
    }
    const int n_keep = rd.n_keep;
    const double residual = lane < n_keep ? fmax(p - q / prop_total, 0.0) : 0.0;
    const double upto = wave_running_sum(0.0, residual, n_keep), residual_total = chain_bcast(upto, n_keep - 1);
    if (!(isfinite(residual_total) && residual_total > 0.0)) {
        o.err = DFLASH_ERR_NO_CANDIDATES;
        return o;
    }
    const double x = u_residual * residual_total;
    o.token = __builtin_amdgcn_readlane(token, wave_first(x < upto, n_keep));
    return o;
}

// The correction token of rejected row `row` where its candidates are a wide set, as in decide_row: the residual weights
// are summed first, then walked again for the pick; the second pass recomputes the same values,
// so no per-candidate array is needed.  By the whole wave: lane j computes the weight of candidate base + j (one f64
// exponential each under a dense proposal, the expensive part), and the sums add those values in candidate order,
// one addition after the other.
__device__ __forceinline__ void residual_pick(const DecideArgs &a, int mode, const RowDist &rd, int row, RowOutcome &o) {
    const int lane = threadIdx.x & 63;
    const uint64_t *keys = a.wide_keys + row * a.wide_stride;
    const double *weights = a.wide_w + row * a.wide_stride;
    const dflash_weighted_candidate *pc = mode == 1 ? a.prop_cands + a.prop_offsets[row] : nullptr;
    const int n_pc = mode == 1 ? a.prop_counts[row] : 0;
    const double prop_total = o.prop_total;
    auto token_at = [&](int i) { return static_cast<int32_t>(keys[i] & kWideTokenMask); };
    auto residual_at = [&](int i) {
        const double p = weights[i] / rd.total;
        double q;
        if (mode == 1) {
            const int32_t ti = token_at(i);
            double qs = -0.0;
            for (int j = 0; j < n_pc; j++)
                if (pc[j].token == ti) qs += pc[j].weight;
            q = qs / prop_total;
        } else {
            const float dl = a.draft[row * a.draft_stride + token_at(i)];
            q = exp(static_cast<double>(dl) / static_cast<double>(a.draft_temperature) - rd.d_max_scaled) / prop_total;
        }
        return fmax(p - q, 0.0);
    };
    const int n_keep = rd.n_keep;
    double residual_total = 0.0;
    for (int base = 0; base < n_keep; base += 64) {
        const double r = base + lane < n_keep ? residual_at(base + lane) : 0.0;
        const int m = min(64, n_keep - base);
        residual_total = chain_bcast(wave_running_sum(residual_total, r, m), m - 1);
    }
    if (!(isfinite(residual_total) && residual_total > 0.0)) {
        o.err = DFLASH_ERR_NO_CANDIDATES;
        return;
    }
    const double x = o.u_residual * residual_total;
    int pick = n_keep - 1;
    double cumulative = 0.0;
    for (int base = 0; base < n_keep; base += 64) {
        const double r = base + lane < n_keep ? residual_at(base + lane) : 0.0;
        const int m = min(64, n_keep - base);
        const double upto = wave_running_sum(cumulative, r, m);
        const uint64_t above = __builtin_amdgcn_ballot_w64(lane < m && x < upto);
        if (above) {
            pick = base + static_cast<int>(__builtin_ctzll(above));
            break;
        }
        cumulative = chain_bcast(upto, m - 1);
    }
    o.token = token_at(pick);
}

// Wave r evaluates row r (all rows at once); the first wave then finds the row at which the serial
// loop of accept.rs:147-183 stops: rows behind the first rejection, stop or error are never looked at.
// A chain of latencies: what the kernel reads was written by other XCDs and comes from memory at about two microseconds a
// trip, so everything is asked for at once, and a draft row's tile sums are 150 dependent additions.  (Rows walked by one wave, each
// scan over its candidates a loop over LDS, the exponentials and the residual of the row it stops at behind the walk: 13.2 us for
// a 16-row block with dense proposals.)
constexpr int kDecThreads = 64 * kMaxRows;
__global__ void __launch_bounds__(kDecThreads)
    decide_kernel(const RowDist *__restrict__ rows, const double *__restrict__ tile_sums, dflash_accept_decision *__restrict__ out, int mode,
                  int n_tiles, int n_tokens, DecideArgs a) {
    constexpr int kStage = 256, kAhead = 16;  // tile sums per row and round, and of those that are read ahead of their additions
    __shared__ double p_total[kMaxRows];
    __shared__ RowOutcome outcome[kMaxRows];
    // (a row's last read ahead is behind its sums, never used; a row per lane is read, two sums at a time: two more words a row make
    // the lanes' banks differ)
    __shared__ alignas(16) double staged[kMaxRows][kStage + kAhead + 2];
    static_assert(kStage % kAhead == 0 && sizeof(staged[0]) >= (kStage + kAhead) * sizeof(double), "the last read ahead stays in its row");
    const int tid = threadIdx.x, lane = tid & 63, row = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n_drafts = n_tokens - 1;
    const bool dense = mode == 2, live = row < n_tokens;
    const RowDist &rd = rows[live ? row : 0];
    double sums[kStage / 64];
#pragma unroll
    for (int j = 0; j < kStage / 64; j++) sums[j] = dense && row < n_drafts && 64 * j + lane < n_tiles ? tile_sums[row * n_tiles + 64 * j + lane] : 0.0;
    const int32_t token = rd.tokens[lane];
    const double weight = rd.weights[lane], q = rd.q[lane];
    const int draw = a.temperature == 0.0f || !live ? 0 : row;
    const double u = a.walk.uniforms[draw], u_residual = a.walk.uniforms[draw + 1];
    bool stop = false;
    if (row < n_drafts)
        for (int base = 0; base < a.n_stop; base += 64)
            stop = stop || __builtin_amdgcn_ballot_w64(base + lane < a.n_stop && a.stop_ids[base + lane < a.n_stop ? base + lane : 0] == a.walk.verified[row + 1]) != 0;
    const double total = rd.total, p = weight / total, target_probability = rd.draft_weight / total;  // (while the last wave adds)
    if (dense) {
        // P = sequential sum of a row's tile sums, in tile order, by lane r of the last wave (its own row has no draft) from the LDS copies
        double P = 0.0;
        for (int t0 = 0;; t0 += kStage) {
#pragma unroll
            for (int j = 0; j < kStage / 64; j++) staged[row][64 * j + lane] = sums[j];
            __syncthreads();
            if (row == kMaxRows - 1 && lane < n_drafts) {
                // (the next sixteen are read ahead of these sixteen's additions; past the last tile is +0, which changes no sum of
                // exponentials)
                const int n = min(kStage, n_tiles - t0);
                double v[kAhead], next[kAhead];
#pragma unroll
                for (int j = 0; j < kAhead; j++) v[j] = staged[lane][j];
                for (int i = 0; i < n; i += kAhead) {
#pragma unroll
                    for (int j = 0; j < kAhead; j++) next[j] = staged[lane][i + kAhead + j];
#pragma unroll
                    for (int j = 0; j < kAhead; j++) P += v[j];
#pragma unroll
                    for (int j = 0; j < kAhead; j++) v[j] = next[j];
                }
            }
            if (t0 + kStage >= n_tiles) break;  // (more rounds: vocabularies above 262144 tokens)
#pragma unroll
            for (int j = 0; j < kStage / 64; j++) {
                const int t = t0 + kStage + 64 * j + lane;
                sums[j] = row < n_drafts && t < n_tiles ? tile_sums[row * n_tiles + t] : 0.0;
            }
            __syncthreads();
        }
        if (row == kMaxRows - 1 && lane < n_drafts) p_total[lane] = P;
        __syncthreads();
    }
    if (live) {
        RowOutcome o = decide_row(a, mode, rd, row, token, p, q, target_probability, u, u_residual, dense && row < n_drafts ? p_total[row] : 0.0);
        o.stop = stop;
        if (lane == 0) outcome[row] = o;
    }
    __syncthreads();
    if (row > 0) return;
    // The decision is put together in LDS and
    // leaves as one coalesced store: `out` may be host memory, where every separate store is a transaction over the
    // bus.
    __shared__ dflash_accept_decision d_sh;
    static_assert(sizeof(dflash_accept_decision) % 4 == 0, "copied as words");
    constexpr int kWords = sizeof(dflash_accept_decision) / 4;
    static_assert(kWords <= 64, "a word per lane");
    const RowOutcome &mine = outcome[min(lane, n_drafts)];
    const int my_draws = mine.draws;
    const bool ends = lane >= n_drafts || mine.err || !mine.acc || mine.stop || lane + 1 == a.budget;
    const int at = static_cast<int>(__builtin_ctzll(__builtin_amdgcn_ballot_w64(ends)));
    RowOutcome o = outcome[at];
    if (o.need_residual) residual_pick(a, mode, rows[at], at, o);  // (its row has no error of its own)
    const uint64_t reached = (uint64_t(2) << at) - 1;
    const int draws = __popcll(__builtin_amdgcn_ballot_w64(my_draws & 1) & reached) + 2 * __popcll(__builtin_amdgcn_ballot_w64(my_draws & 2) & reached);
    const bool bonus = at == n_drafts, accepted_last = !bonus && o.acc;
    const int accepted = at + accepted_last, stop_reason = !accepted_last ? DFLASH_STOP_NONE : o.stop ? DFLASH_STOP_EOS : DFLASH_STOP_TOKEN_LIMIT;
    if (lane < kWords) reinterpret_cast<uint32_t *>(&d_sh)[lane] = 0;
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    if (lane < accepted && !o.err) d_sh.accepted_drafts[lane] = a.walk.verified[lane + 1];
    if (lane == 0) {
        d_sh.err_row = o.err ? at : -1;
        d_sh.err_index = o.err ? o.err_index : -1;
        d_sh.err_code = o.err;
        if (!o.err) {
            d_sh.n_accepted = accepted;
            d_sh.carry_kind = bonus ? DFLASH_CARRY_BONUS : accepted_last ? DFLASH_CARRY_NONE : DFLASH_CARRY_CORRECTION;
            d_sh.carry_token = accepted_last ? 0 : o.token;
            d_sh.stop_reason = stop_reason;
            d_sh.retain_input_count = 1 + accepted - (stop_reason != DFLASH_STOP_NONE ? 1 : 0);
            d_sh.draws_used = draws;
        }
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    if (lane < kWords) reinterpret_cast<uint32_t *>(out)[lane] = reinterpret_cast<const uint32_t *>(&d_sh)[lane];
}

// ------------------------------------------------------------------------------------------
// host: random streams (sampling.rs:1621-1670; Philox4x32-10 after Salmon et al.)
// ------------------------------------------------------------------------------------------
uint64_t splitmix_next(uint64_t &state) {
    state += 0x9e3779b97f4a7c15ull;
    uint64_t v = state;
    v = (v ^ (v >> 30)) * 0xbf58476d1ce4e5b9ull;
    v = (v ^ (v >> 27)) * 0x94d049bb133111ebull;
    return v ^ (v >> 31);
}
uint64_t rotl64(uint64_t x, int k) { return (x << k) | (x >> (64 - k)); }
uint64_t xoshiro_next(uint64_t s[4]) {
    uint64_t result = rotl64(s[0] + s[3], 23) + s[0];
    uint64_t t = s[1] << 17;
    s[2] ^= s[0];
    s[3] ^= s[1];
    s[1] ^= s[2];
    s[0] ^= s[3];
    s[2] ^= t;
    s[3] = rotl64(s[3], 45);
    return result;
}
void philox4x32_10(const uint32_t ctr[4], const uint32_t key[2], uint32_t out[4]) {
    uint32_t c0 = ctr[0], c1 = ctr[1], c2 = ctr[2], c3 = ctr[3], k0 = key[0], k1 = key[1];
    for (int r = 0; r < 10; r++) {
        uint64_t p0 = static_cast<uint64_t>(0xD2511F53u) * c0;
        uint64_t p1 = static_cast<uint64_t>(0xCD9E8D57u) * c2;
        uint32_t n0 = static_cast<uint32_t>(p1 >> 32) ^ c1 ^ k0, n1 = static_cast<uint32_t>(p1);
        uint32_t n2 = static_cast<uint32_t>(p0 >> 32) ^ c3 ^ k1, n3 = static_cast<uint32_t>(p0);
        c0 = n0;
        c1 = n1;
        c2 = n2;
        c3 = n3;
        k0 += 0x9E3779B9u;
        k1 += 0xBB67AE85u;
    }
    out[0] = c0;
    out[1] = c1;
    out[2] = c2;
    out[3] = c3;
}
uint64_t sampler_raw_next(dflash_sampler *s) {
    if (s->cfg.rng_kind == 1) {
        uint64_t pos = s->s[0]++;
        uint32_t ctr[4] = {static_cast<uint32_t>(pos), static_cast<uint32_t>(pos >> 32), 0, 0};
        uint32_t key[2] = {static_cast<uint32_t>(s->cfg.seed), static_cast<uint32_t>(s->cfg.seed >> 32)};
        uint32_t out[4];
        philox4x32_10(ctr, key, out);
        return static_cast<uint64_t>(out[0]) | (static_cast<uint64_t>(out[1]) << 32);
    }
    return xoshiro_next(s->s);
}

int32_t status_of_hip(hipError_t e) { return e == hipSuccess ? DFLASH_OK : DFLASH_ERR_HIP; }

int32_t check_rows(dflash_ctx *ctx, const char *what, const float *logits, int32_t n_rows, int64_t vocab,
                   int64_t stride) {
    if (!logits) return dfl_fail(ctx, DFLASH_ERR_INVALID_INPUT, "%s: null pointer", what);
    if (n_rows < 1 || n_rows > 4096) return dfl_fail(ctx, DFLASH_ERR_BAD_SHAPE, "%s: n_rows %d", what, n_rows);
    if (vocab < 1) return dfl_fail(ctx, DFLASH_ERR_EMPTY_LOGITS, "%s: empty logits row", what);
    if (vocab > 0x7fffffffll) return dfl_fail(ctx, DFLASH_ERR_VOCAB_TOO_LARGE, "%s: vocabulary %lld", what, static_cast<long long>(vocab));
    if (stride < vocab) return dfl_fail(ctx, DFLASH_ERR_BAD_SHAPE, "%s: stride %lld < vocab", what, static_cast<long long>(stride));
    return DFLASH_OK;
}

}  // namespace

int32_t dfl_argmax_top2(dflash_ctx *ctx, const float *logits, int32_t n_rows, int64_t vocab, int64_t stride, int32_t *idx, float *gap,
                        int32_t *page, const int32_t *also, hipStream_t st) {
    if (!ctx) return DFLASH_ERR_INVALID_INPUT;
    int32_t rc = check_rows(ctx, "argmax_top2", logits, n_rows, vocab, stride);
    if (rc) return rc;
    if (!idx || !gap) return dfl_fail(ctx, DFLASH_ERR_INVALID_INPUT, "argmax_top2: null output");
    const int n_chunks = static_cast<int>((vocab + kChunk - 1) / kChunk);
    size_t off = 0;
    Top2 *part = dfl_ws_take<Top2>(ctx, &off, sizeof(Top2) * n_rows * n_chunks);
    if (!part) return dfl_fail(ctx, DFLASH_ERR_WORKSPACE, "argmax_top2: workspace too small");
    dfl_timed timer(ctx, st, DFL_T_ARGMAX);
    top2_chunk_kernel<<<dim3(n_chunks, n_rows), kSelThreads, 0, st>>>(logits, vocab, stride, part);
    top2_final_kernel<<<n_rows, 64, 0, st>>>(part, n_chunks, idx, gap, page, also);
    DFL_HIP_CHECK(ctx, hipGetLastError());
    return DFLASH_OK;
}

extern "C" {

int32_t dflash_argmax_top2(dflash_ctx *ctx, const float *logits, int32_t n_rows, int64_t vocab, int64_t stride,
                           int32_t *idx, float *gap, dflash_stream_t stream) {
    return dfl_argmax_top2(ctx, logits, n_rows, vocab, stride, idx, gap, nullptr, nullptr, static_cast<hipStream_t>(stream));
}

int32_t dflash_argmax_greedy(dflash_ctx *ctx, const float *logits, int32_t n_rows, int64_t vocab, int64_t stride,
                             int32_t *idx, dflash_stream_t stream) {
    if (!ctx) return DFLASH_ERR_INVALID_INPUT;
    int32_t rc = check_rows(ctx, "argmax_greedy", logits, n_rows, vocab, stride);
    if (rc) return rc;
    if (!idx) return dfl_fail(ctx, DFLASH_ERR_INVALID_INPUT, "argmax_greedy: null output");
    hipStream_t st = static_cast<hipStream_t>(stream);
    const int n_chunks = static_cast<int>((vocab + kSelChunk - 1) / kSelChunk);
    if (n_chunks > 2 * kSelThreads) return dfl_fail(ctx, DFLASH_ERR_UNSUPPORTED, "argmax_greedy: vocabulary too large");
    size_t off = 0;
    uint64_t *chunks = dfl_ws_take<uint64_t>(ctx, &off, sizeof(uint64_t) * n_rows * n_chunks);
    if (!chunks) return dfl_fail(ctx, DFLASH_ERR_WORKSPACE, "argmax_greedy: workspace too small");
    ChainCfg cfg = {};
    cfg.k = 1;
    dfl_timed timer(ctx, st, DFL_T_ARGMAX);
    select_chunk_kernel<<<dim3(n_chunks, n_rows), kSelThreads, 0, st>>>(logits, stride, chunks, static_cast<int>(vocab), 1, false);
    row_merge_kernel<<<n_rows, kSelThreads, 0, st>>>(chunks, nullptr, idx, n_chunks, 1, cfg, BlockWalk{});
    DFL_HIP_CHECK(ctx, hipGetLastError());
    return DFLASH_OK;
}

int32_t dflash_top16(dflash_ctx *ctx, const float *logits, int32_t n_rows, int64_t vocab, int64_t stride,
                     int32_t *ids, float *vals, dflash_stream_t stream) {
    if (!ctx) return DFLASH_ERR_INVALID_INPUT;
    int32_t rc = check_rows(ctx, "top16", logits, n_rows, vocab, stride);
    if (rc) return rc;
    if (!ids || !vals) return dfl_fail(ctx, DFLASH_ERR_INVALID_INPUT, "top16: null output");
    hipStream_t st = static_cast<hipStream_t>(stream);
    const int n_chunks = static_cast<int>((vocab + kSelChunk - 1) / kSelChunk);
    if (n_chunks * 16 > 2 * kSelThreads) return dfl_fail(ctx, DFLASH_ERR_UNSUPPORTED, "top16: vocabulary too large");
    size_t off = 0;
    uint64_t *chunks = dfl_ws_take<uint64_t>(ctx, &off, sizeof(uint64_t) * 16 * n_rows * n_chunks);
    if (!chunks) return dfl_fail(ctx, DFLASH_ERR_WORKSPACE, "top16: workspace too small");
    dfl_timed timer(ctx, st, DFL_T_ARGMAX);
    select_chunk_kernel<<<dim3(n_chunks, n_rows), kSelThreads, 0, st>>>(logits, stride, chunks, static_cast<int>(vocab), 16, true);
    top16_merge_kernel<<<n_rows, kSelThreads, 0, st>>>(chunks, n_chunks, ids, vals);
    DFL_HIP_CHECK(ctx, hipGetLastError());
    return DFLASH_OK;
}

// sampling.rs:133-144, 346-366
int32_t dflash_sampler_init(dflash_sampler *s, const dflash_sampling_config *cfg) {
    if (!s || !cfg) return DFLASH_ERR_INVALID_INPUT;
    if (!std::isfinite(cfg->temperature) || cfg->temperature < 0.0f) return DFLASH_ERR_INVALID_TEMPERATURE;
    if (!std::isfinite(cfg->top_p) || !(0.0f < cfg->top_p && cfg->top_p <= 1.0f)) return DFLASH_ERR_INVALID_TOP_P;
    if (!std::isfinite(cfg->min_p) || !(0.0f <= cfg->min_p && cfg->min_p <= 1.0f)) return DFLASH_ERR_INVALID_MIN_P;
    s->cfg = *cfg;
    s->draws = 0;
    if (cfg->rng_kind == 1) {
        s->s[0] = s->s[1] = s->s[2] = s->s[3] = 0;
    } else {
        uint64_t sm = cfg->seed;
        for (int i = 0; i < 4; i++) s->s[i] = splitmix_next(sm);
    }
    return DFLASH_OK;
}

int32_t dflash_sampler_at_draw(dflash_sampler *s, const dflash_sampling_config *cfg, uint64_t draws) {
    int32_t rc = dflash_sampler_init(s, cfg);
    if (rc) return rc;
    dflash_sampler_advance(s, draws);
    return DFLASH_OK;
}

void dflash_sampler_peek(const dflash_sampler *s, int32_t n, double *out_host) {
    dflash_sampler copy = *s;
    for (int32_t i = 0; i < n; i++)
        out_host[i] = static_cast<double>(sampler_raw_next(&copy) >> 11) / 9007199254740992.0;
}

void dflash_sampler_advance(dflash_sampler *s, uint64_t draws) {
    for (uint64_t i = 0; i < draws; i++) sampler_raw_next(s);
    s->draws += draws;
}

int32_t dflash_accept_prefix(dflash_ctx *ctx, const int32_t *verified, int32_t n_tokens, const float *target_logits,
                             int64_t vocab, int32_t mode, int32_t n_proposals, const int32_t *prop_tokens,
                             const int32_t *prop_counts, const dflash_weighted_candidate *prop_cands,
                             const float *draft_logits, float draft_temperature, dflash_sampler *sampler,
                             int64_t budget, const int32_t *stop_ids, int32_t n_stop, dflash_accept_decision *out,
                             dflash_stream_t stream) {
    if (!ctx) return DFLASH_ERR_INVALID_INPUT;
    if (!out || !sampler) return dfl_fail(ctx, DFLASH_ERR_INVALID_INPUT, "accept_prefix: null sampler / output");
    memset(out, 0, sizeof(*out));
    out->err_row = -1;
    out->err_index = -1;
    // ---- whole-block validation before anything is drawn (accept.rs:85-130)
    if (n_tokens < 1 || !verified) return dfl_fail(ctx, DFLASH_ERR_INVALID_INPUT, "missing carry token");
    if (vocab <= 0 || vocab > 0x7fffffffll) return dfl_fail(ctx, DFLASH_ERR_INVALID_INPUT, "invalid vocabulary size");
    if (n_tokens > kMaxRows)
        return dfl_fail(ctx, DFLASH_ERR_BAD_SHAPE, "accept_prefix: %d verified tokens (at most %d)", n_tokens, kMaxRows);
    if (!target_logits) return dfl_fail(ctx, DFLASH_ERR_INVALID_INPUT, "target logits extent mismatch");
    if (mode < 0 || mode > 2) return dfl_fail(ctx, DFLASH_ERR_INVALID_INPUT, "accept_prefix: proposal mode %d", mode);
    if (n_stop < 0 || (n_stop > 0 && !stop_ids)) return dfl_fail(ctx, DFLASH_ERR_INVALID_INPUT, "accept_prefix: stop ids");
    for (int i = 0; i < n_tokens; i++) {
        if (verified[i] < 0 || verified[i] >= vocab) {
            out->err_row = i;
            out->err_index = verified[i];
            return dfl_fail(ctx, DFLASH_ERR_INVALID_TOKEN, "verified input token %d at index %d is outside vocabulary %lld",
                            verified[i], i, static_cast<long long>(vocab));
        }
    }
    const int n_drafts = n_tokens - 1;
    int prop_offsets[kMaxRows] = {0};
    int n_cands = 0;
    if (mode == 1) {
        if (n_proposals != n_drafts || (n_drafts > 0 && (!prop_tokens || !prop_counts)))
            return dfl_fail(ctx, DFLASH_ERR_INVALID_INPUT, "proposal row count mismatch");
        for (int r = 0; r < n_drafts; r++) {
            if (prop_tokens[r] != verified[r + 1]) {
                out->err_row = r;
                out->err_index = prop_tokens[r];
                return dfl_fail(ctx, DFLASH_ERR_PROPOSAL_MISMATCH, "proposal row %d sampled token %d, but verified draft is %d",
                                r, prop_tokens[r], verified[r + 1]);
            }
            if (prop_counts[r] < 0 || (prop_counts[r] > 0 && !prop_cands))
                return dfl_fail(ctx, DFLASH_ERR_INVALID_INPUT, "accept_prefix: proposal candidates");
            prop_offsets[r] = n_cands;
            for (int j = 0; j < prop_counts[r]; j++) {
                int32_t t = prop_cands[n_cands + j].token;
                if (t < 0 || t >= vocab) {
                    out->err_row = r;
                    out->err_code = DFLASH_ERR_PROPOSAL_TOKEN_OUT_OF_RANGE;
                    out->err_index = t;
                    return dfl_fail(ctx, DFLASH_ERR_PROPOSAL_TOKEN_OUT_OF_RANGE, "proposal token %d is outside the target vocabulary", t);
                }
            }
            n_cands += prop_counts[r];
        }
    }
    if (mode == 2) {
        if (!draft_logits) return dfl_fail(ctx, DFLASH_ERR_INVALID_INPUT, "accept_prefix: draft logits");
        if (!(std::isfinite(draft_temperature) && draft_temperature > 0.0f))
            return dfl_fail(ctx, DFLASH_ERR_INVALID_TEMPERATURE, "accept_prefix: draft temperature %f", draft_temperature);
    }
    // ---- terminal anchor / exhausted budget: no draw, nothing retained (accept.rs:131-145)
    bool anchor_eos = false;
    for (int i = 0; i < n_stop; i++) anchor_eos = anchor_eos || stop_ids[i] == verified[0];
    if (anchor_eos || budget == 0) {
        out->stop_reason = anchor_eos ? DFLASH_STOP_EOS : DFLASH_STOP_TOKEN_LIMIT;
        return DFLASH_OK;
    }
    const dflash_sampling_config &sc = sampler->cfg;
    int64_t k_eff = (sc.temperature == 0.0f) ? 1 : ((sc.top_k == 0 || static_cast<int64_t>(sc.top_k) >= vocab) ? vocab : static_cast<int64_t>(sc.top_k));
    const bool wide = k_eff > kMaxK;  // top_k = 0 or a large top_k: accept_wide.hip
    const int n_chunks = static_cast<int>((vocab + kSelChunk - 1) / kSelChunk);
    if (!wide && n_chunks * k_eff > 2 * kSelThreads)
        return dfl_fail(ctx, DFLASH_ERR_UNSUPPORTED, "accept_prefix: vocabulary %lld x top_k %lld too large", static_cast<long long>(vocab), static_cast<long long>(k_eff));

    hipStream_t st = static_cast<hipStream_t>(stream);
    const int n_tiles = static_cast<int>((vocab + 1023) / 1024);
    size_t off = 0;
    // (wide sets order their candidates elsewhere: no lists of the target's chunks)
    uint64_t *chunks = dfl_ws_take<uint64_t>(ctx, &off, sizeof(uint64_t) * (wide ? 0 : k_eff) * n_tokens * n_chunks);
    uint64_t *draft_best = dfl_ws_take<uint64_t>(ctx, &off, sizeof(uint64_t) * n_tokens * n_chunks);
    RowDist *rows = dfl_ws_take<RowDist>(ctx, &off, sizeof(RowDist) * n_tokens);
    double *tile_sums = dfl_ws_take<double>(ctx, &off, sizeof(double) * n_tokens * n_tiles);
    int32_t *d_stop = dfl_ws_take<int32_t>(ctx, &off, sizeof(int32_t) * (n_stop + 8));
    dflash_weighted_candidate *d_cands =
        dfl_ws_take<dflash_weighted_candidate>(ctx, &off, sizeof(dflash_weighted_candidate) * (n_cands + 1));
    dflash_accept_decision *d_out = dfl_ws_take<dflash_accept_decision>(ctx, &off, sizeof(dflash_accept_decision));
    if (!chunks || !draft_best || !rows || !tile_sums || !d_stop || !d_cands || !d_out)
        return dfl_fail(ctx, DFLASH_ERR_WORKSPACE, "accept_prefix: workspace too small");

    // small host inputs: by value in the decision kernel's arguments; only the variable-length lists are copied
    DecideArgs a;
    memset(&a, 0, sizeof(a));
    dflash_sampler_peek(sampler, n_tokens + 1, a.walk.uniforms);
    a.walk.n_tokens = n_tokens;
    for (int i = 0; i < n_tokens; i++) a.walk.verified[i] = verified[i];
    for (int r = 0; r < n_drafts && mode == 1; r++) {
        a.prop_offsets[r] = prop_offsets[r];
        a.prop_counts[r] = prop_counts[r];
    }
    if (n_stop > 0)
        DFL_HIP_CHECK(ctx, hipMemcpyAsync(d_stop, stop_ids, sizeof(int32_t) * n_stop, hipMemcpyHostToDevice, st));
    if (n_cands > 0)
        DFL_HIP_CHECK(ctx, hipMemcpyAsync(d_cands, prop_cands, sizeof(dflash_weighted_candidate) * n_cands,
                                          hipMemcpyHostToDevice, st));

    ChainCfg cfg;
    cfg.temperature = sc.temperature;
    cfg.top_p = sc.top_p;
    cfg.min_p = sc.min_p;
    cfg.k = static_cast<int32_t>(k_eff);
    cfg.ln_min_p = sc.min_p > 0.0f ? std::log(static_cast<double>(sc.min_p)) : 0.0;
    cfg.draft_temperature = draft_temperature;
    cfg.mode = mode;
    {
        dfl_timed timer(ctx, st, DFL_T_ACCEPT);
        const bool dense = mode == 2 && n_drafts > 0;
        const uint64_t *wide_keys = nullptr;
        const double *wide_w = nullptr;
        if (wide) {
            if (const int32_t rc_ = dfl_accept_wide_rows(ctx, target_logits, n_tokens, vocab, vocab, cfg, a.walk, rows, &off, &wide_keys, &wide_w,
                                                         &a.wide_stride, st))
                return rc_;
            if (dense) select_chunk_kernel<<<dim3(n_chunks, n_drafts), kSelThreads, 0, st>>>(draft_logits, vocab, draft_best, static_cast<int>(vocab), 1, false);
        } else if (dense) {
            select_pair_kernel<<<dim3(n_chunks, n_tokens + n_drafts), kSelThreads, 0, st>>>(target_logits, draft_logits, vocab, chunks, draft_best,
                                                                                         static_cast<int>(vocab), n_tokens, cfg.k);
        } else {
            select_chunk_kernel<<<dim3(n_chunks, n_tokens), kSelThreads, 0, st>>>(target_logits, vocab, chunks, static_cast<int>(vocab), cfg.k, false);
        }
        // the rows' chains and, for dense proposals, the tile sums of the draft rows: one launch (wide: the chain has run; only the
        // draft side is merged)
        if (dense) {
            rows_and_tiles_kernel<<<dim3(n_tokens, 1 + (n_tiles + 3) / 4), kSelThreads, 0, st>>>(
                chunks, draft_logits, draft_best, tile_sums, static_cast<int>(vocab), n_chunks, cfg.k, n_tokens, draft_temperature, n_tiles, rows, wide,
                cfg, a.walk);
        } else if (!wide) {
            row_merge_kernel<<<n_tokens, kSelThreads, 0, st>>>(chunks, rows, nullptr, n_chunks, cfg.k, cfg, a.walk);
        }
        a.wide_keys = wide_keys;
        a.wide_w = wide_w;
        a.n_stop = n_stop;
        a.budget = budget;
        a.stop_ids = d_stop;
        a.prop_cands = d_cands;
        a.draft = draft_logits;
        a.draft_stride = vocab;
        a.temperature = sc.temperature;
        a.draft_temperature = draft_temperature;
        // the decision goes straight to the context's pinned page when the device can address it (one copy less
        // between the last kernel and the host)
        static_assert(sizeof(dflash_accept_decision) <= DFL_PINNED_BYTES, "the decision is read back through the pinned page");
        void *const pinned_dev = ctx->pinned_dev;
        const bool direct = pinned_dev != nullptr;
        decide_kernel<<<1, kDecThreads, 0, st>>>(rows, tile_sums, direct ? static_cast<dflash_accept_decision *>(pinned_dev) : d_out, mode, n_tiles,
                                                 n_tokens, a);
        DFL_HIP_CHECK(ctx, hipGetLastError());
        if (!direct) DFL_HIP_CHECK(ctx, hipMemcpyAsync(ctx->pinned, d_out, sizeof(*out), hipMemcpyDeviceToHost, st));
    }
    DFL_HIP_CHECK(ctx, hipStreamSynchronize(st));
    memcpy(out, ctx->pinned, sizeof(*out));
    if (out->err_code) {
        int32_t code = out->err_code;
        return dfl_fail(ctx, code, "DFlash target row %d: %s (index %lld)", out->err_row, dflash_status_name(code),
                        static_cast<long long>(out->err_index));
    }
    dflash_sampler_advance(sampler, static_cast<uint64_t>(out->draws_used));  // committed only on success
    return DFLASH_OK;
}

}  // extern "C"
