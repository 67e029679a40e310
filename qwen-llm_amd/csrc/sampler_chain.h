// The sampler-v1 filter chain on the device (sampling.rs:1541-1615), its ordering keys
// (sampling.rs:1206-1235) and the categorical pick (sampling.rs:1587-1596): shared by the
// accept-prefix kernels and the sampled DFlash-2 selector walk.  Everything that feeds a
// comparison with a uniform draw is f64 and sequential, in the order of the reference's loops.
#pragma once

#include "common.h"

#include <cmath>

// f64 arithmetic that is compared with uniform draws keeps the reference's separately rounded
// operations: no fused multiply-adds from here on in the including file.
#pragma clang fp contract(off)

constexpr int kMaxK = 64;  // most candidates a row keeps inline (wider sets live in device arrays, accept_wide.hip)

// ------------------------------------------------------------------------------------------
// per-row results
// ------------------------------------------------------------------------------------------
struct RowDist {
    int32_t n_keep;     // candidates after every filter (above kMaxK: tokens / weights are in the wide arrays instead)
    int32_t err;        // DFLASH_ERR_* or 0
    int64_t err_index;  // NaN index etc.
    double total;       // sum of the kept weights (sequential)
    int32_t tokens[kMaxK];
    double weights[kMaxK];
    // dense proposal side
    int32_t d_err;
    int32_t pick;  // the token the row's draw falls on
    int64_t d_err_index;
    double d_max_scaled;  // f64(max draft logit) / T
    double draft_weight;  // weight of the row's draft among the kept candidates, -0 if it is not one
    double q_draft;       // exp(draft's draft logit / T - d_max_scaled)
    double q[kMaxK];      // the same of the kept candidates (inline sets)
};

// What the block's decision asks of a row's candidates: row r's draw is uniforms[r] (every row before it accepted,
// each with one draw) and its draft verified[r + 1].
struct BlockWalk {
    int32_t n_tokens;
    int32_t verified[16];
    double uniforms[17];
};

struct ChainCfg {
    float temperature, top_p, min_p;
    int32_t k;          // effective top-k
    double ln_min_p;    // ln(f64(min_p)), computed on the host
    float draft_temperature;
    int32_t mode;       // proposal mode
};

namespace {

// sampling.rs:1206-1220: a u32 whose ascending order is descending f32 total order
__device__ __host__ __forceinline__ uint32_t desc_bits(uint32_t bits) {
    uint32_t asc = (bits & 0x80000000u) ? ~bits : (bits | 0x80000000u);
    return ~asc;
}
__device__ __forceinline__ uint64_t cand_key(uint32_t token, float logit) {
    return (static_cast<uint64_t>(desc_bits(__float_as_uint(logit))) << 32) | token;
}
// sampling.rs:1223-1231
__device__ __forceinline__ float key_logit(uint64_t key) {
    uint32_t asc = ~static_cast<uint32_t>(key >> 32);
    uint32_t bits = (asc & 0x80000000u) ? (asc & 0x7fffffffu) : ~asc;
    return __uint_as_float(bits);
}
__device__ __forceinline__ int32_t key_token(uint64_t key) { return static_cast<int32_t>(static_cast<uint32_t>(key)); }

// Minimum of a key over the wave, in every lane: data-parallel-primitive moves within rows of 16 lanes (shift right
// by 1, 2, 4, 8: lane 15 of a row then holds the row's minimum), then lane 15 of rows 0 and 2 into rows 1 and 3, then
// lane 31 into rows 2 and 3; lane 63 has the result.  Lanes without a source read the identity.  No LDS round trips.
__device__ __forceinline__ uint64_t wave_min_u64(uint64_t v) {
#define DFL_MIN_STEP(ctrl, row_mask)                                                                                     \
    do {                                                                                                                 \
        const unsigned lo = __builtin_amdgcn_update_dpp(0xffffffffu, static_cast<unsigned>(v), ctrl, row_mask, 0xf, false);       \
        const unsigned hi = __builtin_amdgcn_update_dpp(0xffffffffu, static_cast<unsigned>(v >> 32), ctrl, row_mask, 0xf, false); \
        const uint64_t o = (static_cast<uint64_t>(hi) << 32) | lo;                                                       \
        v = o < v ? o : v;                                                                                               \
    } while (0)
    DFL_MIN_STEP(0x111, 0xf);  // row_shr:1
    DFL_MIN_STEP(0x112, 0xf);  // row_shr:2
    DFL_MIN_STEP(0x114, 0xf);  // row_shr:4
    DFL_MIN_STEP(0x118, 0xf);  // row_shr:8
    DFL_MIN_STEP(0x142, 0xa);  // row_bcast:15 into rows 1 and 3
    DFL_MIN_STEP(0x143, 0xc);  // row_bcast:31 into rows 2 and 3
#undef DFL_MIN_STEP
    const unsigned lo = __builtin_amdgcn_readlane(static_cast<unsigned>(v), 63);
    const unsigned hi = __builtin_amdgcn_readlane(static_cast<unsigned>(v >> 32), 63);
    return (static_cast<uint64_t>(hi) << 32) | lo;
}

// Inclusive sum over the wave's lanes, by the same moves.
__device__ __forceinline__ int wave_scan_i32(int v) {
#define DFL_SUM_STEP(ctrl, row_mask) v += __builtin_amdgcn_update_dpp(0, v, ctrl, row_mask, 0xf, false)
    DFL_SUM_STEP(0x111, 0xf);
    DFL_SUM_STEP(0x112, 0xf);
    DFL_SUM_STEP(0x114, 0xf);
    DFL_SUM_STEP(0x118, 0xf);
    DFL_SUM_STEP(0x142, 0xa);
    DFL_SUM_STEP(0x143, 0xc);
#undef DFL_SUM_STEP
    return v;
}

// Minimum / maximum of a word over the wave, in every lane: the same moves, one instruction each.
__device__ __forceinline__ uint32_t wave_min_u32(uint32_t v) {
#define DFL_MIN_STEP(ctrl, row_mask)                                                                                            \
    do {                                                                                                                        \
        const uint32_t o = __builtin_amdgcn_update_dpp(0xffffffffu, v, ctrl, row_mask, 0xf, false);                             \
        v = o < v ? o : v;                                                                                                      \
    } while (0)
    DFL_MIN_STEP(0x111, 0xf);
    DFL_MIN_STEP(0x112, 0xf);
    DFL_MIN_STEP(0x114, 0xf);
    DFL_MIN_STEP(0x118, 0xf);
    DFL_MIN_STEP(0x142, 0xa);
    DFL_MIN_STEP(0x143, 0xc);
#undef DFL_MIN_STEP
    return __builtin_amdgcn_readlane(v, 63);
}
__device__ __forceinline__ uint32_t wave_max_u32(uint32_t v) { return ~wave_min_u32(~v); }

// sampling.rs:1541-1615 on the ordered candidates of one row (keys ascending = best first)
// Work arrays of the chain (kMaxK entries each): a caller that runs the chain on one thread of a workgroup
// keeps them in LDS; private arrays of this size live in scratch memory, where every access is a trip to memory.
struct ChainScratch {
    double *l, *w;
    int *tok;
};

__device__ void run_chain(const uint64_t *keys, int len, const ChainCfg &c, RowDist *d, const ChainScratch &scratch) {
    double *l = scratch.l;
    int *tok = scratch.tok;
    for (int i = 0; i < len; i++) {
        l[i] = static_cast<double>(key_logit(keys[i]));
        tok[i] = key_token(keys[i]);
    }
    if (c.min_p > 0.0f) {
        double max_logit = l[0];
        if (isfinite(max_logit)) {
            double threshold = max_logit + c.ln_min_p;
            int keep = 0;
            for (int i = 0; i < len; i++)
                if (l[i] >= threshold) {
                    l[keep] = l[i];
                    tok[keep] = tok[i];
                    keep++;
                }
            len = keep;
        }
    }
    if (len == 0) {
        d->err = DFLASH_ERR_NO_CANDIDATES;
        return;
    }
    if (l[0] == INFINITY) {
        int keep = 0;
        for (int i = 0; i < len; i++)
            if (l[i] == INFINITY) {
                l[keep] = l[i];
                tok[keep] = tok[i];
                keep++;
            }
        len = keep;
    }
    const double temperature = static_cast<double>(c.temperature);
    for (int i = 0; i < len; i++) l[i] /= temperature;
    double *w = scratch.w;
    int n_inf = 0;
    for (int i = 0; i < len; i++) n_inf += (l[i] == INFINITY);
    if (n_inf > 0) {
        for (int i = 0; i < len; i++) w[i] = (l[i] == INFINITY) ? 1.0 : 0.0;
    } else {
        double max_logit = l[0];
        if (max_logit == -INFINITY) {
            d->err = DFLASH_ERR_NO_CANDIDATES;
            return;
        }
        bool finite = true;
        for (int i = 0; i < len; i++) {
            w[i] = exp(l[i] - max_logit);
            finite = finite && isfinite(w[i]);
        }
        if (!finite) {
            d->err = DFLASH_ERR_NO_CANDIDATES;
            return;
        }
    }
    if (c.top_p < 1.0f) {
        double total = -0.0;
        for (int i = 0; i < len; i++) total += w[i];
        double target = total * static_cast<double>(c.top_p);
        double cumulative = 0.0;
        int keep = 0;
        for (int i = 0; i < len; i++) {
            cumulative += w[i];
            keep++;
            if (cumulative >= target) break;
        }
        len = keep < 1 ? 1 : keep;
    }
    double total_weight = -0.0;
    for (int i = 0; i < len; i++) total_weight += w[i];
    if (!(isfinite(total_weight) && total_weight > 0.0)) {
        d->err = DFLASH_ERR_NO_CANDIDATES;
        return;
    }
    d->n_keep = len;
    d->total = total_weight;
    for (int i = 0; i < len; i++) {
        d->tokens[i] = tok[i];
        d->weights[i] = w[i];
    }
}

// A lane's double in every lane (src uniform).
__device__ __forceinline__ double chain_bcast(double v, int src) {
    const unsigned long long b = static_cast<unsigned long long>(__double_as_longlong(v));
    const unsigned lo = __builtin_amdgcn_readlane(static_cast<unsigned>(b), src);
    const unsigned hi = __builtin_amdgcn_readlane(static_cast<unsigned>(b >> 32), src);
    return __longlong_as_double(static_cast<long long>((static_cast<unsigned long long>(hi) << 32) | lo));
}

// Lane i: start + w[0] + .. + w[i], added in that order, one after the other; w of the lanes from len on is +0 (len <= 64,
// uniform).  The lanes' values are read at constant positions, sixteen a round, and move down by sixteen for the next: a
// read at a position that is itself in a register, with its loop, is 70 cycles an addition, this is 30.
__device__ __forceinline__ double wave_running_sum(double start, double w, int len) {
    const int lane = threadIdx.x & 63;
    double acc = start, mine = start;
#pragma unroll 1
    for (int base = 0; base < len; base += 16) {
#pragma unroll
        for (int j = 0; j < 16; j++) {
            acc += chain_bcast(w, j);
            mine = lane - base >= j ? acc : mine;
        }
        w = __shfl(w, lane + 16, 64);
    }
    return mine;
}
// The first lane of [0, len) for which `reached` holds, or len - 1.
__device__ __forceinline__ int wave_first(bool reached, int len) {
    const uint64_t m = __builtin_amdgcn_ballot_w64(static_cast<int>(threadIdx.x & 63) < len && reached);
    return m ? static_cast<int>(__builtin_ctzll(m)) : len - 1;
}

// run_chain by one whole wave (len <= 64): lane i holds candidate i.  What the reference does element by element
// without carrying anything from one element to the next (the conversions, the division by the temperature, the
// exponentials, the filters' comparisons) is done by all lanes at once; every sum that is compared with something is
// still added in candidate order, one addition after the other: each is one of the running sums of the weights (from
// +0 or -0 is the same, no weight is below +0), so they are added up once.  The candidates are in descending logit
// order, so what min-p and the +inf rule keep is a prefix: its length is a population count.
struct WaveChain {
    int len;          // candidates kept, 0 = none (uniform)
    double w, upto;   // lane i: its weight, the running sum up to it
    double total;     // of the kept ones (uniform)
};
__device__ __forceinline__ WaveChain run_chain_wave(float logit, int len, const ChainCfg &c) {
    const int lane = threadIdx.x & 63;
    WaveChain r = {0, 0.0, 0.0, 0.0};
    double l = lane < len ? static_cast<double>(logit) : 0.0;
    const double l0 = chain_bcast(l, 0);
    if (c.min_p > 0.0f && len > 0 && isfinite(l0)) len = __popcll(__builtin_amdgcn_ballot_w64(lane < len && l >= l0 + c.ln_min_p));
    if (len == 0) return r;
    if (l0 == INFINITY) len = __popcll(__builtin_amdgcn_ballot_w64(lane < len && l == INFINITY));
    l = l / static_cast<double>(c.temperature);
    const double max_logit = chain_bcast(l, 0);
    if (max_logit == INFINITY) {
        r.w = lane < len && l == INFINITY ? 1.0 : 0.0;
    } else {
        if (max_logit == -INFINITY) return r;
        r.w = lane < len ? exp(l - max_logit) : 0.0;
        if (__builtin_amdgcn_ballot_w64(!isfinite(r.w)) != 0) return r;
    }
    r.upto = wave_running_sum(0.0, r.w, len);
    if (c.top_p < 1.0f) {
        const double target = chain_bcast(r.upto, len - 1) * static_cast<double>(c.top_p);
        len = wave_first(r.upto >= target, len) + 1;
    }
    r.total = chain_bcast(r.upto, len - 1);
    if (isfinite(r.total) && r.total > 0.0) r.len = len;
    return r;
}

// the same with private work arrays
__device__ void run_chain(const uint64_t *keys, int len, const ChainCfg &c, RowDist *d) {
    double l[kMaxK], w[kMaxK];
    int tok[kMaxK];
    run_chain(keys, len, c, d, ChainScratch{l, w, tok});
}

// first candidate whose running sum exceeds x, else the last (sampling.rs:1587-1596)
__device__ int pick_index(const double *w, int n, double x) {
    double cumulative = 0.0;
    for (int i = 0; i < n; i++) {
        cumulative += w[i];
        if (x < cumulative) return i;
    }
    return n - 1;
}

}  // namespace
