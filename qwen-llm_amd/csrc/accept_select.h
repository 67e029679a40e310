// Selection of the k best of a workgroup's ordering keys without sorting them: shared by the chunk selections of
// accept.hip (k <= 64) and accept_wide.hip (k <= 1024).
#pragma once

#include "sampler_chain.h"

namespace {

constexpr uint64_t kNoKey = ~0ull;  // no key: a NaN's logit bits above the largest token

template <int THREADS>
struct KthShared {
    int hist[3][256];
    uint64_t lo[THREADS / 64], hi[THREADS / 64];
    int n[THREADS / 64];
};

// A bound B <= limit such that at least k and at most `most` >= k of the workgroup's keys are <= B; limit if no more than `most` are <= limit
// (which a bin's end that ends the search early could be above of).
// Digit by digit from the first bit in which the keys differ (most share sign and most of the exponent: a digit
// above it would put every key on one counter), and no further than until a digit's counts end there.  Keys are
// distinct, so the last digit ends at k at the latest.  One barrier per digit: every wave adds up the counters by
// itself, and of three sets of counters one is counted in, one may still be read, one is cleared for the next digit.
template <int PER, int THREADS>
__device__ uint64_t block_kth(const uint64_t (&key)[PER], uint64_t limit, int k, int most, KthShared<THREADS> &sh) {
    constexpr int kWaves = THREADS / 64;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    uint64_t lo = kNoKey, hi = 0;
    int n = 0;
#pragma unroll
    for (int j = 0; j < PER; j++) {
        const bool in = key[j] <= limit;
        lo = in && key[j] < lo ? key[j] : lo;
        hi = in && key[j] > hi ? key[j] : hi;
        n += __popcll(__builtin_amdgcn_ballot_w64(in));
    }
    lo = wave_min_u64(lo);
    hi = ~wave_min_u64(~hi);
    if (lane == 0) {
        sh.lo[wave] = lo;
        sh.hi[wave] = hi;
        sh.n[wave] = n;
    }
    if (tid < 256) sh.hist[0][tid] = 0;
    __syncthreads();
    lo = wave_min_u64(lane < kWaves ? sh.lo[lane] : kNoKey);
    hi = ~wave_min_u64(lane < kWaves ? ~sh.hi[lane] : kNoKey);
    n = __builtin_amdgcn_readlane(wave_scan_i32(lane < kWaves ? sh.n[lane] : 0), 63);
    if (n <= most) return limit;
    const int slack = most - k;
    int shift = 64 - __clzll(static_cast<long long>(lo ^ hi));  // 1 .. 64: n > k >= 1 distinct keys
    uint64_t prefix = (lo >> 1) >> (shift - 1);
    for (int set = 0;; set = set == 2 ? 0 : set + 1) {
        const int digit = shift > 8 ? shift - 8 : 0, mask = (1 << (shift - digit)) - 1;
#pragma unroll
        for (int j = 0; j < PER; j++)
            if (key[j] <= limit && ((key[j] >> 1) >> (shift - 1)) == prefix) atomicAdd(&sh.hist[set][static_cast<int>(key[j] >> digit) & mask], 1);
        if (tid < 256) sh.hist[set == 2 ? 0 : set + 1][tid] = 0;
        __syncthreads();
        const int4 c = *reinterpret_cast<const int4 *>(&sh.hist[set][4 * lane]);
        const int upto = wave_scan_i32(c.x + c.y + c.z + c.w);
        int below = upto - (c.x + c.y + c.z + c.w), bin = 4 * lane, count = c.x;
        const bool here = below < k && k <= upto;  // in one lane
        if (below + count < k) below += count, bin++, count = c.y;
        if (bin == 4 * lane + 1 && below + count < k) below += count, bin++, count = c.z;
        if (bin == 4 * lane + 2 && below + count < k) below += count, bin++, count = c.w;
        const int from = __builtin_ctzll(__builtin_amdgcn_ballot_w64(here));
        k -= __builtin_amdgcn_readlane(below, from);
        prefix = (prefix << (shift - digit)) | static_cast<uint64_t>(__builtin_amdgcn_readlane(bin, from));
        shift = digit;
        if (__builtin_amdgcn_readlane(count, from) - k <= slack) return (prefix << shift) | ((uint64_t(1) << shift) - 1);
    }
}

// The same over ordering words, one a thread, which may be alike: a bound that at least k of them are at or below (the largest word
// if there are no k) and, as far as the words differ, at most `most`.  Bins of the words' own range, 128 to 256 of them, so that
// one round is nearly always the last; a word is one instruction a step where a key is five (2.2 -> 1.1 us of a workgroup of 512).
// The largest word is not counted: of a vocabulary that a mask has left little of, it is nearly all words, on one counter in every round.
template <int THREADS>
__device__ __forceinline__ uint32_t block_kth_word(uint32_t word, int k, int most, KthShared<THREADS> &sh) {
    constexpr int kWaves = THREADS / 64;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, slack = most - k;
    {
        const uint32_t lo = wave_min_u32(word), hi = wave_max_u32(word);
        if (lane == 0) sh.lo[wave] = (static_cast<uint64_t>(hi) << 32) | lo;
    }
    if (tid < 256) sh.hist[0][tid] = 0;
    __syncthreads();
    const uint64_t ends = sh.lo[lane < kWaves ? lane : 0];
    uint32_t lo = wave_min_u32(static_cast<uint32_t>(ends));
    const uint32_t hi = wave_max_u32(static_cast<uint32_t>(ends >> 32));
    if (k >= THREADS || lo == hi) return hi;
    int shift = max(0, 24 - __clz(hi - lo));  // ((hi - lo) >> shift < 256)
    for (int set = 0;; set = set == 2 ? 0 : set + 1) {
        const uint32_t bin_of = (word - lo) >> shift;
        if (word >= lo && bin_of < 256 && word != hi) atomicAdd(&sh.hist[set][bin_of], 1);
        if (tid < 256) sh.hist[set == 2 ? 0 : set + 1][tid] = 0;
        __syncthreads();
        const int4 c = *reinterpret_cast<const int4 *>(&sh.hist[set][4 * lane]);
        const int upto = wave_scan_i32(c.x + c.y + c.z + c.w);
        int below = upto - (c.x + c.y + c.z + c.w), bin = 4 * lane, count = c.x;
        if (__builtin_amdgcn_readlane(upto, 63) < k) return hi;  // (in the first round if at all)
        const bool here = below < k && k <= upto;  // in one lane
        if (below + count < k) below += count, bin++, count = c.y;
        if (bin == 4 * lane + 1 && below + count < k) below += count, bin++, count = c.z;
        if (bin == 4 * lane + 2 && below + count < k) below += count, bin++, count = c.w;
        const int from = __builtin_ctzll(__builtin_amdgcn_ballot_w64(here));
        k -= __builtin_amdgcn_readlane(below, from);
        lo += static_cast<uint32_t>(__builtin_amdgcn_readlane(bin, from)) << shift;
        if (shift == 0 || __builtin_amdgcn_readlane(count, from) - k <= slack) return lo + min((uint32_t(1) << shift) - 1, hi - lo);  // (the last bin may end above every word)
        shift = max(0, shift - 8);
    }
}

// A bound <= limit on the k best keys, out of the threads' best ones (first, with the word best; `word` is what at least k of the threads' best
// words are at or below, or the largest there is): at most the keys of k threads are at or below it.  Where many words are alike (a
// vocabulary of which a mask has left a few) the k-th is one of those: it is looked for among the threads that have that word, whose
// keys differ in their tokens only, two or three digits; all keys together would be counted on one counter, digit after digit.
template <int THREADS>
__device__ __forceinline__ uint64_t block_kth_first(uint64_t first, uint32_t best, uint32_t word, uint64_t limit, int k, KthShared<THREADS> &sh) {
    const int below = __syncthreads_count(best < word);
    const bool alike = below < k;
    const uint64_t mine[1] = {!alike || best == word ? first : kNoKey};
    k -= alike ? below : 0;
    return block_kth<1>(mine, limit, k, k, sh);
}

// The workgroup's keys <= bound to the slots [0, cap) of out, in no order, as far as they fit; *cnt (0 before) becomes
// their number.  A wave asks for its slots with one addition, and a thread's are next to each other.
template <int PER>
__device__ __forceinline__ void compact_keys(const uint64_t (&key)[PER], uint64_t bound, uint64_t *out, int cap, int *cnt) {
    const int lane = threadIdx.x & 63;
    int n = 0;
#pragma unroll
    for (int j = 0; j < PER; j++) n += key[j] <= bound;
    const int upto = wave_scan_i32(n), all = __builtin_amdgcn_readlane(upto, 63);
    if (all == 0) return;
    int at = 0;
    if (lane == 0) at = atomicAdd(cnt, all);
    at = __builtin_amdgcn_readfirstlane(at) + upto - n;
#pragma unroll
    for (int j = 0; j < PER; j++) {
        if (key[j] <= bound) {
            if (at < cap) out[at] = key[j];
            at++;
        }
    }
}

}  // namespace
