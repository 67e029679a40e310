// Norm and rotation of one head by one wave (kernel_qk_rms_norm_rope_f32_packed_consecutive, attn.metal:137-196): RMSNorm over the
// head (weight may be null), NeoX RoPE over all of it (pairs (i, i + hd/2), angle = pos / theta^(2i/hd)).
#pragma once
#include "common.h"

// A pair's sine and cosine.
__device__ __forceinline__ void dfl_rope_angle(int i, int hd, float theta, float pos, float *sn, float *cs) {
    const float freq = pos / powf(theta, static_cast<float>(2 * i) / static_cast<float>(hd));
    sincosf(freq, sn, cs);
}
// What a norm multiplies a head's values by.
template <int HD>
__device__ __forceinline__ float dfl_head_scale(float sum_of_squares, float eps) {
    return 1.0f / sqrtf(sum_of_squares / static_cast<float>(HD) + eps);
}
// One pair's rotation; each result is rounded to f32 before whatever comes next.
// (spelled out, so that all kernels that rotate round alike)
__device__ __forceinline__ void dfl_rope_pair(float a, float b, float sn, float cs, float &ra, float &rb) {
    ra = __builtin_fmaf(a, cs, -(b * sn));
    rb = __builtin_fmaf(b, cs, a * sn);
    asm volatile("" : "+v"(ra), "+v"(rb));
}

// A lane's rotation pairs of one head: pair k is elements (i, i + HD/2), i = lane + 64 k (heads of 64: lanes 0..31).
template <int HD>
struct RopePairs {
    static constexpr int N = HD <= 128 ? 1 : 2, kEl = HD / 64;  // pairs, elements per lane
    float sn[N], cs[N];
    __device__ __forceinline__ void angles(int lane, float theta, float pos) {
#pragma unroll
        for (int k = 0; k < N; k++) {
            const int i = HD == 64 ? (lane & 31) : lane + 64 * k;
            dfl_rope_angle(i, HD, theta, pos, &sn[k], &cs[k]);
        }
    }
};
// ... and the head's values: element lane + 64 k in r[k], its norm weight in wr[k] (heads of 64: a lane also holds the
// other element of its pair)
template <int HD>
struct RopeHead {
    static constexpr int kEl = HD / 64;
    float r[kEl], wr[kEl], r_far = 0.0f, w_far = 1.0f;
    __device__ __forceinline__ void load(const float *v, const float *w, int lane) {
#pragma unroll
        for (int k = 0; k < kEl; k++) r[k] = v[lane + 64 * k];
        if (HD == 64) r_far = v[lane ^ 32];
#pragma unroll
        for (int k = 0; k < kEl; k++) wr[k] = w ? w[lane + 64 * k] : 1.0f;
        if (HD == 64) w_far = w ? w[lane ^ 32] : 1.0f;
    }
    // norm, weight (where there is one), rotation; put(i, value) for elements i and i + HD / 2 of every pair
    template <typename Put>
    __device__ __forceinline__ void finish(const RopePairs<HD> &t, bool weighted, int lane, float eps, Put put) const {
        float s = r[0] * r[0];
#pragma unroll
        for (int k = 1; k < kEl; k++) s = __builtin_fmaf(r[k], r[k], s);
        s = dfl_wave_sum(s);
        const float scale = dfl_head_scale<HD>(s, eps);
#pragma unroll
        for (int k = 0; k < RopePairs<HD>::N; k++) {
            constexpr int kFar = HD / 128;  // the partner's register, from k on
            float a = r[k] * scale, b = (HD == 64 ? r_far : r[k + (HD == 64 ? 0 : kFar)]) * scale;
            if (weighted) {
                a *= wr[k];
                b *= HD == 64 ? w_far : wr[k + (HD == 64 ? 0 : kFar)];
            }
            float ra, rb;
            dfl_rope_pair(a, b, t.sn[k], t.cs[k], ra, rb);
            if (HD > 64 || lane < 32) put(lane + 64 * k, ra, rb);
        }
    }
};
