// Mixture-of-experts FFN of the packed verify: route on the device, then read every selected
// expert's weights ONCE for all block rows that picked it (the reference runs the experts per
// row after a packed route, metal_dflash.rs:10184-10403; CPU form ffn_moe, forward.rs:749-824).
//
//   probs   = softmax(router . x)                       over all experts
//   picks   = top-k by probability, ties to the lower expert id
//   weights = probs[pick] / max(sum(probs[picks]), 2^-14)
//   out     = sum_k weights[k] * down_e(silu(gate_e x) * up_e x)  +  sigmoid(x . w_shexp) * shared(x)
//
// Work items are "slots": slot = row * n_used + k.  The expert kernels run one workgroup column
// per expert; a workgroup first collects the slots that picked its expert and leaves at once
// if there are none, so HBM traffic is the distinct experts of the block, not rows x k.
#include "common.h"
#include "device_quant.h"
#include "mfma_unpack.h"
#include "moe_route.h"

#include <algorithm>
#include <cstdlib>

namespace {

constexpr int kMaxSlots = 16;  // a row picks an expert at most once, and a block has at most 16 rows

// Maximum of a 64-bit key over the wave, in every lane: data-parallel-primitive moves within rows of
// 16 lanes (shift right by 1, 2, 4, 8: lane 15 of a row then holds the row's maximum), then lane 15
// of rows 0 and 2 broadcast into rows 1 and 3, then lane 31 into rows 2 and 3; lane 63 has the
// result.  Lanes without a source read 0, the identity.  No LDS round trips, unlike a shuffle.
__device__ __forceinline__ unsigned long long wave_max_u64(unsigned long long v) {
#define DFL_MAX_STEP(ctrl, row_mask)                                                                            \
    do {                                                                                                        \
        const unsigned lo = __builtin_amdgcn_update_dpp(0u, static_cast<unsigned>(v), ctrl, row_mask, 0xf, false);      \
        const unsigned hi = __builtin_amdgcn_update_dpp(0u, static_cast<unsigned>(v >> 32), ctrl, row_mask, 0xf, false); \
        const unsigned long long o = (static_cast<unsigned long long>(hi) << 32) | lo;                          \
        v = o > v ? o : v;                                                                                      \
    } while (0)
    DFL_MAX_STEP(0x111, 0xf);  // row_shr:1
    DFL_MAX_STEP(0x112, 0xf);  // row_shr:2
    DFL_MAX_STEP(0x114, 0xf);  // row_shr:4
    DFL_MAX_STEP(0x118, 0xf);  // row_shr:8
    DFL_MAX_STEP(0x142, 0xa);  // row_bcast:15 into rows 1 and 3
    DFL_MAX_STEP(0x143, 0xc);  // row_bcast:31 into rows 2 and 3
#undef DFL_MAX_STEP
    const unsigned lo = __builtin_amdgcn_readlane(static_cast<unsigned>(v), 63);
    const unsigned hi = __builtin_amdgcn_readlane(static_cast<unsigned>(v >> 32), 63);
    return (static_cast<unsigned long long>(hi) << 32) | lo;
}

// Routing of a whole block in one workgroup of sixteen waves (n_expert <= 1024, at most 16 rows).
// Wave w serves block row w: softmax, top-k (higher probability first, equal probabilities to the
// lower id), the renormalised weights in pick order, and the
// shared-expert gate; a row's arithmetic does not depend on how many rows the block has.  Then the
// whole workgroup lists the block's distinct experts in ascending id order: ids[0 .. n), then one
// slot with id -1 (the shared expert, which every row uses) if with_shared; *n_slots = n (+ 1); for
// every (row, k) pick, slot_of = the index of its expert in that list.
__global__ void __launch_bounds__(1024)
    moe_route_kernel(const float *__restrict__ logits, const float *__restrict__ x, const float *__restrict__ shexp_gate,
                     int n_rows, int n_expert, int n_used, int hidden, int with_shared, int32_t *__restrict__ sel_e,
                     float *__restrict__ sel_w, float *__restrict__ sg, int32_t *__restrict__ ids,
                     int32_t *__restrict__ n_slots, int32_t *__restrict__ slot_of) {
    typedef float f4 __attribute__((ext_vector_type(4)));
    extern __shared__ __attribute__((aligned(16))) float probs[];  // [16][n_expert], then int32 rank[n_expert]
    __shared__ float pick_w[16][64];
    __shared__ int32_t pick_e[16][64];
    __shared__ int wave_count[16];
    int32_t *rank = reinterpret_cast<int32_t *>(probs + 16 * n_expert);
    const int tid = threadIdx.x, lane = tid & 63, row = tid >> 6;
    const bool live = row < n_rows;
    float *pr = probs + row * n_expert;
    if (live) {
        // Everything this row reads from memory is requested before anything waits for it: its first
        // 256 router logits and (2048 elements at a time) the operands of the shared-expert gate
        // sigmoid(x . w); one memory latency instead of one per phase.
        const float *lg = logits + static_cast<size_t>(row) * n_expert;
        float lgv[4];
#pragma unroll
        for (int j = 0; j < 4; j++) lgv[j] = lane + 64 * j < n_expert ? lg[lane + 64 * j] : -INFINITY;
        const float *xr = x + static_cast<size_t>(row) * hidden;
        float dot = 0.0f;
        if (!shexp_gate) {
            // the gate was computed by the kernel that wrote x
        } else if (hidden % 4 == 0) {
            for (int base = 0; base < hidden; base += 2048) {
                f4 xa[8], gb[8];
#pragma unroll
                for (int j = 0; j < 8; j++) {
                    const int i = base + 4 * lane + 256 * j;
                    xa[j] = gb[j] = f4{0, 0, 0, 0};
                    if (i < hidden) {
                        xa[j] = *reinterpret_cast<const f4 *>(xr + i);
                        gb[j] = *reinterpret_cast<const f4 *>(shexp_gate + i);
                    }
                }
#pragma unroll
                for (int j = 0; j < 8; j++)
                    if (base + 4 * lane + 256 * j < hidden)
                        dot += (xa[j][0] * gb[j][0] + xa[j][1] * gb[j][1]) + (xa[j][2] * gb[j][2] + xa[j][3] * gb[j][3]);
            }
        } else {
            for (int i = lane; i < hidden; i += 64) dot += xr[i] * shexp_gate[i];
        }
        dot = dfl_wave_sum(dot);
        if (shexp_gate && lane == 0) sg[row] = 1.0f / (1.0f + expf(-dot));

        float mx = -INFINITY;
#pragma unroll
        for (int j = 0; j < 4; j++) mx = fmaxf(mx, lgv[j]);
        for (int e = lane + 256; e < n_expert; e += 64) mx = fmaxf(mx, lg[e]);
        for (int off = 32; off > 0; off >>= 1) mx = fmaxf(mx, __shfl_xor(mx, off, 64));
        float sum = 0.0f;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            if (lane + 64 * j < n_expert) {
                const float ex = expf(lgv[j] - mx);
                pr[lane + 64 * j] = ex;
                sum += ex;
            }
        }
        for (int e = lane + 256; e < n_expert; e += 64) {
            const float ex = expf(lg[e] - mx);
            pr[e] = ex;
            sum += ex;
        }
        sum = dfl_wave_sum(sum);
        const float inv = 1.0f / sum;
        for (int e = lane; e < n_expert; e += 64) pr[e] *= inv;
    }
    if (tid < n_expert) rank[tid] = 0;
    __syncthreads();
    if (live) {
        // pick k = the best remaining expert: a wave-wide maximum over 64-bit keys (probability bits,
        // then ~id, so that equal probabilities go to the lower id); the winner's probability is
        // then marked taken (negative).  Same order as ranking every expert against all others, at
        // n_used * n_expert / 64 steps instead of n_expert^2 / 64.
        for (int k = 0; k < n_used; k++) {
            unsigned long long best = 0;
            for (int e = lane; e < n_expert; e += 64) {
                const float p = pr[e];
                const unsigned long long key = (static_cast<unsigned long long>(__float_as_uint(p)) << 32) | (0xffffffffu - static_cast<unsigned>(e));
                if (p >= 0.0f && key > best) best = key;
            }
            best = wave_max_u64(best);
            int e_win = static_cast<int>(0xffffffffu - static_cast<unsigned>(best));
            if (best == 0) e_win = k < n_expert ? k : n_expert - 1;  // nothing comparable left (NaN logits): stay in range
            if (lane == 0) {
                sel_e[row * n_used + k] = e_win;
                pick_e[row][k] = e_win;
                pick_w[row][k] = __uint_as_float(static_cast<unsigned>(best >> 32));
                rank[e_win] = 1;  // picked by some row
                pr[e_win] = -1.0f;
            }
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
        }
    }
    __syncthreads();
    if (live && lane == 0) {
        float wsum = 0.0f;
        for (int k = 0; k < n_used; k++) wsum += pick_w[row][k];  // in pick order, as the reference sums them
        wsum = fmaxf(wsum, 6.103515625e-05f);                     // 2^-14
        for (int k = 0; k < n_used; k++) sel_w[row * n_used + k] = pick_w[row][k] / wsum;
    }
    // distinct experts of the block
    const bool picked = tid < n_expert && rank[tid] != 0;
    const unsigned long long mask = __builtin_amdgcn_ballot_w64(picked);
    if (lane == 0) wave_count[row] = __popcll(mask);
    __syncthreads();
    int base = 0, total = 0;
    for (int w = 0; w < 16; w++) {
        if (w < row) base += wave_count[w];
        total += wave_count[w];
    }
    if (picked) {
        const int idx = base + __popcll(mask & ((1ull << lane) - 1));
        ids[idx] = tid;
        rank[tid] = idx;
    }
    if (tid == 0) {
        if (with_shared) ids[total] = -1;
        *n_slots = total + (with_shared ? 1 : 0);
    }
    __syncthreads();
    if (live && lane < n_used) slot_of[row * n_used + lane] = rank[pick_e[row][lane]];
}

// The same routing for n_expert <= 256, n_used <= 64, with a row's probabilities held in registers
// (four per lane) and one workgroup barrier in all: a row's picks stay in its wave (lane k keeps pick
// k), the row's picked experts go out as a 256-bit mask, and after the barrier every thread derives
// the block's ascending expert list and the slot of each pick from the union of the sixteen masks by
// population counts.  Same arithmetic, in the same order, as moe_route_kernel.
__global__ void __launch_bounds__(1024)
    moe_route_small_kernel(const float *__restrict__ logits, const float *__restrict__ x, const float *__restrict__ shexp_gate,
                           int n_rows, int n_expert, int n_used, int hidden, int with_shared, int32_t *__restrict__ sel_e,
                           float *__restrict__ sel_w, float *__restrict__ sg, int32_t *__restrict__ ids,
                           int32_t *__restrict__ n_slots, int32_t *__restrict__ slot_of) {
    typedef float f4 __attribute__((ext_vector_type(4)));
    __shared__ unsigned long long row_mask[16][4];
    const int tid = threadIdx.x, lane = tid & 63, row = tid >> 6;
    const bool live = row < n_rows;
    int my_e = 0;
    unsigned long long m[4] = {0, 0, 0, 0};
    if (live) {
        const float *lg = logits + static_cast<size_t>(row) * n_expert;
        const float *xr = x + static_cast<size_t>(row) * hidden;
        float dot = 0.0f;
        if (!shexp_gate) {
            // the gate was computed by the kernel that wrote x
        } else if (hidden % 4 == 0) {
            for (int base = 0; base < hidden; base += 2048) {
                f4 xa[8], gb[8];
#pragma unroll
                for (int j = 0; j < 8; j++) {
                    const int i = base + 4 * lane + 256 * j;
                    xa[j] = gb[j] = f4{0, 0, 0, 0};
                    if (i < hidden) {
                        xa[j] = *reinterpret_cast<const f4 *>(xr + i);
                        gb[j] = *reinterpret_cast<const f4 *>(shexp_gate + i);
                    }
                }
#pragma unroll
                for (int j = 0; j < 8; j++)
                    if (base + 4 * lane + 256 * j < hidden)
                        dot += (xa[j][0] * gb[j][0] + xa[j][1] * gb[j][1]) + (xa[j][2] * gb[j][2] + xa[j][3] * gb[j][3]);
            }
        } else {
            for (int i = lane; i < hidden; i += 64) dot += xr[i] * shexp_gate[i];
        }
        dot = dfl_wave_sum(dot);
        if (shexp_gate && lane == 0) sg[row] = 1.0f / (1.0f + expf(-dot));

        const dfl_route::RowPicks pk = dfl_route::route_row(lg, n_expert, n_used, lane);
        my_e = pk.my_e;
#pragma unroll
        for (int j = 0; j < 4; j++) m[j] = pk.m[j];
        if (lane < n_used) {
            sel_e[row * n_used + lane] = my_e;
            sel_w[row * n_used + lane] = pk.my_w;
        }
    }
    if (lane < 4) row_mask[row][lane] = m[lane & 3];
    __syncthreads();
    unsigned long long un[4];
    dfl_route::union_of_rows(&row_mask[0][0], lane, un);
    auto slot = [&](int e) { return dfl_route::slot_below(un, e); };  // experts below e in the union
    if (tid < n_expert && ((un[tid >> 6] >> (tid & 63)) & 1)) ids[slot(tid)] = tid;
    if (tid == 0) {
        const int total = __popcll(un[0]) + __popcll(un[1]) + __popcll(un[2]) + __popcll(un[3]);
        if (with_shared) ids[total] = -1;
        *n_slots = total + (with_shared ? 1 : 0);
    }
    if (live && lane < n_used) slot_of[row * n_used + lane] = slot(my_e);
}

// Collects the slots whose pick is `expert`; returns the count (uniform over the workgroup).
__device__ int collect_slots(const int32_t *__restrict__ sel_e, int n_slots, int expert, int *list, int *count) {
    if (threadIdx.x == 0) *count = 0;
    __syncthreads();
    for (int s = threadIdx.x; s < n_slots; s += blockDim.x)
        if (sel_e[s] == expert) list[atomicAdd(count, 1)] = s;
    __syncthreads();
    return *count;
}

// y[slot][o] = W_expert[o][:] . xin[src(slot)][:]  for the slots of this expert.
// GATE_UP: two stacked matrices, y = silu(gate) * up, xin row = slot / n_used (the block row).
// Otherwise: one matrix, xin row = slot.
// A row of n_in/32 sub-blocks is spread over LPR lanes (32 or 64); a wave does 64/LPR rows at once.
template <bool GATE_UP, int LPR>
__global__ void __launch_bounds__(256)
    moe_expert_kernel(int type, const uint8_t *__restrict__ w0, const uint8_t *__restrict__ w1, size_t row_bytes,
                      const float *__restrict__ xin, const int32_t *__restrict__ sel_e, int n_slots, int n_used, int n_in,
                      int n_out, float *__restrict__ y) {
    __shared__ int list[kMaxSlots];
    __shared__ int count;
    const int expert = blockIdx.y;
    const int n = collect_slots(sel_e, n_slots, expert, list, &count);
    if (n == 0) return;
    constexpr int kRowsPerWave = 64 / LPR;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int sub_lane = lane % LPR, sub_row = lane / LPR;
    const int n_sub = n_in / 32;
    const int rows_per_wg = 4 * kRowsPerWave * 4;  // 4 waves x rows at once x 4 passes
    const int o0 = blockIdx.x * rows_per_wg;
    const size_t expert_off = static_cast<size_t>(expert) * n_out * row_bytes;
    for (int pass = 0; pass < 4; pass++) {
        const int o = o0 + (pass * 4 + wave) * kRowsPerWave + sub_row;
        const bool live = o < n_out;
        const uint8_t *r0 = w0 + expert_off + static_cast<size_t>(live ? o : 0) * row_bytes;
        const uint8_t *r1 = GATE_UP ? w1 + expert_off + static_cast<size_t>(live ? o : 0) * row_bytes : nullptr;
        for (int s0 = 0; s0 < n; s0 += 4) {  // up to 4 slots share one dequantisation
            float acc0[4] = {0, 0, 0, 0}, acc1[4] = {0, 0, 0, 0};
            for (int sb = sub_lane; sb < n_sub; sb += LPR) {
                float wa[32], wb[32];
                dfl_dequant_sub32(type, r0, sb, wa);
                if (GATE_UP) dfl_dequant_sub32(type, r1, sb, wb);
#pragma unroll
                for (int t = 0; t < 4; t++) {
                    if (s0 + t >= n) break;
                    const int slot = list[s0 + t];
                    const float4 *xr = reinterpret_cast<const float4 *>(
                        xin + static_cast<size_t>(GATE_UP ? slot / n_used : slot) * n_in + 32 * sb);
#pragma unroll
                    for (int v = 0; v < 8; v++) {
                        const float4 xv = xr[v];
                        acc0[t] += wa[4 * v] * xv.x + wa[4 * v + 1] * xv.y + wa[4 * v + 2] * xv.z + wa[4 * v + 3] * xv.w;
                        if (GATE_UP)
                            acc1[t] += wb[4 * v] * xv.x + wb[4 * v + 1] * xv.y + wb[4 * v + 2] * xv.z + wb[4 * v + 3] * xv.w;
                    }
                }
            }
#pragma unroll
            for (int t = 0; t < 4; t++) {
                float a = acc0[t], b = acc1[t];
                for (int off = LPR / 2; off > 0; off >>= 1) {
                    a += __shfl_xor(a, off, 64);
                    if (GATE_UP) b += __shfl_xor(b, off, 64);
                }
                if (sub_lane == 0 && live && s0 + t < n) {
                    const float r = GATE_UP ? a / (1.0f + expf(-a)) * b : a;
                    y[static_cast<size_t>(list[s0 + t]) * n_out + o] = r;
                }
            }
        }
    }
}

// x[row] += sum_k w[row][k] * eo[row*n_used + k]  +  sg[row] * shared[row]
__global__ void moe_combine_kernel(const float *__restrict__ eo, const float *__restrict__ sel_w, const float *__restrict__ sg,
                                   const float *__restrict__ shared, int n_used, int hidden, float *__restrict__ x) {
    const int row = blockIdx.y;
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= hidden) return;
    float out = 0.0f;
    for (int k = 0; k < n_used; k++)
        out += sel_w[row * n_used + k] * eo[(static_cast<size_t>(row) * n_used + k) * hidden + i];
    out += sg[row] * shared[static_cast<size_t>(row) * hidden + i];
    x[static_cast<size_t>(row) * hidden + i] += out;
}

__global__ void silu_mul_rows_kernel(float *__restrict__ g, const float *__restrict__ u, size_t n) {
    size_t i = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i < n) {
        const float v = g[i];
        g[i] = v / (1.0f + expf(-v)) * u[i];
    }
}

// x[row] += sum_k w[row][k] * eo[slot_of[row][k]][row]  +  sg[row] * shared[row]
// (shared == nullptr: the shared expert's output is the last slot of eo)
__global__ void moe_combine_slots_kernel(const float *__restrict__ eo, const int32_t *__restrict__ slot_of,
                                         const float *__restrict__ sel_w, const float *__restrict__ sg,
                                         const float *__restrict__ shared, const int32_t *__restrict__ n_slots, int n_used,
                                         int hidden, float *__restrict__ x) {
    const int row = blockIdx.y;
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= hidden) return;
    float out = 0.0f;
    for (int k = 0; k < n_used; k++) {
        const size_t slot = slot_of[row * n_used + k];
        out += sel_w[row * n_used + k] * eo[(slot * 16 + row) * hidden + i];
    }
    const float sh = shared ? shared[static_cast<size_t>(row) * hidden + i]
                            : eo[((static_cast<size_t>(*n_slots) - 1) * 16 + row) * hidden + i];
    out += sg[row] * sh;
    x[static_cast<size_t>(row) * hidden + i] += out;
}

// The same, followed in the same pass by the RMSNorm that consumes x next (the following layer's
// attention norm or the output norm): y = x * rsqrt(mean(x^2) + eps) * norm_w.  One workgroup per
// row, the row (hidden <= 4096, a multiple of 4) in registers; element sums and the sum of squares
// are taken in the order of moe_combine_slots_kernel followed by the norm kernel.
// What bounds it: two trips to memory (the picks, then their rows) and what one CU can take in, (n_used + 3) rows of
// hidden values.  A thread asks for the rows of eight picks at once - unconditionally: past the last pick the last one
// again, its product left out - where a loop over the picks waited for one row at a time; the picks themselves are scalar
// loads (the same for the whole workgroup).  V: vectors of four values per thread.
template <int V, bool grouped>
__global__ void __launch_bounds__(256)
    moe_combine_norm_kernel(const float *__restrict__ eo, const int32_t *__restrict__ slot_of, const float *__restrict__ sel_w,
                            const float *__restrict__ sg, const float *__restrict__ shared, const int32_t *__restrict__ n_slots,
                            int n_used, int hidden, float *__restrict__ x, const float *__restrict__ norm_w,
                            float *__restrict__ y, float eps, const float *__restrict__ pre_add, void *__restrict__ y_xf,
                            int y_xf_kind, size_t xf_stride, float *__restrict__ cap, int cap_ld) {
    // (y: null where the rows go to fragment order; cap: the new residual's rows go there as well, cap_ld floats apart)
    typedef float f4 __attribute__((ext_vector_type(4)));
    __shared__ float sh[4];
    const int row = blockIdx.x, tid = threadIdx.x;
    const size_t row_at = static_cast<size_t>(row) * hidden;
    int at[V];
    f4 v[V], pre[V], nw[V], shv[V], out[V];
#pragma unroll
    for (int j = 0; j < V; j++) at[j] = min(4 * (tid + 256 * j), hidden - 4);
    // grouped (rows of several 16-row blocks, moe_group_slots_kernel): slot_of is the eo row of a pick itself, and the
    // shared expert's slots are the last gridDim.x / 16 (rounded up) of the list, one per block of rows
    const size_t n_slots_now = static_cast<size_t>(*n_slots);
    const float gate = sg[row];
    const size_t last = grouped ? (n_slots_now - (gridDim.x + 15) / 16 + (row >> 4)) * 16 + (row & 15) : (n_slots_now - 1) * 16 + row;
    const float *sh_row = shared ? shared + row_at : eo + last * hidden;
#pragma unroll
    for (int j = 0; j < V; j++) out[j] = f4{0, 0, 0, 0};
    for (int k0 = 0; k0 < n_used; k0 += 8) {
        const float *src[8];
        float wk[8];
#pragma unroll
        for (int k = 0; k < 8; k++) {
            const int pick = row * n_used + min(k0 + k, n_used - 1);
            wk[k] = sel_w[pick];
            src[k] = eo + static_cast<size_t>(grouped ? slot_of[pick] : slot_of[pick] * 16 + row) * hidden;
        }
        f4 e[8][V];
#pragma unroll
        for (int k = 0; k < 8; k++)
#pragma unroll
            for (int j = 0; j < V; j++) e[k][j] = *reinterpret_cast<const f4 *>(src[k] + at[j]);
        if (k0 == 0) {  // (what is needed after the picks, behind their rows in the order of issue)
#pragma unroll
            for (int j = 0; j < V; j++) {
                shv[j] = *reinterpret_cast<const f4 *>(sh_row + at[j]);
                v[j] = *reinterpret_cast<const f4 *>(x + row_at + at[j]);
                if (pre_add) pre[j] = *reinterpret_cast<const f4 *>(pre_add + row_at + at[j]);
                nw[j] = *reinterpret_cast<const f4 *>(norm_w + at[j]);
            }
            dfl_have(y, eps, y_xf, y_xf_kind, xf_stride, cap, cap_ld);
        }
#pragma unroll
        for (int k = 0; k < 8; k++) {
            if (k0 + k < n_used) {
#pragma unroll
                for (int j = 0; j < V; j++) out[j] += wk[k] * e[k][j];
            }
        }
    }
    float s = 0.0f;
#pragma unroll
    for (int j = 0; j < V; j++) {
        // (a residual term the norm before this layer's experts left out: it goes in first, as it would have there)
        if (pre_add) v[j] += pre[j];
        out[j] += gate * shv[j];
        v[j] += out[j];
        if (4 * (tid + 256 * j) >= hidden) v[j] = f4{0, 0, 0, 0};
        s += (v[j][0] * v[j][0] + v[j][1] * v[j][1]) + (v[j][2] * v[j][2] + v[j][3] * v[j][3]);
    }
    s = dfl_wave_sum(s);
    if ((tid & 63) == 0) sh[tid >> 6] = s;
#pragma unroll
    for (int j = 0; j < V; j++)
        if (4 * (tid + 256 * j) < hidden) {
            *reinterpret_cast<f4 *>(x + row_at + at[j]) = v[j];
            if (cap) *reinterpret_cast<f4 *>(cap + static_cast<size_t>(row) * cap_ld + at[j]) = v[j];
        }
    __syncthreads();
    s = ((sh[0] + sh[1]) + sh[2]) + sh[3];
    const float scale = 1.0f / sqrtf(s / static_cast<float>(hidden) + eps);
#pragma unroll
    for (int j = 0; j < V; j++) {
        const int i = 4 * (tid + 256 * j);
        if (i < hidden) {
            const f4 o = v[j] * scale * nw[j];
            if (y) *reinterpret_cast<f4 *>(y + row_at + i) = o;
            // (hidden a multiple of 256 here: whole waves are inside or outside the row)
            if (y_xf)
                dfl_xf_store_pair(static_cast<uint8_t *>(y_xf) + (row >> 4) * xf_stride, y_xf_kind, row & 15, i & ~7, o[0], o[1], o[2], o[3]);
        }
    }
}

void moe_combine_norm(int rows, hipStream_t st, const float *eo, const int32_t *slot_of, const float *sel_w, const float *sg, const float *shared,
                      const int32_t *n_slots, int n_used, int hidden, float *x, const float *norm_w, float *y, float eps, const float *pre_add,
                      void *y_xf, int y_xf_kind, bool grouped, size_t xf_stride, float *cap, int cap_ld) {
#define DFL_COMBINE(V) (grouped ? moe_combine_norm_kernel<V, true> : moe_combine_norm_kernel<V, false>)
    const auto fn = hidden <= 1024 ? DFL_COMBINE(1) : hidden <= 2048 ? DFL_COMBINE(2) : DFL_COMBINE(4);
#undef DFL_COMBINE
    fn<<<rows, 256, 0, st>>>(eo, slot_of, sel_w, sg, shared, n_slots, n_used, hidden, x, norm_w, y_xf ? nullptr : y, eps, pre_add, y_xf, y_xf_kind, xf_stride, cap, cap_ld);
}

// ---- rows of several 16-row blocks through one pass over the experts (prefill) ----
//
// A block of 16 rows touches 60-80 of 128 experts, so block after block re-reads most of a layer's expert weights;
// 256 rows touch all of them about once.  The rows are therefore regrouped by expert: a slot is (expert, up to sixteen
// of the rows that picked it), the expert kernels run their per-slot-activations mode over gathered copies of those
// rows, and every row then sums its picks' outputs in pick order.  A (row, expert) product is one wave's whole-K sum
// over the row's own activations, so it has the bits it has when the row's block runs alone.

// Picks of every row: wave w of workgroup b routes row 16 b + w (dfl_route::route_row, as in the block kernels).
__global__ void __launch_bounds__(1024)
    moe_group_route_kernel(const float *__restrict__ logits, int n_rows, int n_expert, int n_used, int32_t *__restrict__ sel_e,
                           float *__restrict__ sel_w) {
    const int lane = threadIdx.x & 63, row = blockIdx.x * 16 + (threadIdx.x >> 6);
    if (row >= n_rows) return;
    const dfl_route::RowPicks pk = dfl_route::route_row(logits + static_cast<size_t>(row) * n_expert, n_expert, n_used, lane);
    if (lane < n_used) {
        sel_e[row * n_used + lane] = pk.my_e;
        sel_w[row * n_used + lane] = pk.my_w;
    }
}

// The slot list of a group of rows.  Expert e with c picks gets ceil(c / 16) consecutive slots, experts in ascending
// order; behind them one slot per block of sixteen rows for the shared expert (rows 16 b .. 16 b + 15).
//   *n_slots;  slot_rows[slot][16]: the rows whose activations the slot multiplies (unused places repeat
//   row 0: computed, never read);  pick_pos[row][k] = 16 slot + place of the pick's output row;
//   tiles[*n_tiles] = {expert (-1: the shared one), first slot, slots, 0}: an expert's slots in runs of at most tile_slots, as
//   even as they come (a tile of one slot unpacks its weights for that one alone), the row tiles of the expert products.
// Places inside an expert's slots are handed out by an atomic counter, so they vary from run to run; no sum does.
// One workgroup; n_rows * n_used <= 1024 kGroupPicksPerThread, n_expert <= 256.
constexpr int kGroupPicksPerThread = 16;
__global__ void __launch_bounds__(1024)
    moe_group_slots_kernel(const int32_t *__restrict__ sel_e, int n_rows, int n_used, int n_expert, int32_t *__restrict__ n_slots,
                           int32_t *__restrict__ slot_rows, int32_t *__restrict__ pick_pos, int4 *__restrict__ tiles,
                           int32_t *__restrict__ n_tiles, int max_slots, int tile_slots, uint32_t by_used) {
    __shared__ int cnt[256], base[257], wave_s[4], wave_t[4];
    // the experts' slot rows are put together here and leave in whole lines: a row's place is anywhere, and 16384 stores of four
    // bytes to a line each were 7 us of one CU's address path (16.4 us a launch, 12.5 now, at 2048 rows of 8 picks)
    extern __shared__ __attribute__((aligned(16))) int32_t rows_sh[];
    const int tid = threadIdx.x, lane = tid & 63;
    if (tid < 256) cnt[tid] = 0;
    __syncthreads();
    const int n_picks = n_rows * n_used;
    int my_e[kGroupPicksPerThread], my_place[kGroupPicksPerThread];
#pragma unroll
    for (int j = 0; j < kGroupPicksPerThread; j++) {
        const int p = tid + 1024 * j;
        my_e[j] = p < n_picks ? min(max(sel_e[p], 0), n_expert - 1) : -1;
    }
#pragma unroll
    for (int j = 0; j < kGroupPicksPerThread; j++) my_place[j] = my_e[j] >= 0 ? atomicAdd(&cnt[my_e[j]], 1) : 0;
    __syncthreads();
    // exclusive prefix sums over the experts of their slots and of their row tiles (four waves, then across them)
    const int c = tid < n_expert ? cnt[tid] : 0, ns = (c + 15) >> 4, nt = (ns + tile_slots - 1) / tile_slots;
    int ps = ns, pt = nt;
    for (int off = 1; off < 64; off <<= 1) {
        const int us = __shfl_up(ps, off, 64), ut = __shfl_up(pt, off, 64);
        if (lane >= off) {
            ps += us;
            pt += ut;
        }
    }
    if (tid < 256 && lane == 63) {
        wave_s[tid >> 6] = ps;
        wave_t[tid >> 6] = pt;
    }
    __syncthreads();
    int total = 0, total_t = 0;
    for (int w = 0; w < 4; w++) {
        if (w < (tid >> 6)) {
            ps += wave_s[w];
            pt += wave_t[w];
        }
        total += wave_s[w];
        total_t += wave_t[w];
    }
    if (tid < n_expert) base[tid] = ps - ns;
    const int n_blocks = (n_rows + 15) >> 4, shared_t = (n_blocks + tile_slots - 1) / tile_slots;
    if (tid == 0) {
        *n_slots = min(total + n_blocks, max_slots);  // (the host sizes max_slots for the worst case)
        *n_tiles = total_t + shared_t;
    }
    if (tid < n_expert) {
        const int b = ps - ns;
        for (int t = 0; t < nt; t++) {
            const int first = ns * t / nt;
            tiles[pt - nt + t] = int4{tid, b + first, ns * (t + 1) / nt - first, 0};
        }
        if (c & 15)
            for (int m = c & 15; m < 16; m++) rows_sh[(b + (c >> 4)) * 16 + m] = 0;
    }
    for (int t = tid; t < shared_t; t += 1024) {
        const int first = n_blocks * t / shared_t;
        tiles[total_t + t] = int4{-1, total + first, n_blocks * (t + 1) / shared_t - first, 0};
    }
    for (int r = tid; r < 16 * n_blocks; r += 1024) slot_rows[total * 16 + r] = min(r, n_rows - 1);
    __syncthreads();
#pragma unroll
    for (int j = 0; j < kGroupPicksPerThread; j++) {
        if (my_e[j] >= 0) {
            const int p = tid + 1024 * j;
            const int at = (base[my_e[j]] + (my_place[j] >> 4)) * 16 + (my_place[j] & 15);
            rows_sh[at] = n_used == 1 ? p : static_cast<int>(__umulhi(p, by_used));  // p / n_used
            pick_pos[p] = at;
        }
    }
    __syncthreads();
    for (int i = tid; i < 4 * total; i += 1024) reinterpret_cast<int4 *>(slot_rows)[i] = reinterpret_cast<const int4 *>(rows_sh)[i];
}

// A slot's rows in fragment order (kind Q4K) with their sub-block sums, rounded to f16 as every few-row kernel rounds its
// activations: one wave per (super-block, slot).  Lane (m, q) reads sixteenths of 64 bytes of row m, the q-th 16 of each, so a load
// takes half lines of sixteen rows; in the output it has the 64 values of chunk q, the (4 x 4) blocks of the four lanes of a row
// being exchanged by swaps of lanes 32 and 16 apart.  (Each lane its own 64 values: 64 lines a load, the address path's 16 us of 30
// at 2048 rows of 8 picks; 25.5 now, the 90 MB it writes being most of it.)
__global__ void __launch_bounds__(64)
    moe_group_gather_kernel(const float *__restrict__ cur, const int32_t *__restrict__ slot_rows, const int32_t *__restrict__ n_slots,
                            int hidden, uint8_t *__restrict__ xg, uint8_t *__restrict__ sums) {
    typedef _Float16 h2 __attribute__((ext_vector_type(2)));
    const int b = blockIdx.x, slot = blockIdx.y, lane = threadIdx.x, m = lane & 15, q = lane >> 4, nb = hidden >> 8;
    if (slot >= *n_slots) return;
    const float4_t *src = reinterpret_cast<const float4_t *>(cur + static_cast<size_t>(slot_rows[slot * 16 + m]) * hidden + 256 * b) + q;
    half8_t *dst = reinterpret_cast<half8_t *>(xg + (static_cast<size_t>(slot) * nb + b) * 8192) + lane;
    float4_t v[16];
#pragma unroll
    for (int i = 0; i < 16; i++) v[i] = src[4 * i];
    // p[c][2 j + k]: pair k of the four values 64 c + 16 j + 4 q
    float p[4][8];
#pragma unroll
    for (int i = 0; i < 16; i++) {
        p[i >> 2][2 * (i & 3)] = __builtin_bit_cast(float, h2{static_cast<_Float16>(v[i][0]), static_cast<_Float16>(v[i][1])});
        p[i >> 2][2 * (i & 3) + 1] = __builtin_bit_cast(float, h2{static_cast<_Float16>(v[i][2]), static_cast<_Float16>(v[i][3])});
    }
#pragma unroll
    for (int e = 0; e < 8; e++) {
        dfl_swap32(p[0][e], p[2][e]);  // chunks 0 and 1 to the lower lanes, 2 and 3 to the upper, of the other half's lane in p[2], p[3]
        dfl_swap32(p[1][e], p[3][e]);
        dfl_swap16(p[0][e], p[1][e]);
        dfl_swap16(p[2][e], p[3][e]);
    }
    // p[k]: what lane k of the row had of this lane's chunk
    float o[8];
#pragma unroll
    for (int t = 0; t < 8; t++) {
        const h2 a = __builtin_bit_cast(h2, p[2 * (t & 1)][t & ~1]), c = __builtin_bit_cast(h2, p[2 * (t & 1)][(t & ~1) + 1]);
        const h2 d = __builtin_bit_cast(h2, p[2 * (t & 1) + 1][t & ~1]), f = __builtin_bit_cast(h2, p[2 * (t & 1) + 1][(t & ~1) + 1]);
        const _Float16 h[8] = {a[0], a[1], c[0], c[1], d[0], d[1], f[0], f[1]};
        const half8_t frag = {h[0], h[2], h[1], h[3], h[4], h[6], h[5], h[7]};
        dst[t * 64] = frag;
        o[t] = q4k_octet_sum_seq(h);
    }
    const half8_t r = q4k_sum_operand((o[0] + o[1]) + (o[2] + o[3]), (o[4] + o[5]) + (o[6] + o[7]));
    reinterpret_cast<half8_t *>(sums + (static_cast<size_t>(slot) * nb + b) * 1024)[lane] = r;
}

}  // namespace

namespace {
// whether the layer's expert stacks take the batched launches (one streaming GEMM per projection over the distinct experts)
bool moe_batched(const dflash_model_cfg &c, const dflash_layer &L) {
    static const bool per_slot_forced = getenv("DFLASH_MOE_PERSLOT") != nullptr;  // read once per process
    const int et = L.gate_exps.type, dt = L.down_exps.type;
    const bool tiled = et == DFLASH_TYPE_Q4_K_TILED;
    return (tiled || (et == DFLASH_TYPE_Q4_K && dt == DFLASH_TYPE_Q4_K)) && c.hidden % DFL_QK_K == 0 && c.ffn_expert % DFL_QK_K == 0 &&
           !per_slot_forced;
}
}  // namespace

bool dfl_moe_norm_fusable(const dflash_ctx *ctx, const dflash_model_cfg &c, const dflash_layer &L, int n) {
    // the residual term is added back by moe_combine_norm_kernel, which the batched path ends with
    return c.n_expert > 0 && L.shexp_gate && L.router.data && L.gate_exps.data && L.down_exps.data && moe_batched(c, L) &&
           c.hidden <= 4096 && c.hidden % 4 == 0 && dfl_router_norm_fits(ctx, L.router.type, L.router.data, c.hidden, c.n_expert, n);
}

int32_t dfl_moe_ffn(dflash_ctx *ctx, const dflash_model_cfg &c, const dflash_layer &L, float *cur, int n,
                    const dfl_moe_scratch &s, float *x_resid, bool gate_done, const float *next_norm_w, float *next_cur,
                    bool *next_done, hipStream_t st, const float *pre_add, const float *pre_norm_w, void *next_xf, int next_xf_kind, float *cap, int cap_ld) {
    if (next_done) *next_done = false;
    if ((pre_add != nullptr) != (pre_norm_w != nullptr) ||
        (pre_add && !(next_norm_w && next_cur && next_done && dfl_moe_norm_fusable(ctx, c, L, n))))
        return dfl_fail(ctx, DFLASH_ERR_INVALID_INPUT, "moe: the norm can ride in the router's launch only where dfl_moe_norm_fusable() holds");
    const int E = c.n_expert, used = c.n_expert_used < E ? c.n_expert_used : E;
    const int H = c.hidden, fe = c.ffn_expert, fs = c.ffn_shared;
    const int n_slots = n * used;
    if (used < 1 || used > 64 || E > 8192 || fe % 32 || H % 32)
        return dfl_fail(ctx, DFLASH_ERR_UNSUPPORTED, "moe: n_expert %d / n_expert_used %d / ffn_expert %d unsupported", E, used, fe);
    if (!L.router.data || !L.gate_exps.data || !L.up_exps.data || !L.down_exps.data || !L.shexp_gate || !L.gate.data ||
        !L.up.data || !L.down.data)
        return dfl_fail(ctx, DFLASH_ERR_INVALID_INPUT,
                        "moe: a mixture-of-experts layer needs router, gate/up/down_exps, shexp_gate and the shared expert's gate/up/down");
    const int et = L.gate_exps.type;
    const bool tiled = et == DFLASH_TYPE_Q4_K_TILED;  // every expert matrix repacked on its own (stack stride = tiled size)
    if (et != L.up_exps.type || (et != DFLASH_TYPE_Q4_K && et != DFLASH_TYPE_Q6_K && et != DFLASH_TYPE_Q8_0 && !tiled))
        return dfl_fail(ctx, DFLASH_ERR_UNSUPPORTED, "moe: expert weight type %d", et);
    const int dt = L.down_exps.type;
    if ((dt != DFLASH_TYPE_Q4_K && dt != DFLASH_TYPE_Q6_K && dt != DFLASH_TYPE_Q8_0 && dt != DFLASH_TYPE_Q4_K_TILED) ||
        (dt == DFLASH_TYPE_Q4_K_TILED) != tiled)
        return dfl_fail(ctx, DFLASH_ERR_UNSUPPORTED, "moe: expert weight types %d / %d (tiled stacks go together)", et, dt);
    const size_t rb_in = dflash_row_bytes(et, H), rb_dn = dflash_row_bytes(dt, fe);
    if (rb_in == 0 || rb_dn == 0) return dfl_fail(ctx, DFLASH_ERR_BAD_SHAPE, "moe: row sizes do not fit the block size");

    int32_t rc;
    if (pre_add) {
        rc = dfl_router_norm(ctx, L.router.data, x_resid, pre_add, pre_norm_w, L.shexp_gate, c.eps, cur, s.sg, s.probs, H, E, n, st);
        gate_done = true;
    } else {
        rc = dfl_gemm_fewrow_checked(ctx, L.router.type, L.router.data, cur, DFLASH_TYPE_F32, s.probs, H, E, n, st);
    }
    if (rc) return rc;
    if (E > 1024) return dfl_fail(ctx, DFLASH_ERR_UNSUPPORTED, "moe: %d experts (at most 1024)", E);
    const bool batched = moe_batched(c, L);
    if (tiled && !batched) return dfl_fail(ctx, DFLASH_ERR_UNSUPPORTED, "moe: tiled expert stacks need the batched path");
    // the shared expert rides along as one more slot of the batched GEMMs when it has the experts' shape (and order)
    const bool folded_shared = batched && fs == fe && L.gate.type == et && L.up.type == et && L.down.type == et;
    const size_t stride_in = tiled ? dflash_q4k_tiled_bytes(H, fe) : static_cast<size_t>(fe) * rb_in;
    const size_t stride_dn = tiled ? dflash_q4k_tiled_bytes(fe, H) : static_cast<size_t>(H) * rb_dn;
    const size_t route_lds = static_cast<size_t>(17) * E * sizeof(float);
    if (route_lds > 48 * 1024) {
        if (const int32_t rc_ = dfl_raise_lds_limit(ctx, reinterpret_cast<const void *>(moe_route_kernel), 17 * 1024 * sizeof(float)))
            return rc_;
    }
    const float *gate_w = gate_done ? nullptr : L.shexp_gate;  // null: sg is already there
    // the routing can ride in the gate/up launch (every workgroup derives the expert list itself): one launch fewer
    const bool route_inside = batched && tiled && !gate_w && n <= 16 &&
                              dfl_q4k_batched_can_route(ctx, 1, fe, E, used);
    if (route_inside) {
        // nothing to launch here
    } else if (E <= 256)
        moe_route_small_kernel<<<1, 1024, 0, st>>>(s.probs, cur, gate_w, n, E, used, H, folded_shared ? 1 : 0, s.sel_e,
                                                   s.sel_w, s.sg, s.ids, s.n_distinct, s.slot_of);
    else
        moe_route_kernel<<<1, 1024, route_lds, st>>>(s.probs, cur, gate_w, n, E, used, H, folded_shared ? 1 : 0,
                                                     s.sel_e, s.sel_w, s.sg, s.ids, s.n_distinct, s.slot_of);
    if (batched) {
        // the selected experts' matrices form one streaming GEMM each for gate, up and down: every
        // distinct expert's weights are read once, with all block rows riding along on the MFMA;
        // no split K, so a row's result is the same whichever other experts the block uses
        const bool fold = folded_shared;
        const int max_slots = (n_slots < E ? n_slots : E) + (fold ? 1 : 0);
        const size_t per_slot = static_cast<size_t>(16) * fe;
        // gate and up of every selected expert in one launch, silu(gate) * up applied to the tiles
        // while they are still in registers
        // (handed to the down product as f16 where the path writes it: the down kernel rounds its activations to f16
        // as it loads them, so the bits it computes with are the same and the hand-off is half the size)
        const int32_t mid_type = dfl_q4k_batched_f16_out(ctx, tiled ? 1 : 0, 1, fe) ? DFLASH_TYPE_F16 : DFLASH_TYPE_F32;
        const dfl_route_args route = {s.probs, E, used, folded_shared ? 1 : 0, s.sel_e, s.sel_w, s.slot_of};
        if ((rc = dfl_gemm_q4k_batched(ctx, L.gate_exps.data, stride_in, fold ? L.gate.data : nullptr, s.ids,
                                       s.n_distinct, max_slots, cur, DFLASH_TYPE_F32, 0, s.gate_out, mid_type, per_slot, H, fe, n, 1,
                                       L.up_exps.data, fold ? L.up.data : nullptr, tiled ? 1 : 0, st, route_inside ? &route : nullptr)))
            return rc;
        if ((rc = dfl_gemm_q4k_batched(ctx, L.down_exps.data, stride_dn, fold ? L.down.data : nullptr, s.ids,
                                       s.n_distinct, max_slots, s.gate_out, mid_type, per_slot, s.eo, DFLASH_TYPE_F32,
                                       static_cast<size_t>(16) * H, fe, H, n, 1, nullptr, nullptr, tiled ? 1 : 0, st)))
            return rc;
    } else {
        {
            dim3 grid(1, E);  // x: 16 * (64 / LPR) output rows per workgroup
            const int n_sub = H / 32;
            if (n_sub <= 32) {
                grid.x = (fe + 31) / 32;
                moe_expert_kernel<true, 32><<<grid, 256, 0, st>>>(et, static_cast<const uint8_t *>(L.gate_exps.data),
                                                                 static_cast<const uint8_t *>(L.up_exps.data), rb_in, cur, s.sel_e,
                                                                 n_slots, used, H, fe, s.act);
            } else {
                grid.x = (fe + 15) / 16;
                moe_expert_kernel<true, 64><<<grid, 256, 0, st>>>(et, static_cast<const uint8_t *>(L.gate_exps.data),
                                                                 static_cast<const uint8_t *>(L.up_exps.data), rb_in, cur, s.sel_e,
                                                                 n_slots, used, H, fe, s.act);
            }
        }
        {
            dim3 grid(1, E);
            const int n_sub = fe / 32;
            if (n_sub <= 32) {
                grid.x = (H + 31) / 32;
                moe_expert_kernel<false, 32><<<grid, 256, 0, st>>>(dt, static_cast<const uint8_t *>(L.down_exps.data), nullptr, rb_dn,
                                                                  s.act, s.sel_e, n_slots, used, fe, H, s.eo);
            } else {
                grid.x = (H + 15) / 16;
                moe_expert_kernel<false, 64><<<grid, 256, 0, st>>>(dt, static_cast<const uint8_t *>(L.down_exps.data), nullptr, rb_dn,
                                                                  s.act, s.sel_e, n_slots, used, fe, H, s.eo);
            }
        }
    }
    if (!folded_shared) {  // shared expert: plain dense SwiGLU through the few-row GEMM
        if ((rc = dfl_gemm_fewrow_checked(ctx, L.gate.type, L.gate.data, cur, DFLASH_TYPE_F32, s.g, H, fs, n, st))) return rc;
        if ((rc = dfl_gemm_fewrow_checked(ctx, L.up.type, L.up.data, cur, DFLASH_TYPE_F32, s.u, H, fs, n, st))) return rc;
        const size_t nf = static_cast<size_t>(n) * fs;
        silu_mul_rows_kernel<<<static_cast<unsigned>((nf + 255) / 256), 256, 0, st>>>(s.g, s.u, nf);
        if ((rc = dfl_gemm_fewrow_checked(ctx, L.down.type, L.down.data, s.g, DFLASH_TYPE_F32, s.shared, fs, H, n, st))) return rc;
    }
    if (batched && next_norm_w && next_cur && next_done && H <= 4096 && H % 4 == 0) {
        moe_combine_norm(n, st, s.eo, s.slot_of, s.sel_w, s.sg, folded_shared ? nullptr : s.shared, s.n_distinct,
                                                   used, H, x_resid, next_norm_w, next_cur, c.eps, pre_add,
                                                   H % DFL_QK_K == 0 ? next_xf : nullptr, next_xf_kind, false, 0, cap, cap_ld);
        *next_done = true;
    } else if (batched)
        moe_combine_slots_kernel<<<dim3((H + 255) / 256, n), 256, 0, st>>>(s.eo, s.slot_of, s.sel_w, s.sg,
                                                                         folded_shared ? nullptr : s.shared, s.n_distinct, used,
                                                                         H, x_resid);
    else
        moe_combine_kernel<<<dim3((H + 255) / 256, n), 256, 0, st>>>(s.eo, s.sel_w, s.sg, s.shared, used, H, x_resid);
    DFL_HIP_CHECK(ctx, hipGetLastError());
    return DFLASH_OK;
}

int dfl_moe_group_max_picks() { return 1024 * kGroupPicksPerThread; }

int dfl_moe_group_max_slots(const dflash_model_cfg &c, int n_rows) {
    const int used = c.n_expert_used < c.n_expert ? c.n_expert_used : c.n_expert;
    const int picks = n_rows * used;
    // sum over experts of ceil(count / 16) <= distinct experts + picks / 16, and one shared-expert slot per block
    return (picks < c.n_expert ? picks : c.n_expert) + picks / 16 + (n_rows + 15) / 16;
}

bool dfl_moe_group_fits(const dflash_ctx *ctx, const dflash_model_cfg &c, const dflash_layer &L, int n_rows) {
    const int E = c.n_expert, used = c.n_expert_used < E ? c.n_expert_used : E;
    const bool tiled = L.gate_exps.type == DFLASH_TYPE_Q4_K_TILED && L.up_exps.type == DFLASH_TYPE_Q4_K_TILED &&
                       L.down_exps.type == DFLASH_TYPE_Q4_K_TILED;
    const bool folded = c.ffn_shared == c.ffn_expert && L.gate.type == DFLASH_TYPE_Q4_K_TILED && L.up.type == DFLASH_TYPE_Q4_K_TILED &&
                        L.down.type == DFLASH_TYPE_Q4_K_TILED;
    return E >= 1 && E <= 256 && used >= 1 && used <= 64 && n_rows >= 1 && n_rows * used <= 1024 * kGroupPicksPerThread && tiled && folded &&
           c.hidden % DFL_QK_K == 0 && c.ffn_expert % DFL_QK_K == 0 && c.hidden <= 4096 && L.shexp_gate && L.router.data &&
           dfl_router_norm_fits(ctx, L.router.type, L.router.data, c.hidden, E, 16) &&
           dfl_q4k_batched_f16_out(ctx, 1, 1, c.ffn_expert);
}

int32_t dfl_moe_ffn_group(dflash_ctx *ctx, const dflash_model_cfg &c, const dflash_layer &L, float *x_resid,
                          float *cur, int n_rows, const dfl_moe_group_scratch &s, const float *next_norm_w, void *next_xf,
                          int next_xf_kind, size_t next_xf_stride, hipStream_t st, float *cap, int cap_ld) {
    if (!dfl_moe_group_fits(ctx, c, L, n_rows) || !x_resid || !cur || !next_norm_w)
        return dfl_fail(ctx, DFLASH_ERR_UNSUPPORTED, "moe group: layer or row count (%d) not taken", n_rows);
    const int E = c.n_expert, used = c.n_expert_used < E ? c.n_expert_used : E, H = c.hidden, fe = c.ffn_expert;
    const int max_slots = dfl_moe_group_max_slots(c, n_rows);
    if (max_slots > s.max_slots) return dfl_fail(ctx, DFLASH_ERR_INVALID_INPUT, "moe group: scratch sized for %d slots, %d needed", s.max_slots, max_slots);
    int32_t rc;
    if ((rc = dfl_router_rows(ctx, L.router.data, cur, s.logits, H, E, n_rows, st))) return rc;
    moe_group_route_kernel<<<(n_rows + 15) / 16, 1024, 0, st>>>(s.logits, n_rows, E, used, s.sel_e, s.sel_w);
    // Row tiles of eight blocks (a workgroup of eight waves fills a CU) take in half the weights and fewer activations for a
    // product, those of four (two workgroups on a CU) hide each other's waits, leave less of a tile empty and make more
    // workgroups.  Eight where an expert has 85 rows on average and the experts alone are two rounds of the chip in the
    // narrower product.  A layer in us, 4 : 8 (hidden 2048; 94 pairs over 14 mixtures of 8 to 256 experts; the better side, or
    // within 7 us of it, in all but two, 9 and 11 us):
    //   two rounds, 80 / 90 / 100 / 128 rows an expert: 128 experts top-8 FFN 768 482 : 481, 519 : 514, 563 : 550, 693 : 677;
    //               64 top-6 of 1536 388 : 390, 410 : 402, 467 : 454, 552 : 543 (50 rows 287 : 308)
    //   fewer, 80 / 100 / 130 / 200 rows: 8 top-2 of 3584 183 : 197, 209 : 216, 254 : 256, 332 : 325; 32 top-4 of 2048 296 : 307,
    //               340 : 338, 422 : 419, 565 : 554; 64 top-8 of 512 249 : 262, 293 : 300, 367 : 370, 482 : 485; 48 top-4 of 1024 323 : 320,
    //               385 : 385, 468 : 468, 575 : 590
    const int narrow_ct = std::min(fe / 128, H / 256);  // column tiles of the narrower product, gate and up or down
    const int tile_slots = n_rows * used >= 85 * E && E * narrow_ct >= 2 * ctx->n_cu ? 8 : 4;
    const size_t slots_lds = static_cast<size_t>(max_slots - (n_rows + 15) / 16) * 16 * sizeof(int32_t);  // (at most 1280 slots of experts)
    if ((rc = dfl_raise_lds_limit(ctx, reinterpret_cast<const void *>(moe_group_slots_kernel), slots_lds))) return rc;
    moe_group_slots_kernel<<<1, 1024, slots_lds, st>>>(s.sel_e, n_rows, used, E, s.n_slots, s.slot_rows, s.pick_pos, reinterpret_cast<int4 *>(s.tiles),
                                                     s.n_tiles, max_slots, tile_slots,
                                                     static_cast<uint32_t>(((1ull << 32) + used - 1) / used));  // (exact: picks x used < 2^32)
    moe_group_gather_kernel<<<dim3(H / DFL_QK_K, max_slots), 64, 0, st>>>(cur, s.slot_rows, s.n_slots, H, s.xg, s.xg_sums);
    const size_t stride_in = dflash_q4k_tiled_bytes(H, fe), stride_dn = dflash_q4k_tiled_bytes(fe, H);
    // most row tiles the list can have: one per tile_slots slots, and a short one per expert and for the shared one
    const int max_tiles = std::min(max_slots, max_slots / tile_slots + E + 1);
    if ((rc = dfl_gemm_rows_experts(ctx, L.gate_exps.data, L.gate.data, L.up_exps.data, L.up.data, stride_in, s.xg, s.xg_sums, s.tiles, s.n_tiles,
                                    max_tiles, tile_slots, nullptr, H, fe, s.act, s.act_sums, st)))
        return rc;
    if ((rc = dfl_gemm_rows_experts(ctx, L.down_exps.data, L.down.data, nullptr, nullptr, stride_dn, s.act, s.act_sums, s.tiles, s.n_tiles,
                                    max_tiles, tile_slots, s.eo, fe, H, nullptr, nullptr, st)))
        return rc;
    moe_combine_norm(n_rows, st, s.eo, s.pick_pos, s.sel_w, s.sg, nullptr, s.n_slots, used, H, x_resid, next_norm_w,
                                                    cur, c.eps, nullptr, next_xf, next_xf_kind, true, next_xf_stride, cap, cap_ld);
    DFL_HIP_CHECK(ctx, hipGetLastError());
    return DFLASH_OK;
}
