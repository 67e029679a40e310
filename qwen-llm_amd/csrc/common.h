// Internal declarations shared by the HIP translation units of libdflash_hip.
#pragma once

#include <hip/hip_runtime.h>
#include <hip/hip_fp16.h>

#include <cstdarg>
#include <cstdint>
#include <cstdio>
#include <vector>

#include "../../include/dflash_hip.h"

struct dflash_ctx {
    int device = 0;
    char *workspace = nullptr;  // device scratch, owned
    size_t workspace_bytes = 0;
    int n_cu = 256;
    // split-K partial tiles of the Q4_K GEMM (written by the streaming kernel, added up by its reduce kernel)
    void *partials = nullptr;
    int n_partial_wgs = 0;
    // workgroups of a batched (expert) launch; 0 = one per CU.  The pipelined prefill sets it on its lanes' contexts for
    // the duration of a call: an expert workgroup fills a CU's LDS, so launches of different lanes cannot share a CU,
    // and with half the CUs each two of them run side by side, one's start-up and tail under the other's streaming.
    int batch_wgs = 0;
    size_t lds_bytes = 65536;  // LDS available to one workgroup
    char err[512] = {0};
    // per-kernel timers (off by default; when on, timed launches synchronise)
    bool timing = false;
    // Set by a caller inside the library for the duration of one few-row GEMM call on a fused gate | up matrix
    // (2 ffn output rows, ffn a multiple of 16): if the call is split over K, its reduction writes
    // silu(gate) * up to swiglu_out[n_rows][ffn] instead of the sums to Y and sets swiglu_done; if it is not (Y is
    // complete), swiglu_done stays false and the caller applies the activation itself.
    float *swiglu_out = nullptr;
    bool swiglu_done = false;
    hipEvent_t ev0 = nullptr, ev1 = nullptr;
    // start / stop stamps of single dispatches (hipExtLaunchKernelGGL), see DFL_T_KERNEL_*: while `stamping` is on, a stamped
    // launch takes the next event pair of the pool and does not wait; the pairs are read when the timers are queried
    bool stamping = false;
    std::vector<hipEvent_t> stamp_events;  // pairs
    std::vector<int> stamp_slot;           // slot of pair i
    size_t stamps_used = 0;
    double timed_ms[8] = {0};
    int64_t timed_launches[8] = {0};
    // captured-graph replay of the packed verify: a stream of the library's own to capture on and
    // launch into (the caller's may be the legacy default stream, which cannot be captured) and
    // the two events that order it against the caller's stream
    bool graphs = false;
    bool capturing = false;     // the launches being enqueued go into a graph: position-dependent values come from device memory
    bool draft_graphs = false;  // graph replay of the drafter's block forward (measured: no faster than direct launches)
    hipStream_t gstream = nullptr;
    hipEvent_t g_in = nullptr, g_out = nullptr;
    // pinned host staging for the few words a blocking call reads back (a device-to-host copy into pageable
    // memory is staged by the runtime and costs several microseconds each); one page, owned
    void *pinned = nullptr;
    void *pinned_dev = nullptr;  // its address on the device (null: the device cannot write it)
    // kernels whose dynamic-LDS limit has already been raised for this context (the attribute is kept per
    // device by the runtime, so the record lives with the context, not in process-wide flags)
    const void *lds_attr_fn[96] = {nullptr};
    size_t lds_attr_bytes[96] = {0};
    int n_lds_attr = 0;
};
enum { DFL_PINNED_BYTES = 8192 };

// Slots of the per-kernel timers.
enum { DFL_T_GEMM = 0, DFL_T_ATTN = 1, DFL_T_ACCEPT = 2, DFL_T_ARGMAX = 3, DFL_T_REDUCE = 4,
       // the kernel of a single Q4_K product and the tiled order's reduction by the device's own start / stop stamps of that one dispatch (what a
       // kernel trace reports as its duration), not by events recorded around the launch (which add the dispatch latency)
       DFL_T_KERNEL_Q4K_TILED = 5, DFL_T_KERNEL_Q4K_REDUCE = 6 };

// Brackets the dominant kernel of a call with events on its stream when timing is on.
// The event pair a stamped launch passes to hipExtLaunchKernelGGL: null pointers while stamping is off.
struct dfl_stamp {
    hipEvent_t start = nullptr, stop = nullptr;
    dfl_stamp(dflash_ctx *ctx, int slot) {
        if (!ctx->stamping) return;
        if (ctx->stamps_used * 2 + 2 > ctx->stamp_events.size()) {
            hipEvent_t a = nullptr, b = nullptr;
            if (hipEventCreate(&a) != hipSuccess || hipEventCreate(&b) != hipSuccess) return;
            ctx->stamp_events.push_back(a);
            ctx->stamp_events.push_back(b);
            ctx->stamp_slot.push_back(slot);
        }
        start = ctx->stamp_events[2 * ctx->stamps_used];
        stop = ctx->stamp_events[2 * ctx->stamps_used + 1];
        ctx->stamp_slot[ctx->stamps_used] = slot;
        ctx->stamps_used++;
    }
};

struct dfl_timed {
    dflash_ctx *ctx;
    hipStream_t st;
    int slot;
    dfl_timed(dflash_ctx *c, hipStream_t s, int k) : ctx(c), st(s), slot(k) {
        if (ctx->timing) (void)hipEventRecord(ctx->ev0, st);
    }
    ~dfl_timed() {
        if (!ctx->timing) return;
        (void)hipEventRecord(ctx->ev1, st);
        (void)hipEventSynchronize(ctx->ev1);
        float ms = 0.0f;
        if (hipEventElapsedTime(&ms, ctx->ev0, ctx->ev1) == hipSuccess) {
            ctx->timed_ms[slot] += ms;
            ctx->timed_launches[slot] += 1;
        }
    }
};

// Records a message on the context and returns `status`.
int32_t dfl_fail(dflash_ctx *ctx, int32_t status, const char *fmt, ...);

#define DFL_HIP_CHECK(ctx, expr)                                                          \
    do {                                                                                  \
        hipError_t e_ = (expr);                                                           \
        if (e_ != hipSuccess)                                                             \
            return dfl_fail((ctx), DFLASH_ERR_HIP, "%s: %s", #expr, hipGetErrorString(e_)); \
    } while (0)

// Makes sure kernel `fn` may be launched with `bytes` of dynamic LDS on the context's device
// (hipFuncAttributeMaxDynamicSharedMemorySize), calling the runtime only the first time.
int32_t dfl_raise_lds_limit(dflash_ctx *ctx, const void *fn, size_t bytes);

// Carves `bytes` (256-aligned) out of the context workspace starting at *offset.
template <typename T>
static inline T *dfl_ws_take(dflash_ctx *ctx, size_t *offset, size_t bytes) {
    size_t start = (*offset + 255) & ~size_t(255);
    if (start + bytes > ctx->workspace_bytes) return nullptr;
    *offset = start + bytes;
    return reinterpret_cast<T *>(ctx->workspace + start);
}

static inline bool dfl_ranges_overlap(const void *a, size_t na, const void *b, size_t nb) {
    const char *pa = static_cast<const char *>(a), *pb = static_cast<const char *>(b);
    return pa < pb + nb && pb < pa + na;
}

enum { DFL_QK_K = 256, DFL_Q4_K_BYTES = 144, DFL_Q6_K_BYTES = 210, DFL_Q8_0_BYTES = 34, DFL_QK8_0 = 32 };

// ---- activations in MFMA fragment order ("XF") -----------------------------------------------------------------
// The hand-off format between a kernel that produces the 16 activation rows of a few-row GEMM and the whole-K GEMM
// kernels (gemm_whole.hip) that consume them: f16, already in the order the consumer's MFMA A operands are read in,
// so that a wave loads a stage's eight fragments with eight coalesced 16-byte loads and no trip through LDS.
// Per super-block b (256 values of K) 512 slots of 16 bytes: slot (t, lane) at byte ((b * 8 + t) * 64 + lane) * 16,
// lane = 16 g + m (m = row), holds row m's eight consecutive values k = 256 b + 8 o + {0,2,1,3,4,6,5,7}[i] (the order
// in which the nibble unpack emits a lane's weights), with octet o = 8 g + t for a Q4_K consumer and
// o = 16 (g >> 1) + 8 (t >> 2) + 4 (g & 1) + (t & 3) for a Q6_K consumer (its quarters interleave).  Rows a producer
// does not write keep whatever the buffer held: a row of the product depends on its own activation row only.
enum { DFL_XF_NONE = 0, DFL_XF_Q4K = 1, DFL_XF_Q6K = 2 };
static inline size_t dfl_xf_bytes(int64_t n_in) { return static_cast<size_t>(n_in / 256) * 8192; }
#ifdef __HIPCC__
// byte offset of the slot of row m's values k0 .. k0 + 7 (k0 a multiple of 8)
__host__ __device__ static inline uint32_t dfl_xf_slot(int kind, int m, int k0) {
    const int b = k0 >> 8, o = (k0 >> 3) & 31;
    int g, t;
    if (kind == DFL_XF_Q6K) {
        const int h = o >> 4, quarter = (o >> 2) & 3;
        g = 2 * h + (quarter & 1);
        t = 4 * (quarter >> 1) + (o & 3);
    } else {
        g = o >> 3;
        t = o & 7;
    }
    return static_cast<uint32_t>(((b * 8 + t) * 64 + 16 * g + m) * 16);
}
__device__ static inline void dfl_xf_store(void *xf, int kind, int m, int k0, float v0, float v1, float v2, float v3, float v4,
                                           float v5, float v6, float v7) {
    typedef _Float16 h8 __attribute__((ext_vector_type(8)));
    const h8 frag = {static_cast<_Float16>(v0), static_cast<_Float16>(v2), static_cast<_Float16>(v1), static_cast<_Float16>(v3),
                     static_cast<_Float16>(v4), static_cast<_Float16>(v6), static_cast<_Float16>(v5), static_cast<_Float16>(v7)};
    *reinterpret_cast<h8 *>(static_cast<uint8_t *>(xf) + dfl_xf_slot(kind, m, k0)) = frag;
}
// A kernel's arguments beyond the first fourteen words are loaded where they are first used, 0.3 us of a wave that waits for
// nothing else at that place.  This asks for them here, behind a kernel's first loads, under which they arrive.
template <typename T>
__device__ static __forceinline__ void dfl_have_one(T v) {
    asm volatile("" ::"s"(v));
}
template <typename... T>
__device__ static __forceinline__ void dfl_have(T... v) {
    (dfl_have_one(v), ...);
}
// Reductions over a wave without LDS (a shuffle is a trip through it, and six in a row stand in the middle of most small
// kernels): the lane 32 or 16 away by v_permlane32/16_swap, the nearer ones by DPP moves.  The tree is that of
// `for (off = 32; off; off >>= 1) v += __shfl_xor(v, off)`, lane for lane, so a sum has that loop's bits.
// (The swaps as asm: through the builtins the compiler used one of the two results twice.  Both want two wait states
// behind the write of their operands.)
template <int CTRL>
__device__ static inline float dfl_dpp(float v) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xF, 0xF, true));
}
__device__ static inline void dfl_swap16(float &a, float &b) { asm("s_nop 1\n\tv_permlane16_swap_b32 %0, %1" : "+v"(a), "+v"(b)); }
__device__ static inline void dfl_swap32(float &a, float &b) { asm("s_nop 1\n\tv_permlane32_swap_b32 %0, %1" : "+v"(a), "+v"(b)); }
__device__ static inline float dfl_xor4(float v) {  // the value of the lane 4 away: banks 0 and 2 of a row from above, 1 and 3 from below
    const int up = __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x104, 0xF, 0x5, false);
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(up, __builtin_bit_cast(int, v), 0x114, 0xF, 0xA, false));
}
__device__ static inline float dfl_wave_sum(float v) {
    float a = v, b = v;
    dfl_swap32(a, b);
    v = a + b;
    a = v, b = v;
    dfl_swap16(a, b);
    v = a + b;
    v += dfl_dpp<0x128>(v);  // row_ror:8
    v += dfl_xor4(v);
    v += dfl_dpp<0x4E>(v);   // quad_perm [2,3,0,1]
    v += dfl_dpp<0xB1>(v);   // quad_perm [1,0,3,2]
    return v;
}
__device__ static inline float dfl_max_far(float v) {  // maximum over the four lanes 16 apart, in each of them
    float a = v, b = v;
    dfl_swap32(a, b);
    v = fmaxf(a, b);
    a = v, b = v;
    dfl_swap16(a, b);
    return fmaxf(a, b);
}
__device__ static inline float dfl_wave_max(float v) {
    v = dfl_max_far(v);
    v = fmaxf(v, dfl_dpp<0x128>(v));
    v = fmaxf(v, dfl_xor4(v));
    v = fmaxf(v, dfl_dpp<0x4E>(v));
    return fmaxf(v, dfl_dpp<0xB1>(v));
}
// Lanes (2 p, 2 p + 1) of a wave hold values i .. i + 3 and i + 4 .. i + 7 of row m (i a multiple of 8 on the even lane):
// the even lane stores the octet.  Every lane of the wave must call it.
__device__ static inline void dfl_xf_store_pair(void *xf, int kind, int m, int i, float a, float b, float c, float d) {
    const float e = dfl_dpp<0x101>(a), f = dfl_dpp<0x101>(b), g = dfl_dpp<0x101>(c), h = dfl_dpp<0x101>(d);  // row_shl:1
    if ((threadIdx.x & 1) == 0) dfl_xf_store(xf, kind, m, i, a, b, c, d, e, f, g, h);
}
#endif

// Whole-K few-row GEMM over activations in XF order (gemm_whole.hip): y[n_rows][n_out] = x . w^T with every output tile's
// whole K inside one workgroup (its waves split K and add up in LDS in a fixed order): no partial tiles, no second launch.
// dfl_whole_kind: the XF kind a producer must write for this matrix (DFL_XF_NONE: the shape or type does not take
// this path: more than two stages per wave, or more tiles than one round of the chip).  pair_ffn > 0: w is a fused
// gate | up matrix of 2 * pair_ffn rows and the output is silu(gate) * up, [n_rows][pair_ffn]: as f32 in y (may be null)
// and / or as XF of kind y_xf_kind in y_xf (may be null), the activations of the down projection that follows.
int dfl_whole_kind(const dflash_ctx *ctx, int32_t w_type, int64_t n_in, int64_t n_out, int64_t pair_ffn);
int32_t dfl_gemm_whole(dflash_ctx *ctx, int32_t w_type, const void *w, const void *xf, float *y, int64_t n_in, int64_t n_out,
                       int32_t n_rows, int64_t pair_ffn, void *y_xf, int y_xf_kind, hipStream_t stream, bool by_sums = false);
// by_sums: where dfl_whole_by_sums says so, minima through the activations' sub-block sums, as dfl_gemm_rows has them (a target's
// layers); else through twin products (a drafter's, and the public operator).  It says so for a Q4_K matrix of 16 super-blocks of K
// or more whose tiles are one round of the chip (the looping kernel has twins alone).
bool dfl_whole_by_sums(const dflash_ctx *ctx, int32_t w_type, int64_t n_in, int64_t n_out, int64_t pair_ffn);
// The same for n_rows_total rows, sixteen to a block (the last one may be shorter): block i's rows are in XF order at
// xf + i * dfl_xf_bytes(n_in), its result at y + i * 16 * n_out (pair mode: 16 * pair_ffn; y_xf + i * dfl_xf_bytes(pair_ffn)).
// The weights are read once and stay in registers while the blocks pass; a row's bits are those of dfl_gemm_whole.  A looping
// plan takes one block; by sums, several only where dfl_whole_holds_weights says so (else DFLASH_ERR_UNSUPPORTED).
int32_t dfl_gemm_whole_blocks(dflash_ctx *ctx, int32_t w_type, const void *w, const void *xf, float *y, int64_t n_in, int64_t n_out,
                              int32_t n_rows_total, int64_t pair_ffn, void *y_xf, int y_xf_kind, hipStream_t stream, bool by_sums = false);
// Whether a wave has one super-block of one tile, whose unpacked weights it then keeps from block to block.
bool dfl_whole_holds_weights(const dflash_ctx *ctx, int32_t w_type, int64_t n_in, int64_t n_out);

// The whole-K kernel on rows in row order (f32 or f16), for the public operator: y[n_rows][n_out] = x . w^T in one launch, for Q4_K in either
// order and Q6_K in row order; the same bits for both orders.  (Null and misaligned weights and overlapping buffers are gemm_fewrow_impl's to refuse,
// which every caller comes through.)
bool dfl_gemm_direct_takes(const dflash_ctx *ctx, int32_t w_type, int64_t n_in, int64_t n_out);
int32_t dfl_gemm_direct(dflash_ctx *ctx, int32_t w_type, const void *w, const void *x, int32_t x_type, float *y, int64_t n_in, int64_t n_out,
                        int32_t n_rows, hipStream_t stream);

// silu(x . gate^T) * (x . up^T) of up to sixteen rows as f16, [n_rows][ffn], in one launch (gemm_dense.hip): the fused gate | up matrix of a
// dense layer in the tiled order, of more tiles than a whole-K launch takes.  xf, xs: the rows in fragment order (Q4K) and their
// sub-block sums.
bool dfl_gemm_dense_pair_takes(const dflash_ctx *ctx, int32_t w_type, int64_t n_in, int64_t ffn);
int32_t dfl_gemm_dense_pair(dflash_ctx *ctx, int32_t w_type, const void *w, const void *xf, const void *xs, void *y_f16, int64_t n_in, int64_t ffn,
                            int32_t n_rows, hipStream_t stream);

// ---- many rows at once (gemm_rows.hip): the products of a prompt's prefill ----
// Every row gets the bits the 16-row kernels give it in its own block: dfl_gemm_rows_plan says which of their
// arithmetics the matrix takes there and where K is cut.  kind == DFL_XF_NONE: not taken (only the tiled orders are).
// row_major: the block's rows reach this matrix in row order, so that its 16-row kernel is the streaming one whatever its
// shape (Q4_K; a tiled Q6_K matrix has no such kernel).
struct dfl_rows_plan {
    int kind;      // fragment order the activations must be in
    int whole;     // the 16-row kernel is the whole-K kernel (K is cut at its slices)
    int sums;      // the activations' sub-block sums are needed (else: twin products)
    int total, n_cut, by_group;
};
dfl_rows_plan dfl_gemm_rows_plan(const dflash_ctx *ctx, int32_t w_type, int64_t n_in, int64_t n_out, int64_t pair_ffn, bool row_major = false);
// Sub-block sums of n_blocks blocks of rows in fragment order (kind Q4K), for the plans with `sums`:
// dfl_xs_bytes(n_in) bytes per block.
static inline size_t dfl_xs_bytes(int64_t n_in) { return static_cast<size_t>(n_in / 256) * 1024; }
int32_t dfl_xf_sums(dflash_ctx *ctx, const void *xf, int64_t n_in, int32_t n_blocks, void *xs, hipStream_t stream);
// y[n_rows][n_out] = X . W^T, block b of sixteen rows at xf + b * dfl_xf_bytes(n_in) (sums: xs + b * dfl_xs_bytes(n_in)).
// pair_ffn > 0: W is a fused gate | up matrix and silu(gate) * up goes to y_xf in fragment order y_kind (and its sub-block
// sums to y_xs unless null) instead.  make_sums: xs is to be computed first, where the plan needs it.
int32_t dfl_gemm_rows(dflash_ctx *ctx, const dfl_rows_plan &plan, int32_t w_type, const void *w, const void *xf, void *xs, bool make_sums, float *y,
                      int64_t n_in, int64_t n_out, int32_t n_rows, int64_t pair_ffn, void *y_xf, void *y_xs, int y_kind, hipStream_t stream);
// What a product of n_rows rows costs by the measure that picks its tiles: rounds of the chip times what a tile takes, over its super-blocks.
double dfl_gemm_rows_cost(const dflash_ctx *ctx, const dfl_rows_plan &p, int64_t n_in, int64_t n_out, int32_t n_rows, int64_t pair_ffn);
// The experts' products over row tiles listed on the device, tiles[i] = {expert (-1: the extra matrix), first block,
// blocks (1..tile_blocks, which is 4 or 8), -}: the arithmetic of gemm_q4k_experts_kernel.  w_up != null: silu(x . w^T) * (x . w_up^T) to y_xf / y_xs.
int32_t dfl_gemm_rows_experts(dflash_ctx *ctx, const void *w, const void *w_extra, const void *w_up, const void *w_up_extra, size_t w_stride,
                              const void *xf, const void *xs, const int32_t *tiles, const int32_t *n_tiles, int32_t max_tiles,
                              int32_t tile_blocks, float *y, int64_t n_in, int64_t n_out, void *y_xf, void *y_xs, hipStream_t stream);
// How dfl_gemm_fewrow_checked splits a Q4_K matrix in tiled order: workgroup i of n_wg takes stages
// [total i / n_wg, total (i + 1) / n_wg) of the (256-row tile group x super-block) space; false where it does not take it.
bool dfl_q4k_tiled_split(const dflash_ctx *ctx, int64_t n_in, int64_t n_out, int *total, int *n_wg);

// dflash_dflash2_conv whose result also goes to y_xf in fragment order (XF; h a multiple of 256), for the whole-K
// projection that reads it.
int32_t dfl_dflash2_conv(dflash_ctx *ctx, const float *x, const float *dyn, const float *base, float *y, int32_t n_tokens, int32_t h,
                         int32_t kernel_size, int32_t group_size, int32_t side, dflash_stream_t stream, void *y_xf, int y_xf_kind);

// A DFlash-2 sublayer's coefficient projection (a tiled Q4_K matrix whose rows are in fragment order at xf) and its side-0
// convolution in one launch: the convolved rows to y_xf in fragment order (which must not overlap xf), side 1's coefficients to dyn, whose
// side 0 is left as it is.  The bits of dfl_gemm_whole followed by dfl_dflash2_conv.
bool dfl_gemm_conv_takes(const dflash_ctx *ctx, int32_t w_type, int64_t h, int32_t kernel_size, int32_t group_size, int32_t y_xf_kind);
int32_t dfl_gemm_conv(dflash_ctx *ctx, const void *w, const void *xf, const float *x, const float *base, int64_t h, int32_t group_size, int32_t n_rows,
                      float *dyn, void *y_xf, int y_xf_kind, hipStream_t stream);

// Device scratch of the mixture-of-experts FFN (owned by the target session).
struct dfl_moe_scratch {
    float *probs = nullptr;   // [16][n_expert] router logits
    int32_t *sel_e = nullptr; // [16][n_used]
    float *sel_w = nullptr;   // [16][n_used]
    float *sg = nullptr;      // [16] shared-expert gate
    float *act = nullptr;     // [16*n_used][ffn_expert]           (per-slot path)
    float *eo = nullptr;      // [slots][16][hidden]; per-slot path: [16*n_used][hidden]
    float *gate_out = nullptr;  // [slots][16][ffn_expert]: silu(gate) * up of every slot (batched path)
    int32_t *ids = nullptr, *n_distinct = nullptr, *slot_of = nullptr;  // distinct experts, their count, pick -> slot
    float *shared = nullptr;  // [16][hidden]
    float *g = nullptr, *u = nullptr;  // [16][ffn_shared]
};

// x_resid[n][hidden] += moe_ffn(cur[n][hidden]) for one layer; enqueue only.  gate_done: scratch.sg
// already holds sigmoid(cur . shexp_gate) per row (the norm kernel that wrote cur computed it).
// next_norm_w / next_cur / next_done (all or none): the RMSNorm that reads x_resid next may be done
// in the same pass, next_cur = rms_norm(x_resid) * next_norm_w; *next_done says whether it was.
// next_xf / next_xf_kind: where that norm is done here, its rows go to next_xf in fragment order (XF) instead.  cap / cap_ld: where it is
// done here, x_resid's new rows also go to cap, cap_ld floats apart (16-byte aligned, cap_ld a multiple of 4).
// pre_add / pre_norm_w (both or neither; only where dfl_moe_norm_fusable() holds): the layer's input has not been
// normalised yet, x_resid still lacks pre_add (the attention's output projection), and `cur` is where the normalised rows
// go: cur = rms_norm(x_resid + pre_add) * pre_norm_w, computed inside the router's launch with the shared-expert gate
// (gate_done is then implied); x_resid += pre_add happens where the experts' sum is added.
int32_t dfl_moe_ffn(dflash_ctx *ctx, const dflash_model_cfg &cfg, const dflash_layer &layer, float *cur, int n,
                    const dfl_moe_scratch &scratch, float *x_resid, bool gate_done, const float *next_norm_w,
                    float *next_cur, bool *next_done, hipStream_t stream, const float *pre_add = nullptr,
                    const float *pre_norm_w = nullptr, void *next_xf = nullptr, int next_xf_kind = 0, float *cap = nullptr, int cap_ld = 0);
bool dfl_moe_norm_fusable(const dflash_ctx *ctx, const dflash_model_cfg &cfg, const dflash_layer &layer, int n);

// The same FFN for the rows of several consecutive 16-row blocks at once (a prompt's prefill): the rows are regrouped
// by expert, so a pass reads every touched expert about once however many blocks there are.  cur holds the layer's
// normalised input and scratch.sg the rows' shared-expert gates (the norm kernel's work); x_resid += experts(cur),
// then cur = rms_norm(x_resid) * next_norm_w, also to next_xf (block b of sixteen rows at
// next_xf + b * next_xf_stride bytes) where next_xf_kind says so.  Every row gets the bits dfl_moe_ffn gives it inside
// its own block.  Takes layers with tiled Q4_K expert stacks and a shared expert of the experts' shape
// (dfl_moe_group_fits); scratch of dfl_moe_group_max_slots(cfg, n_rows) slots.  Enqueue only.
struct dfl_moe_group_scratch {
    float *logits = nullptr;      // [rows][n_expert]
    float *sg = nullptr;          // [rows]
    int32_t *sel_e = nullptr;     // [rows][n_used]
    float *sel_w = nullptr;       // [rows][n_used]
    int32_t *pick_pos = nullptr;  // [rows][n_used]: row of eo that holds the pick's output
    int32_t *n_slots = nullptr;
    int32_t *slot_rows = nullptr; // [max_slots][16]
    int32_t *tiles = nullptr;     // [max_slots][4]: row tiles of dfl_gemm_rows_experts
    int32_t *n_tiles = nullptr;
    uint8_t *xg = nullptr, *xg_sums = nullptr;    // every slot's rows in fragment order, and their sub-block sums
    uint8_t *act = nullptr, *act_sums = nullptr;  // the same of silu(gate) * up
    float *eo = nullptr;          // [max_slots][16][hidden]
    int max_slots = 0;
};
int dfl_moe_group_max_slots(const dflash_model_cfg &cfg, int n_rows);
int dfl_moe_group_max_picks();  // rows * picks per row that one pass takes
bool dfl_moe_group_fits(const dflash_ctx *ctx, const dflash_model_cfg &cfg, const dflash_layer &layer, int n_rows);
int32_t dfl_moe_ffn_group(dflash_ctx *ctx, const dflash_model_cfg &cfg, const dflash_layer &layer, float *x_resid,
                          float *cur, int n_rows, const dfl_moe_group_scratch &scratch, const float *next_norm_w, void *next_xf,
                          int next_xf_kind, size_t next_xf_stride, hipStream_t stream, float *cap = nullptr, int cap_ld = 0);

// Residual add + RMSNorm + shared-expert gate + Q8_0 router product of a mixture-of-experts layer as one launch:
// cur[n_rows][hidden] = rms_norm(x + add) * norm_w, gate_out[r] = sigmoid(cur[r] . gate_w),
// logits[n_rows][n_expert] = cur . router_w^T, bit-identical to the norm kernel followed by the few-row GEMM.
// x is left as it is.  dfl_router_norm_fits: whether the shape is one the kernel takes (hidden a multiple of 256, at
// most 2048; every row is a workgroup column of its own, 1..4096 of them); switched off by DFLASH_MOE_FUSED_NORM=0.  Enqueue only.
bool dfl_router_norm_fits(const dflash_ctx *ctx, int32_t router_type, const void *router_w, int64_t hidden, int32_t n_expert,
                          int32_t n_rows);
// The router product alone for any number of rows, sixteen to a workgroup row: logits[n_rows][n_expert] = cur . router_w^T
// with the bits dfl_router_norm (and the few-row GEMM of a Q8_0 router) gives each row.  Same shapes as dfl_router_norm_fits.
int32_t dfl_router_rows(dflash_ctx *ctx, const void *router_w, const float *cur, float *logits, int64_t hidden, int32_t n_expert,
                        int32_t n_rows, hipStream_t stream);
int32_t dfl_router_norm(dflash_ctx *ctx, const void *router_w, const float *x, const float *add, const float *norm_w,
                        const float *gate_w, float eps, float *cur, float *gate_out, float *logits, int64_t hidden,
                        int32_t n_expert, int32_t n_rows, hipStream_t stream);

// dflash_attn_verify_block with the drafter's masks: full_block != 0 lets every row see the whole
// block (non-causal), window > 0 keeps only keys with |distance| < window.  ctx_len_dev != null:
// the context length is read from that device word when the kernels run, so that the call can sit
// in a captured graph that is replayed at other positions.  How the keys are cut into chunks and
// the heads into workgroups depends on dfl_attn_bucket(ctx_len + n_rows) only, and with ctx_len_dev
// the launches are sized for the largest context of that bucket: a captured call stays valid, and
// bit-identical to a direct one, at every context of the bucket it was captured in (a graph key
// must therefore include the bucket).  out_xf / out_xf_kind: the rows [n_rows][n_q * head_dim] also go to out_xf in
// fragment order (XF), for the output projection that reads them.
// Lower bound of the power-of-two range [b, 2 b) that holds n_pos visible positions (at least 256).
inline int64_t dfl_attn_bucket(int64_t n_pos) {
    int64_t b = 256;
    while (2 * b <= n_pos) b *= 2;
    return b;
}
// dflash_argmax_top2 whose results also go to page (a host page the device can write, as the context's pinned one; may be null): [16] indices,
// [16] of also (null: left alone), [16] gaps.
int32_t dfl_argmax_top2(dflash_ctx *ctx, const float *logits, int32_t n_rows, int64_t vocab, int64_t stride, int32_t *idx, float *gap,
                        int32_t *page, const int32_t *also, hipStream_t stream);
// dflash_select_draft_path whose tokens also go to page (as above; may be null).
int32_t dfl_select_draft_path(dflash_ctx *ctx, const dflash_codebook *predecessor, const dflash_codebook *successor, int32_t rank, int32_t top_k,
                              int32_t carry_token, int32_t n, const int32_t *topk_ids, const float *topk_vals, const float *sel_h, int32_t *out_tokens,
                              int32_t *out_tokens_host, int32_t *page, dflash_stream_t stream);

// A block's rows as the projections leave them, [row][query heads | key heads | value heads] in f32: the attention norms and rotates them itself,
// and writes the block's rows of both caches (dfl_attn_block with rope; its q is then those rows).
struct dfl_attn_rope {
    const float *q_w, *k_w;  // the norms' weights
    const float *table;      // [row][head_dim / 2 cosines, head_dim / 2 sines] of the rows' positions
    float eps;
};
bool dfl_attn_rope_takes(const dflash_ctx *ctx, const dfl_attn_rope &r, const void *rows, int32_t n_q, int32_t n_kv, int64_t ctx_len, int32_t n_rows,
                         int32_t head_dim, int64_t kv_capacity);
int32_t dfl_attn_block(dflash_ctx *ctx, const void *q, int32_t q_type, const void *k_cache, const void *v_cache,
                       int32_t v_layout, int64_t ctx_len, int32_t n_rows, int32_t n_q, int32_t n_kv, int32_t head_dim,
                       int64_t kv_capacity, float scale, float *out, dflash_stream_t stream, int32_t full_block,
                       int64_t window, const int32_t *ctx_len_dev, void *out_xf = nullptr, int out_xf_kind = 0, const struct dfl_attn_rope *rope = nullptr);

// Block-causal attention of n_rows_total consecutive query rows, sixteen to a block, each block exactly as
// dfl_attn_block would run it alone at its own context length (ctx_len + 16 b): the same split of the keys, so the same
// bits.  The leading blocks whose splits are merged in order go out as one launch that needs no workspace where they are
// enough workgroups for it; else blocks whose context lengths fall in the same bucket go out as one launch pair (as many
// of them as the workspace holds partial tiles for).  Transposed V cache; block b's rows at q + 16 b rows, out likewise,
// out_xf + b * dfl_xf_bytes(n_q * head_dim).  The K/V rows of all the blocks are in the cache already.
int32_t dfl_attn_blocks(dflash_ctx *ctx, const void *q, int32_t q_type, const void *k_cache, const void *vt_cache, int64_t ctx_len,
                        int32_t n_rows_total, int32_t n_q, int32_t n_kv, int32_t head_dim, int64_t kv_capacity, float scale,
                        float *out, dflash_stream_t stream, void *out_xf, int out_xf_kind);

// dflash_gemm_fewrow for a tensor of a model that passed dfl_model_tensors_checked (the fast kernels).
int32_t dfl_gemm_fewrow_checked(dflash_ctx *ctx, int32_t w_type, const void *w, const void *x, int32_t x_type, float *y,
                                int64_t n_in, int64_t n_out, int32_t n_rows, dflash_stream_t stream);
// The same by the public operator's routes: small matrices in one launch, whose cuts of K a prompt's products do not share.
int32_t dfl_gemm_fewrow_one(dflash_ctx *ctx, int32_t w_type, const void *w, const void *x, int32_t x_type, float *y, int64_t n_in,
                            int64_t n_out, int32_t n_rows, dflash_stream_t stream);

// Few-row Q6_K GEMMs of up to three matrices over the same activations (a layer's q, k and v
// projections) as one launch: y[m] = x . w[m]^T, [n_rows][n_out[m]] each.
int32_t dfl_gemm_q6k_set(dflash_ctx *ctx, int n_mats, const void *const *w, float *const *y, const int64_t *n_out, const void *x,
                         int32_t x_type, int64_t n_in, int32_t n_rows, dflash_stream_t stream);

// Few-row Q4_K GEMM over the matrices that the device-side list ids[0 .. *n_slots) picks out of a stack
// (w_stack + id * w_stride_bytes; id -1 = extra_w): slot j reads activations x + j * x_stride (elements; 0 = shared) and
// writes y + j * y_stride (floats) as [n_rows][n_out].  max_slots bounds *n_slots.  whole_groups != 0:
// no split K (results independent of the other matrices in the batch).  w_stack_up != null (needs
// whole_groups): SwiGLU pair, y = silu(x . gate^T) * (x . up^T) with the gate matrices from w_stack /
// extra_w and the up matrices, same ids, from w_stack_up / extra_w_up.  tiled != 0: every matrix (the stacks'
// members, the extras) is in the tiled order of dflash_repack_q4k_tiled and w_stride_bytes is the tiled size.
// y_type: DFLASH_TYPE_F32, or DFLASH_TYPE_F16 (y then points to f16 and y_stride counts f16 elements) where
// dfl_q4k_batched_f16_out() says the path that will run can write it.  Enqueue only.
bool dfl_q4k_batched_f16_out(const dflash_ctx *ctx, int32_t tiled, int32_t whole_groups, int64_t n_out);
// Routing folded into the launch (route != null; where dfl_q4k_batched_can_route() allows it): ids and n_slots are
// then OUTPUTS.  Every workgroup derives the block's expert list from the router logits itself (the arithmetic of
// the stand-alone routing kernel, n_expert <= 256), workgroup 0 writes ids, *n_slots, sel_e, sel_w and slot_of for
// the launches that follow; the shared-expert gate is not computed here.
struct dfl_route_args {
    const float *logits;  // [n_rows][n_expert]
    int32_t n_expert, n_used, with_shared;
    int32_t *sel_e;   // [n_rows][n_used]
    float *sel_w;     // [n_rows][n_used]
    int32_t *slot_of; // [n_rows][n_used]
};
bool dfl_q4k_batched_can_route(const dflash_ctx *ctx, int32_t tiled, int64_t n_out, int32_t n_expert, int32_t n_used);
int32_t dfl_gemm_q4k_batched(dflash_ctx *ctx, const void *w_stack, size_t w_stride_bytes, const void *extra_w,
                             const int32_t *ids, const int32_t *n_slots, int max_slots, const void *x, int32_t x_type,
                             size_t x_stride,
                             void *y, int32_t y_type, size_t y_stride, int64_t n_in, int64_t n_out, int32_t n_rows,
                             int32_t whole_groups, const void *w_stack_up, const void *extra_w_up, int32_t tiled,
                             dflash_stream_t stream, const dfl_route_args *route = nullptr);
