// Many-row quantised GEMM of a prompt's prefill: Y[rows][n_out] = X[rows][n_in] . W^T for the rows of many 16-row
// blocks at once, X handed over in MFMA fragment order (common.h, "XF"), W in the library's tiled orders.
// Same contraction as encode_mat_mat_dispatch_dflash_verify (metal_forward/dispatch.rs:365-378).
//
// What bounds it.  With sixteen rows a weight is unpacked for one MFMA and the kernel streams weights; here a weight
// unpacked once serves up to 128 rows, and the matrix cores are what there is most of to do.  A workgroup of eight waves
// computes 16 RB rows x 256 columns (a SwiGLU pair: 128 gate and the 128 up columns that go with them); a wave, 16 RB rows
// x 32 columns:
//   * per super-block of K the activations of its row blocks (8 KB each) and the raw quant blocks of its 16-row weight
//     tiles are copied into LDS with direct-to-LDS loads, both as they lie in memory (contiguous pieces), the weights a
//     super-block ahead, the activations half a super-block;
//   * no two waves unpack the same weights (with the waves two by four, which halves the LDS reads, the unpacking on the
//     vector ALU took as long as the products); an activation fragment read from LDS feeds two products;
//   * the weights stay quantised up to the registers: a matrix is read from memory once and from L2 once per row tile, at
//     4.5 or 6.6 bits a weight instead of 16.
// Workgroups that share weights are dispatched to one XCD (rows_linear), so that a matrix passes through one L2.
// Measured for 2032 rows (four blocks per pass through the 16-row kernels before): 5120 -> 2 x 17408 with SwiGLU 795 us
// (0.92 PFLOP/s; 30 us per block before), 17408 -> 5120 428 us (0.85), 5120 -> 6144 226 us and 4096 -> 5120 175 us (0.57
// and 0.49: their twin MFMAs, which the block path's bits ask for, are as many again); a 64-layer prompt of 1000 rows
// 72.6 ms against 292 (65 with the attention's splits merged in registers).
// The experts' tiles (a list, mostly one to four row blocks) take workgroups of half the columns, two of them on a CU:
// each waits for its own weights while the other computes (2 - 4 % of a prompt of 33 - 130 rows).
//
// Bits.  Every row of Y has the bits that the 16-row kernels give it in its own block.  The arithmetic of a
// super-block is theirs (the same unpacking, the same v_mfma_f32_16x16x32_f16 sequence into the same accumulator); K is
// walked in order, and where those kernels cut K - the whole-K kernel's slices (gemm_whole.hip), the stream-K ranges
// (gemm_fewrow.hip) - the accumulator is added to a running total and starts again from zero, in the order their
// partial tiles are added in.  That order is also what a split of K over workgroups has to keep: each range between two
// cuts goes to memory on its own and rows_reduce_kernel adds them up (kSplit; few rows against a narrow matrix).
#include "common.h"
#include "mfma_unpack.h"

#include <algorithm>
#include <type_traits>

namespace {

typedef const __attribute__((address_space(1))) void *gptr_t;
typedef __attribute__((address_space(3))) void *lptr_t;

constexpr int kRowsWaves = 8, kListWaves = 4;

struct RowsArgs {
    const uint8_t *w[2];       // matrix of column segment 0 and 1 (a list: the stacks' first matrices)
    const uint8_t *w_extra[2]; // list entries with expert -1
    size_t w_stride;           // bytes between the matrices of a stack
    int tile0_up;              // SwiGLU pair: first 16-row tile of the up half in w[1]
    int nb;                    // super-blocks of K
    int n_ct, n_rt;            // column tiles, row tiles (no list)
    int n_blocks;              // 16-row blocks of X (no list)
    int n_rows;                // rows of X (no list)
    const uint8_t *xf;         // block b at xf + b * nb * 8192
    const uint8_t *xs;         // its sub-block sums at xs + b * nb * 1024 (kinds that need them)
    const int4 *tiles;         // list: {expert, first block, blocks, -}
    const int32_t *n_tiles;    // list: how many
    int total, n_cut;          // where K is cut: see Cut
    int cut_by_group;          // the cuts differ from tile group to tile group
    int n_split;               // workgroups that share a tile's K (kSplit)
    float *y;                  // plain epilogue; kSplit: partial tiles [range of K][16 n_blocks][n_out]
    int n_out;                 // columns of y (= its row stride)
    uint8_t *y_xf, *y_xs;      // SwiGLU epilogue: fragment order and (may be null) sub-block sums, blocks nb_out super-blocks wide
    int y_kind, nb_out;
};

// The cut positions of one tile group: range i of the split takes stages [total i / n, total (i + 1) / n) of the
// flattened (group, super-block) space; `next` is the first super-block of the group behind the current range.
struct Cut {
    int wg, first, next, base;
    __device__ __forceinline__ int end(const RowsArgs &a) const {
        return static_cast<int>(static_cast<uint32_t>(a.total) * (wg + 1) / static_cast<uint32_t>(a.n_cut)) - base;
    }
    __device__ __forceinline__ static int range_of(int at, const RowsArgs &a) {
        return static_cast<int>((static_cast<uint32_t>(at + 1) * a.n_cut + a.total - 1) / static_cast<uint32_t>(a.total)) - 1;
    }
    __device__ __forceinline__ void start(int group, const RowsArgs &a) {
        base = group * a.nb;
        first = wg = range_of(base, a);
        next = end(a);
    }
    __device__ __forceinline__ int ranges(const RowsArgs &a) const { return range_of(base + a.nb - 1, a) - first + 1; }
    __device__ __forceinline__ bool at(int b, const RowsArgs &a) {  // K is cut in front of super-block b
        if (b != next) return false;
        wg++;
        next = end(a);
        return true;
    }
};

__device__ __forceinline__ half8_t splat8(_Float16 v) {
    const half8_t r = {v, v, v, v, v, v, v, v};
    return r;
}

// One tile's raw weights of one super-block in a lane's registers; operand<H>(t) is that of MFMA 4 H + t.
struct TileQ4 {
    static constexpr int kBytes = 16 * DFL_Q4_K_BYTES;
    u32x4_t q0, q1;
    half2_t S, Cs, m;
    __device__ __forceinline__ void load(const uint8_t *tile, int n, int g, uint32_t sc_sel, bool negate_min) {
        const u32x4_t *blk = reinterpret_cast<const u32x4_t *>(tile) + n * 9;
        const u32x4_t hdr = blk[0];
        q0 = blk[1 + 2 * g];
        q1 = blk[2 + 2 * g];
        const uint32_t upper = 0u - static_cast<uint32_t>(g >> 1);
        const uint32_t sc_lo = hdr.y & 0x3F3F3F3Fu, sc_hi = (hdr.w & 0x0F0F0F0Fu) | ((hdr.y >> 2) & 0x30303030u);
        const uint32_t mn_lo = hdr.z & 0x3F3F3F3Fu, mn_hi = ((hdr.w >> 4) & 0x0F0F0F0Fu) | ((hdr.z >> 2) & 0x30303030u);
        const uint32_t sc_word = (sc_hi & upper) | (sc_lo & ~upper), mn_word = (mn_hi & upper) | (mn_lo & ~upper);
        const half2_t dm = as_half2(hdr.x);
        const half2_t p_sc = as_half2(__builtin_amdgcn_perm(0x64646464u, sc_word, sc_sel));
        const half2_t p_mn = as_half2(__builtin_amdgcn_perm(0x64646464u, mn_word, sc_sel));
        const half2_t neg = dm * splat(static_cast<_Float16>(-1024.0f));
        S = __builtin_elementwise_fma(p_sc, splat(dm[0]), splat(neg[0]));
        m = negate_min ? __builtin_elementwise_fma(p_mn, splat(-dm[1]), splat(-neg[1])) : __builtin_elementwise_fma(p_mn, splat(dm[1]), splat(neg[1]));
        const half2_t unbias = {static_cast<_Float16>(-1024.0f), static_cast<_Float16>(-64.0f)};
        Cs = S * unbias;
    }
    template <int H>
    __device__ __forceinline__ half8_t operand(int t, Q4KMagic magic) const {  // t = 0..3
        const uint32_t qw[8] = {q0.x, q0.y, q0.z, q0.w, q1.x, q1.y, q1.z, q1.w};
        return unpack_scale<H == 1>(qw[2 * t], qw[2 * t + 1], splat(S[H]), splat(Cs[H]), H ? magic.hi : magic.lo);
    }
    template <int H>
    __device__ __forceinline__ half8_t twin(int) const {
        return splat8(m[H]);
    }
};

struct TileQ6 {
    static constexpr int kBytes = kQ6TileBytes;
    u32x4_t qa, qb, ha, hb;
    _Float16 s[4];
    int odd2;
    __device__ __forceinline__ void load(const uint8_t *tile, int n, int g, uint32_t, bool) {
        const int h = g >> 1, odd = g & 1;
        qa = *reinterpret_cast<const u32x4_t *>(tile + q6t_ql_piece(n, 4 * h + 2 * odd));
        qb = *reinterpret_cast<const u32x4_t *>(tile + q6t_ql_piece(n, 4 * h + 2 * odd + 1));
        ha = *reinterpret_cast<const u32x4_t *>(tile + q6t_qh_piece(n, 2 * h));
        hb = *reinterpret_cast<const u32x4_t *>(tile + q6t_qh_piece(n, 2 * h + 1));
        const uint2 sc = *reinterpret_cast<const uint2 *>(tile + kQ6TSc + n * 16 + 8 * h);
        const float d = __half2float(__ushort_as_half(*reinterpret_cast<const uint16_t *>(tile + kQ6TD + n * 2)));
#pragma unroll
        for (int j = 0; j < 2; j++) {
            s[j] = static_cast<_Float16>(d * static_cast<float>(static_cast<int8_t>(sc.x >> (16 * odd + 8 * j))));
            s[2 + j] = static_cast<_Float16>(d * static_cast<float>(static_cast<int8_t>(sc.y >> (16 * odd + 8 * j))));
        }
        odd2 = 2 * odd;
    }
    template <int H>
    __device__ __forceinline__ half8_t operand(int t, Q4KMagic magic) const {
        const uint32_t ql[8] = {qa.x, qa.y, qa.z, qa.w, qb.x, qb.y, qb.z, qb.w};
        const uint32_t hq[8] = {ha.x, ha.y, ha.z, ha.w, hb.x, hb.y, hb.z, hb.w};
        const _Float16 sv = s[2 * H + (t >> 1)];
        const int hs = odd2 + 4 * H;
        return unpack6<H == 1>(ql[2 * t], ql[2 * t + 1], hq[2 * t] >> hs, hq[2 * t + 1] >> hs, splat(sv),
                               splat(sv * static_cast<_Float16>(H ? -64.0f : -1024.0f)), H ? magic.hi : magic.lo);
    }
    template <int H>
    __device__ __forceinline__ half8_t twin(int t) const {
        return splat8(s[2 * H + (t >> 1)] * static_cast<_Float16>(32.0f));
    }
};

// Dispatch index -> linear tile index: the hardware deals consecutive workgroups to the eight XCDs in turn, so dispatch
// indices i, i + 8, i + 16, ... share an L2; they get consecutive tiles.  Returns -1 past the end.
__device__ __forceinline__ int rows_linear(int dispatch, int count) {
    const int per = (count + 7) >> 3, at = dispatch >> 3, l = (dispatch & 7) * per + at;
    return at < per && l < count ? l : -1;
}

enum { kEpiY = 0, kEpiSwiglu = 1, kEpiSplit = 2 };

// kTwin: the minima / offsets through a twin MFMA per activation fragment into a second accumulator (the whole-K
// kernel's arithmetic); else one MFMA per super-block over the sub-block sums (the streaming and expert kernels').
// kCut: K is cut somewhere.  RB: 16-row blocks of the tile.
template <typename Tile, bool kTwin, bool kCut, int RB, int kEpi, bool kList>
__global__ void __launch_bounds__(64 * (kList ? kListWaves : kRowsWaves)) gemm_rows_kernel(RowsArgs a) {
    constexpr int W = kList ? kListWaves : kRowsWaves;  // waves, 32 columns each
    constexpr bool kPair = kEpi == kEpiSwiglu, kSplit = kEpi == kEpiSplit, kTotal = kCut && !kSplit;
    constexpr int NSEG = kPair ? 2 : 1, kSegTiles = 2 * W / NSEG;
    constexpr int kABytes = RB * 4096, kWSeg = kSegTiles * Tile::kBytes, kWBytes = NSEG * kWSeg, kSBytes = kTwin ? 0 : RB * 1024;
    static_assert(2 * (kABytes + kWBytes + kSBytes) <= 160 * 1024, "one workgroup per CU, all of its LDS");
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    uint8_t *const lds_w = lds + 2 * kABytes, *const lds_s = lds_w + 2 * kWBytes;
    const int tid = threadIdx.x, lane = tid & 63, n = lane & 15, g = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);

    int ct, block0, blocks_left, part = 0;  // column tile, first row block, how many row blocks there are from it on, share of K
    const uint8_t *wbase[NSEG];
    if constexpr (kList) {
        const int l = rows_linear(blockIdx.x, *a.n_tiles * a.n_ct);
        if (l < 0) return;
        const int4 t = a.tiles[l / a.n_ct];
        ct = l % a.n_ct;
        block0 = __builtin_amdgcn_readfirstlane(t.y);
        blocks_left = __builtin_amdgcn_readfirstlane(t.z);
        const int expert = __builtin_amdgcn_readfirstlane(t.x);
#pragma unroll
        for (int s = 0; s < NSEG; s++) wbase[s] = expert < 0 ? a.w_extra[s] : a.w[s] + static_cast<size_t>(expert) * a.w_stride;
    } else {
        int l = rows_linear(blockIdx.x, a.n_ct * a.n_rt * (kSplit ? a.n_split : 1));
        if (l < 0) return;
        if constexpr (kSplit) {
            const int u = l / a.n_split;
            part = l - u * a.n_split;
            l = u;
        }
        ct = l / a.n_rt;
        block0 = (l - ct * a.n_rt) * RB;
        blocks_left = a.n_blocks - block0;
#pragma unroll
        for (int s = 0; s < NSEG; s++) wbase[s] = a.w[s];
    }
    int tile0[NSEG], b_begin = 0, b_end = a.nb;
    Cut cut[NSEG];
#pragma unroll
    for (int s = 0; s < NSEG; s++) {
        tile0[s] = ct * kSegTiles + (s ? a.tile0_up : 0);
        // stage b of segment s: kWSeg contiguous bytes at wbase[s] + b * 16 tiles
        wbase[s] += (static_cast<size_t>(tile0[s] >> 4) * a.nb * 16 + (tile0[s] & 15)) * Tile::kBytes;
        if constexpr (kCut) cut[s].start(a.cut_by_group ? tile0[s] >> 4 : 0, a);
    }
    if constexpr (kSplit) {  // this workgroup's ranges of K
        const int ranges = cut[0].ranges(a), r0 = ranges * part / a.n_split, r1 = ranges * (part + 1) / a.n_split;
        if (r0 >= r1) return;
        cut[0].wg = cut[0].first + r1 - 1;
        b_end = min(cut[0].end(a), a.nb);
        cut[0].wg = cut[0].first + r0 - 1;
        b_begin = r0 ? cut[0].end(a) : 0;
        cut[0].wg++;
        cut[0].next = cut[0].end(a);
    }
    const uint8_t *xf0 = a.xf + static_cast<size_t>(block0) * a.nb * 8192;
    const uint8_t *xs0 = kTwin ? nullptr : a.xs + static_cast<size_t>(block0) * a.nb * 1024;
    const size_t xf_stride = static_cast<size_t>(a.nb) * 8192, xs_stride = static_cast<size_t>(a.nb) * 1024;

    // ---- copies into LDS; a wave-load is 64 lanes x 16 bytes, consecutive in memory and in LDS ----
    auto copy = [&](const uint8_t *src, uint8_t *dst) {
        __builtin_amdgcn_global_load_lds((gptr_t)(src + lane * 16), (lptr_t)(dst), 16, 0, 0);
    };
    auto issue_x = [&](int b, int h) {  // half h of super-block b: 4 KB per row block (blocks past the end repeat the last one)
        uint8_t *dst = lds + h * kABytes;
#pragma unroll
        for (int j = 0; j < (RB * 4 + W - 1) / W; j++) {
            const int p = wave + W * j, blk = min(p >> 2, blocks_left - 1);
            if (RB * 4 % W == 0 || p < RB * 4)
                copy(xf0 + blk * xf_stride + static_cast<size_t>(b) * 8192 + h * 4096 + (p & 3) * 1024, dst + p * 1024);
        }
    };
    constexpr int kFull = kWSeg / 1024, kRest = (kWSeg % 1024) / 16;  // whole wave-loads of a segment, lanes of its last one
    auto issue_w = [&](int b) {
        uint8_t *dst = lds_w + (b & 1) * kWBytes;
#pragma unroll
        for (int s = 0; s < NSEG; s++) {
            const uint8_t *src = wbase[s] + static_cast<size_t>(b) * 16 * Tile::kBytes;
#pragma unroll
            for (int j = 0; j < (kFull + W - 1) / W; j++) {
                const int p = ((wave + W / 2 * s) & (W - 1)) + W * j;
                if (p < kFull) copy(src + p * 1024, dst + s * kWSeg + p * 1024);
            }
            if (kRest > 0 && wave == W - 1 - s && lane < kRest) copy(src + kFull * 1024, dst + s * kWSeg + kFull * 1024);
        }
        if constexpr (!kTwin) {
            static_assert(RB <= W, "a wave copies one block's sums");
            if (wave < RB) {
                const int blk = min(wave, blocks_left - 1);
                copy(xs0 + blk * xs_stride + static_cast<size_t>(b) * 1024, lds_s + (b & 1) * kSBytes + wave * 1024);
            }
        }
    };
    // how many copies issue_w makes in this wave: what may still be in flight when the activations issued before it are needed
    int w_copies = 0;
#pragma unroll
    for (int s = 0; s < NSEG; s++) {
        const int v = (wave + W / 2 * s) & (W - 1);
        w_copies += (kFull - v + W - 1) / W + (kRest > 0 && wave == W - 1 - s ? 1 : 0);
    }
    if (!kTwin && wave < RB) w_copies++;
    auto landed = [&](bool weights_in_flight) {  // this wave's copies are in LDS, then everybody's
        if (!weights_in_flight) {
            __builtin_amdgcn_s_waitcnt(0x0070);  // vmcnt(0), and its LDS reads (lgkmcnt(0)) before others overwrite what they read
        } else {
            switch (w_copies) {  // vmcnt(w_copies), lgkmcnt(0)
                case 4: __builtin_amdgcn_s_waitcnt(0x0074); break;
                case 5: __builtin_amdgcn_s_waitcnt(0x0075); break;
                case 6: __builtin_amdgcn_s_waitcnt(0x0076); break;
                case 7: __builtin_amdgcn_s_waitcnt(0x0077); break;
                default: __builtin_amdgcn_s_waitcnt(0x0070); break;
            }
        }
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };

    const uint32_t sc_sel = (lane & 16) ? 0x04030402u : 0x04010400u;
    const Q4KMagic magic = q4k_magic();
    const float4_t zero4 = {0, 0, 0, 0};
    float4_t acc[RB][2], sub[kTwin ? RB : 1][2], sum[kTotal ? RB : 1][2];
#pragma unroll
    for (int r = 0; r < RB; r++)
#pragma unroll
        for (int j = 0; j < 2; j++) {
            acc[r][j] = zero4;
            if (kTwin) sub[kTwin ? r : 0][j] = zero4;
        }
    bool first[NSEG];
#pragma unroll
    for (int s = 0; s < NSEG; s++) first[s] = true;

    // A tile with fewer than RB row blocks (an expert's few rows, a prompt's tail) computes those alone, behind uniform
    // branches that the full tile's code does not have.
    const int live = min(blocks_left, RB);
    Tile tile[2];
    auto compute = [&](auto half, auto partial, int b) {
        constexpr int H = decltype(half)::value;
        constexpr bool kPart = decltype(partial)::value != 0;
        if constexpr (H == 0) {
            const uint8_t *wt = lds_w + (b & 1) * kWBytes;
#pragma unroll
            for (int j = 0; j < 2; j++) tile[j].load(wt + (kPair ? j * kWSeg + wave * Tile::kBytes : (2 * wave + j) * Tile::kBytes), n, g, sc_sel, !kTwin);
            if constexpr (!kTwin) {
                const half8_t *sm = reinterpret_cast<const half8_t *>(lds_s + (b & 1) * kSBytes) + lane;
                const half8_t m0 = q4k_min_operand(tile[0].m), m1 = q4k_min_operand(tile[1].m);
#pragma unroll
                for (int r = 0; r < RB; r++) {
                    if (kPart && r >= live) break;
                    const half8_t am = sm[r * 64];
                    acc[r][0] = __builtin_amdgcn_mfma_f32_16x16x32_f16(am, m0, acc[r][0], 0, 0, 0);
                    acc[r][1] = __builtin_amdgcn_mfma_f32_16x16x32_f16(am, m1, acc[r][1], 0, 0, 0);
                }
            }
        }
        const half8_t *xa = reinterpret_cast<const half8_t *>(lds + H * kABytes) + lane;
#pragma unroll
        for (int t = 0; t < 4; t++) {
            const half8_t b0 = tile[0].template operand<H>(t, magic), b1 = tile[1].template operand<H>(t, magic);
#pragma unroll
            for (int r = 0; r < RB; r++) {
                if (kPart && r >= live) break;
                const half8_t af = xa[r * 256 + t * 64];
                acc[r][0] = __builtin_amdgcn_mfma_f32_16x16x32_f16(af, b0, acc[r][0], 0, 0, 0);
                acc[r][1] = __builtin_amdgcn_mfma_f32_16x16x32_f16(af, b1, acc[r][1], 0, 0, 0);
                if constexpr (kTwin) {
                    constexpr int z = kTwin ? 1 : 0;
                    sub[z * r][0] = __builtin_amdgcn_mfma_f32_16x16x32_f16(af, tile[0].template twin<H>(t), sub[z * r][0], 0, 0, 0);
                    sub[z * r][1] = __builtin_amdgcn_mfma_f32_16x16x32_f16(af, tile[1].template twin<H>(t), sub[z * r][1], 0, 0, 0);
                }
            }
        }
    };
    auto range_result = [&](int r, int j) -> float4_t {
        if constexpr (kTwin) return acc[r][j] - sub[kTwin ? r : 0][j];
        return acc[r][j];
    };
    auto store_y = [&](float *y, int r, int j, float4_t v) {
        if (r >= live) return;
        const int64_t row0 = static_cast<int64_t>(block0 + r) * 16 + 4 * g;
        const int col = (tile0[0] + 2 * wave + j) * 16 + n;
        if (col < a.n_out) {
#pragma unroll
            for (int i = 0; i < 4; i++)
                if (kList || kSplit || row0 + i < a.n_rows) y[(row0 + i) * a.n_out + col] = v[i];
        }
    };
    auto fold = [&](int s) {  // the range that ends here joins the total of segment s (kSplit: goes to memory by itself)
        float *py = kSplit ? a.y + static_cast<size_t>(cut[0].wg - cut[0].first) * a.n_blocks * 16 * a.n_out : nullptr;
#pragma unroll
        for (int r = 0; r < RB; r++)
#pragma unroll
            for (int j = 0; j < 2; j++) {
                if (kPair && j != s) continue;
                const float4_t v = range_result(r, j);
                if constexpr (kSplit) {
                    store_y(py, r, j, v);
                } else {
                    float4_t &t = sum[kTotal ? r : 0][j];
                    t = first[s] ? v : t + v;
                }
                acc[r][j] = zero4;
                if (kTwin) sub[kTwin ? r : 0][j] = zero4;
            }
        first[s] = false;
    };

    auto walk_k = [&](auto partial) {
        for (int b = b_begin; b < b_end; b++) {
            landed(false);
            issue_x(b, 1);
            const bool more = b + 1 < b_end;
            if (more) issue_w(b + 1);
            compute(std::integral_constant<int, 0>(), partial, b);
            landed(more);
            if (more) issue_x(b + 1, 0);
            compute(std::integral_constant<int, 1>(), partial, b);
            if constexpr (kCut) {
#pragma unroll
                for (int s = 0; s < NSEG; s++) {
                    if constexpr (kSplit) {  // (the range's own number is needed before it moves on)
                        if (b + 1 == cut[s].next || !more) {
                            fold(s);
                            if (more) (void)cut[s].at(b + 1, a);
                        }
                    } else if (more && cut[s].at(b + 1, a)) {
                        fold(s);
                    }
                }
            }
        }
    };
    issue_x(b_begin, 0);
    issue_w(b_begin);
    if (blocks_left >= RB)
        walk_k(std::integral_constant<int, 0>());
    else
        walk_k(std::integral_constant<int, 1>());
    if constexpr (kSplit) return;
    if constexpr (kTotal) {
#pragma unroll
        for (int s = 0; s < NSEG; s++) fold(s);
    }
    auto result = [&](int r, int j) -> float4_t {
        if constexpr (kTotal) return sum[kTotal ? r : 0][j];
        return range_result(r, j);
    };

    if constexpr (kEpi == kEpiY) {
#pragma unroll
        for (int r = 0; r < RB; r++)
#pragma unroll
            for (int j = 0; j < 2; j++) store_y(a.y, r, j, result(r, j));
    } else if constexpr (kPair) {
        // out = silu(gate) * up, f16, the tile's 16 W columns through LDS (which the waves are done with) so that a lane holds
        // eight consecutive columns of a row - one slot of the fragment order - and a quad one sub-block
        __syncthreads();
        constexpr int kStride = 32 * W + 16;  // bytes per row of 16 W columns in f16
#pragma unroll
        for (int r = 0; r < RB; r++) {
            const float4_t gt = result(r, 0), up = result(r, 1);
#pragma unroll
            for (int i = 0; i < 4; i++) {
                float o = gt[i] / (1.0f + expf(-gt[i])) * up[i];
                asm volatile("" : "+v"(o));  // (the product is rounded to f32 first, as the block path's: not fused into the conversion)
                *reinterpret_cast<_Float16 *>(lds + (r * 16 + 4 * g + i) * kStride + (16 * wave + n) * 2) = static_cast<_Float16>(o);
            }
        }
        __syncthreads();
        const int oct = tid & (2 * W - 1), col = ct * 16 * W + 8 * oct;
#pragma unroll
        for (int it = 0; it < RB / 2 + (RB & 1); it++) {
            const int row = it * 32 + tid / (2 * W), blk = row >> 4, m = row & 15;
            if (RB % 2 && row >= RB * 16) break;
            const half8_t h = *reinterpret_cast<const half8_t *>(lds + row * kStride + oct * 16);
            const half8_t frag = {h[0], h[2], h[1], h[3], h[4], h[6], h[5], h[7]};
            _Float16 hv[8];
#pragma unroll
            for (int i = 0; i < 8; i++) hv[i] = h[i];
            float s = kList ? q4k_octet_sum_seq(hv) : q4k_octet_sum(hv);
            s += __shfl_xor(s, 1, 64);
            s += __shfl_xor(s, 2, 64);
            if (blk >= live) continue;
            *reinterpret_cast<half8_t *>(a.y_xf + static_cast<size_t>(block0 + blk) * a.nb_out * 8192 + dfl_xf_slot(a.y_kind, m, col)) = frag;
            if (a.y_xs && (oct & 3) == 0) {
                const int sb = col >> 8, jj = (col >> 5) & 7;
                _Float16 *o = reinterpret_cast<_Float16 *>(a.y_xs + (static_cast<size_t>(block0 + blk) * a.nb_out + sb) * 1024) +
                              (m + 16 * (jj >> 1)) * 8 + (jj & 1);
                const Q4KSumParts p = q4k_sum_parts(s);
                o[0] = p.hi;
                o[2] = p.lo;
                o[4] = p.over;
                o[6] = static_cast<_Float16>(0.0f);
            }
        }
    }
}

// y[row][col] = the ranges' partial products of a kSplit launch, added in the order of K (four columns per thread).
__global__ void __launch_bounds__(256) rows_reduce_kernel(RowsArgs a, const float *__restrict__ part, float *__restrict__ y) {
    const int col = 4 * (blockIdx.x * 256 + threadIdx.x), row = blockIdx.y;
    if (col >= a.n_out) return;
    Cut cut;
    cut.start(a.cut_by_group ? col >> 8 : 0, a);
    const int ranges = cut.ranges(a);
    const size_t stride = static_cast<size_t>(a.n_blocks) * 16 * a.n_out;
    const float *p = part + static_cast<size_t>(row) * a.n_out + col;
    if (a.n_out % 4 == 0) {
        float4_t s = *reinterpret_cast<const float4_t *>(p);
        for (int i = 1; i < ranges; i++) s += *reinterpret_cast<const float4_t *>(p + i * stride);
        *reinterpret_cast<float4_t *>(y + static_cast<size_t>(row) * a.n_out + col) = s;
        return;
    }
    for (int j = 0; j < 4 && col + j < a.n_out; j++) {
        float s = p[j];
        for (int i = 1; i < ranges; i++) s += p[j + i * stride];
        y[static_cast<size_t>(row) * a.n_out + col + j] = s;
    }
}

// Sub-block sums of rows in fragment order (kind Q4K), as the A operand of the minima's MFMA: one wave per (super-block, row block).
__global__ void __launch_bounds__(64) xf_sums_kernel(const uint8_t *__restrict__ xf, int nb, uint8_t *__restrict__ xs) {
    const int b = blockIdx.x, blk = blockIdx.y, lane = threadIdx.x;
    const half8_t *p = reinterpret_cast<const half8_t *>(xf + (static_cast<size_t>(blk) * nb + b) * 8192) + lane;
    float o[8];
#pragma unroll
    for (int t = 0; t < 8; t++) {
        const half8_t f = p[t * 64];  // element order 0 2 1 3 4 6 5 7
        const _Float16 h[8] = {f[0], f[2], f[1], f[3], f[4], f[6], f[5], f[7]};
        o[t] = q4k_octet_sum(h);
    }
    const half8_t r = q4k_sum_operand((o[0] + o[1]) + (o[2] + o[3]), (o[4] + o[5]) + (o[6] + o[7]));
    reinterpret_cast<half8_t *>(xs + (static_cast<size_t>(blk) * nb + b) * 1024)[lane] = r;
}

template <typename Tile, bool kTwin, int RB, int W>
constexpr size_t rows_lds() {
    return 2 * (static_cast<size_t>(RB) * 4096 + static_cast<size_t>(2 * W) * Tile::kBytes + (kTwin ? 0 : static_cast<size_t>(RB) * 1024));
}

}  // namespace

dfl_rows_plan dfl_gemm_rows_plan(const dflash_ctx *ctx, int32_t w_type, int64_t n_in, int64_t n_out, int64_t pair_ffn) {
    dfl_rows_plan p = {};
    if (w_type != DFLASH_TYPE_Q4_K_TILED && w_type != DFLASH_TYPE_Q6_K_TILED) return p;
    if (n_in <= 0 || n_in % DFL_QK_K || n_out <= 0 || n_out >= (1 << 24) || n_in >= (1 << 24)) return p;
    if (pair_ffn && (n_out != 2 * pair_ffn || pair_ffn % DFL_QK_K || w_type != DFLASH_TYPE_Q4_K_TILED)) return p;
    if (ctx->lds_bytes < 160 * 1024) return p;
    const int nb = static_cast<int>(n_in / DFL_QK_K);
    const int kind = dfl_whole_kind(ctx, w_type, n_in, n_out, pair_ffn);
    if (kind != DFL_XF_NONE) {
        p.kind = kind;
        p.twin = 1;
        p.total = nb;
        p.n_cut = nb < 16 ? nb : 16;  // the whole-K kernel's slices
        return p;
    }
    if (w_type != DFLASH_TYPE_Q4_K_TILED) return p;
    int total = 0, n_wg = 0;
    if (!dfl_q4k_tiled_split(ctx, n_in, n_out, &total, &n_wg)) return p;
    p.kind = DFL_XF_Q4K;
    p.total = total;
    p.n_cut = n_wg;
    p.by_group = 1;
    return p;
}

int32_t dfl_xf_sums(dflash_ctx *ctx, const void *xf, int64_t n_in, int32_t n_blocks, void *xs, hipStream_t st) {
    if (!xf || !xs || n_in <= 0 || n_in % DFL_QK_K || n_blocks < 1) return dfl_fail(ctx, DFLASH_ERR_BAD_SHAPE, "xf_sums: bad shape");
    xf_sums_kernel<<<dim3(static_cast<unsigned>(n_in / DFL_QK_K), n_blocks), 64, 0, st>>>(static_cast<const uint8_t *>(xf),
                                                                                       static_cast<int>(n_in / DFL_QK_K), static_cast<uint8_t *>(xs));
    DFL_HIP_CHECK(ctx, hipGetLastError());
    return DFLASH_OK;
}

namespace {
template <typename Tile, bool kTwin, bool kCut, int RB, int kEpi, bool kList>
int32_t rows_launch(dflash_ctx *ctx, const RowsArgs &a, int64_t tiles, hipStream_t st) {
    const auto fn = gemm_rows_kernel<Tile, kTwin, kCut, RB, kEpi, kList>;
    constexpr int W = kList ? kListWaves : kRowsWaves;
    const size_t lds = rows_lds<Tile, kTwin, RB, W>();
    if (const int32_t rc = dfl_raise_lds_limit(ctx, reinterpret_cast<const void *>(fn), lds)) return rc;
    if (tiles < 1 || tiles > 0x0fffffff) return dfl_fail(ctx, DFLASH_ERR_BAD_SHAPE, "gemm_rows: %lld tiles", static_cast<long long>(tiles));
    dfl_timed timer(ctx, st, DFL_T_GEMM);
    fn<<<static_cast<unsigned>((tiles + 7) / 8 * 8), 64 * W, lds, st>>>(a);
    DFL_HIP_CHECK(ctx, hipGetLastError());
    return DFLASH_OK;
}

// Row blocks per tile: the largest tile (the fewest unpackings per product) unless a smaller one leaves less of the last
// round of the chip idle: cost = rounds x (row blocks of a tile + what a tile costs besides).
int rows_pick_rb(const dflash_ctx *ctx, int n_blocks, int n_ct, int most) {
    int rb = most;
    int64_t best = -1;
    for (int r = most; r >= 2; r--) {
        const int64_t tiles = static_cast<int64_t>(n_ct) * ((n_blocks + r - 1) / r);
        const int64_t cost = (tiles + ctx->n_cu - 1) / ctx->n_cu * (4 * r + 5);
        if (best < 0 || cost < best) {
            best = cost;
            rb = r;
        }
    }
    return rb;
}

template <typename Tile, bool kTwin, int kEpi>
int32_t rows_dispatch(dflash_ctx *ctx, const RowsArgs &a, int rb, int64_t tiles, hipStream_t st) {
    switch (rb) {
        case 2: return rows_launch<Tile, kTwin, true, 2, kEpi, false>(ctx, a, tiles, st);
        case 3: return rows_launch<Tile, kTwin, true, 3, kEpi, false>(ctx, a, tiles, st);
        case 4: return rows_launch<Tile, kTwin, true, 4, kEpi, false>(ctx, a, tiles, st);
        default: break;
    }
    if constexpr (!kTwin) {
        switch (rb) {
            case 5: return rows_launch<Tile, kTwin, true, 5, kEpi, false>(ctx, a, tiles, st);
            case 6: return rows_launch<Tile, kTwin, true, 6, kEpi, false>(ctx, a, tiles, st);
            case 7: return rows_launch<Tile, kTwin, true, 7, kEpi, false>(ctx, a, tiles, st);
            case 8: return rows_launch<Tile, kTwin, true, 8, kEpi, false>(ctx, a, tiles, st);
            default: break;
        }
    }
    return dfl_fail(ctx, DFLASH_ERR_UNSUPPORTED, "gemm_rows: %d row blocks per tile", rb);
}
}  // namespace

int32_t dfl_gemm_rows(dflash_ctx *ctx, const dfl_rows_plan &p, int32_t w_type, const void *w, const void *xf, const void *xs, float *y,
                      int64_t n_in, int64_t n_out, int32_t n_rows, int64_t pair_ffn, void *y_xf, void *y_xs, int y_kind, hipStream_t st) {
    if (p.kind == DFL_XF_NONE || !w || !xf || n_rows < 1 || (!p.twin && !xs) || (pair_ffn ? !y_xf : !y))
        return dfl_fail(ctx, DFLASH_ERR_UNSUPPORTED, "gemm_rows: shape not taken or null operand");
    if (reinterpret_cast<uintptr_t>(w) % 16 || reinterpret_cast<uintptr_t>(xf) % 16 || reinterpret_cast<uintptr_t>(xs) % 16 ||
        reinterpret_cast<uintptr_t>(y_xf) % 16 || reinterpret_cast<uintptr_t>(y_xs) % 16)
        return dfl_fail(ctx, DFLASH_ERR_ALIGNMENT, "gemm_rows: operand alignment");
    RowsArgs a = {};
    a.w[0] = a.w[1] = static_cast<const uint8_t *>(w);
    a.nb = static_cast<int>(n_in / DFL_QK_K);
    a.n_rows = n_rows;
    a.n_blocks = (n_rows + 15) / 16;
    a.xf = static_cast<const uint8_t *>(xf);
    a.xs = static_cast<const uint8_t *>(xs);
    a.total = p.total;
    a.n_cut = p.n_cut;
    a.cut_by_group = p.by_group;
    a.y = y;
    a.n_out = static_cast<int>(n_out);
    a.tile0_up = static_cast<int>(pair_ffn / 16);
    a.y_xf = static_cast<uint8_t *>(y_xf);
    a.y_xs = static_cast<uint8_t *>(y_xs);
    a.y_kind = y_kind;
    a.nb_out = static_cast<int>(pair_ffn / DFL_QK_K);
    a.n_ct = static_cast<int>(pair_ffn ? pair_ffn / 128 : (n_out + 255) / 256);
    const int most = p.twin ? 4 : 8;
    int rb = rows_pick_rb(ctx, a.n_blocks, a.n_ct, most);
    a.n_rt = (a.n_blocks + rb - 1) / rb;
    int64_t tiles = static_cast<int64_t>(a.n_ct) * a.n_rt;
    if (pair_ffn) return p.twin ? rows_dispatch<TileQ4, true, kEpiSwiglu>(ctx, a, rb, tiles, st) : rows_dispatch<TileQ4, false, kEpiSwiglu>(ctx, a, rb, tiles, st);
    // Tiles for less than half the chip: K is shared by several workgroups, each range between two cuts on its own (as
    // many as there are at least in every tile group), where the workspace holds the partial products.
    const int ranges = p.by_group ? std::max(1, static_cast<int>(static_cast<int64_t>(a.nb) * a.n_cut / a.total)) : a.n_cut;
    const int most_ranges = p.by_group ? static_cast<int>((static_cast<int64_t>(a.nb) * a.n_cut + a.total - 1) / a.total) + 1 : a.n_cut;
    if (2 * tiles <= ctx->n_cu && ranges > 1) {
        // The whole-K kernel does the few blocks of a short prompt in one launch, one block after the other: 1.5 us each past
        // weights it holds unpacked, 4 to 10 us each where a wave has two tiles or two super-blocks and unpacks them again.
        // The split with its reduction costs 9 to 18 us and then the less per block the smaller the matrix.  Crossing points,
        // Q4_K and Q6_K alike (whole : split in us, 2 / 4 / 12 blocks, Q4_K):
        //   held    2048 -> 5120  7.9 : 11.7  10.7 : 16.1  21.9 : 23.3     4096 -> 4096  8.3 : 15.6  11.4 : 19.2  24.4 : 32.9
        //           2560 -> 2560  6.3 : 11.5   8.0 : 12.5  17.1 : 17.8     4096 -> 2048  8.2 : 13.0  11.0 : 15.0  22.8 : 22.4
        //           1024 -> 4096  6.6 :  9.2   9.4 : 10.2  21.2 : 17.0     2048 -> 1024  6.3 :  9.5   9.2 :  9.8  20.6 : 11.6
        //   not     4096 -> 6144 22.1 : 17.9  29.6 : 22.9  (Q6_K 32.5 : 19.5  50.5 : 27.8)
        //           4096 -> 5120 20.4 : 18.9  27.8 : 20.1  (Q6_K 32.1 : 21.8  49.0 : 24.1), 5120 -> 6144 52.6 : 18.1  69.3 : 23.5
        // so: twelve blocks for matrices of 80 super-blocks x column tiles or more, four for smaller ones, none where the
        // weights are not held.
        const int whole_most = a.nb * a.n_ct >= 80 ? 12 : 4;
        if (p.twin && a.n_blocks <= whole_most && dfl_whole_holds_weights(ctx, w_type, n_in, n_out))
            return dfl_gemm_whole_blocks(ctx, w_type, w, xf, y, n_in, n_out, n_rows, 0, nullptr, 0, st);
        a.n_split = std::min<int>(ranges, static_cast<int>(ctx->n_cu / tiles));
        size_t off = 0;
        float *part = dfl_ws_take<float>(ctx, &off, static_cast<size_t>(most_ranges) * a.n_blocks * 16 * n_out * sizeof(float));
        if (part && a.n_split > 1) {
            a.y = part;
            tiles *= a.n_split;
            const int32_t rc = w_type == DFLASH_TYPE_Q6_K_TILED ? rows_dispatch<TileQ6, true, kEpiSplit>(ctx, a, rb, tiles, st)
                               : p.twin                         ? rows_dispatch<TileQ4, true, kEpiSplit>(ctx, a, rb, tiles, st)
                                                                : rows_dispatch<TileQ4, false, kEpiSplit>(ctx, a, rb, tiles, st);
            if (rc) return rc;
            rows_reduce_kernel<<<dim3(static_cast<unsigned>((n_out + 1023) / 1024), n_rows), 256, 0, st>>>(a, part, y);
            DFL_HIP_CHECK(ctx, hipGetLastError());
            return DFLASH_OK;
        }
    }
    if (w_type == DFLASH_TYPE_Q6_K_TILED) return rows_dispatch<TileQ6, true, kEpiY>(ctx, a, rb, tiles, st);
    return p.twin ? rows_dispatch<TileQ4, true, kEpiY>(ctx, a, rb, tiles, st) : rows_dispatch<TileQ4, false, kEpiY>(ctx, a, rb, tiles, st);
}

int32_t dfl_gemm_rows_experts(dflash_ctx *ctx, const void *w, const void *w_extra, const void *w_up, const void *w_up_extra, size_t w_stride,
                              const void *xf, const void *xs, const int32_t *tiles, const int32_t *n_tiles, int32_t max_tiles, float *y,
                              int64_t n_in, int64_t n_out, void *y_xf, void *y_xs, hipStream_t st) {
    if (!w || !w_extra || !xf || !xs || !tiles || !n_tiles || max_tiles < 1 || n_in <= 0 || n_in % DFL_QK_K || n_out <= 0 || n_out % DFL_QK_K ||
        (w_up ? (!w_up_extra || !y_xf || !y_xs) : !y) || ctx->lds_bytes < 160 * 1024)
        return dfl_fail(ctx, DFLASH_ERR_UNSUPPORTED, "gemm_rows_experts: shape not taken or null operand");
    RowsArgs a = {};
    a.w[0] = static_cast<const uint8_t *>(w);
    a.w[1] = static_cast<const uint8_t *>(w_up ? w_up : w);
    a.w_extra[0] = static_cast<const uint8_t *>(w_extra);
    a.w_extra[1] = static_cast<const uint8_t *>(w_up ? w_up_extra : w_extra);
    a.w_stride = w_stride;
    a.nb = static_cast<int>(n_in / DFL_QK_K);
    a.xf = static_cast<const uint8_t *>(xf);
    a.xs = static_cast<const uint8_t *>(xs);
    a.tiles = reinterpret_cast<const int4 *>(tiles);
    a.n_tiles = n_tiles;
    a.y = y;
    a.n_out = static_cast<int>(n_out);
    a.y_xf = static_cast<uint8_t *>(y_xf);
    a.y_xs = static_cast<uint8_t *>(y_xs);
    a.y_kind = DFL_XF_Q4K;
    a.nb_out = static_cast<int>(n_out / DFL_QK_K);
    a.n_ct = static_cast<int>(n_out / ((w_up ? 16 : 32) * kListWaves));
    const int64_t tiles_max = static_cast<int64_t>(max_tiles) * a.n_ct;
    return w_up ? rows_launch<TileQ4, false, false, 4, kEpiSwiglu, true>(ctx, a, tiles_max, st)
                : rows_launch<TileQ4, false, false, 4, kEpiY, true>(ctx, a, tiles_max, st);
}
