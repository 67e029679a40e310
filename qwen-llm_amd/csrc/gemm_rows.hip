// Many-row quantised GEMM of a prompt's prefill: Y[rows][n_out] = X[rows][n_in] . W^T for the rows of many 16-row
// blocks at once, X handed over in MFMA fragment order (common.h, "XF"), W in the library's tiled orders.
// Same contraction as encode_mat_mat_dispatch_dflash_verify (metal_forward/dispatch.rs:365-378).
//
// What bounds it.  With sixteen rows a weight is unpacked for one MFMA and the kernel streams weights; here a weight
// unpacked once serves up to 128 rows, and the matrix cores are what there is most of to do: a wave's 2 MFMAs per
// fragment, with the fragment's LDS read and its share of the unpacking (4 vector instructions), run at 1.5 PFLOP/s where
// nothing else stands in the way (random operands, clock held down to 1.6 GHz by the power they draw; the MFMAs alone 2.0).
// A workgroup of eight waves computes 16 RB rows x 256 columns (a SwiGLU pair: 128 gate and the 128 up columns that go with
// them); a wave, 16 RB rows x 32 columns:
//   * the activations of its row blocks (half a super-block at a time, three halves in LDS) and the raw quant blocks of its
//     own two 16-row weight tiles (one super-block) are copied into LDS with direct-to-LDS loads, both as they lie in memory
//     (contiguous pieces: weights loaded straight into registers touch eighteen lines a load and cost 10 %), the activations
//     one to two halves ahead, the weights one super-block;
//   * the copies stand one by one between the products, and an LDS read six products ahead of its own: a wave that issues a
//     super-block's copies together stands still until the memory pipeline has taken them;
//   * no two waves unpack the same weights (with the waves two by four, which halves the LDS reads, the unpacking on the
//     vector ALU took as long as the products); an activation fragment read from LDS feeds two products;
//   * the weights stay quantised up to the registers: a matrix is read from memory once and from L2 once per row tile, at
//     4.5 or 6.6 bits a weight instead of 16.
// Workgroups that share weights are dispatched to one XCD (rows_linear), so that a matrix passes through one L2.
// Measured for 1000 rows, before (a whole super-block's copies behind a barrier, the compiler's waits: every LDS read waited
// for ahead of its two products) and now, six layers of a prompt: 5120 -> 2 x 17408 with SwiGLU 429 -> 364 us (0.98
// PFLOP/s, matrix cores busy for 57 % of the cycles, 42 % before), 17408 -> 5120 233 -> 193 us (0.92), 5120 -> 6144 105 -> 76 us
// (0.82; the 105 with a twin MFMA for every product, which the block path's bits then asked for); 2048 rows: 2048 -> 5120 and
// 4096 -> 2048 in Q6_K, still with twins, together 220 -> 186 us.  A 64-layer prompt of 1000 rows 64.7 -> 59.7 ms, 53.5 without the twins.
// The experts' tiles (a list) take workgroups of half the columns and up to four row blocks, two of them on a CU, each
// waiting for its own weights while the other computes, or, where an expert has rows enough, of all columns and up to eight blocks
// (the rule and both sides' figures stand in dfl_moe_ffn_group).
//
// Bits.  Every row of Y has the bits that the 16-row kernels give it in its own block.  The arithmetic of a
// super-block is theirs (the same unpacking, the same v_mfma_f32_16x16x32_f16 sequence into the same accumulator); K is
// walked in order, and where those kernels cut K - the whole-K kernel's slices (gemm_whole.hip), the stream-K ranges
// (gemm_fewrow.hip) - the accumulator is added to a running total and starts again from zero, in the order their
// partial tiles are added in.  That order is also what a split of K over workgroups has to keep: each range between two
// cuts goes to memory on its own and rows_reduce_kernel adds them up (kSplit; few rows against a narrow matrix).
#include "common.h"
#include "lds_read.h"
#include "mfma_unpack.h"

#include <algorithm>
#include <type_traits>

namespace {

typedef const __attribute__((address_space(1))) void *gptr_t;
typedef __attribute__((address_space(3))) void *lptr_t;

constexpr int kRowsWaves = 8;

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

typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));

// this wave's loads into LDS but for the last N are done
template <int N>
__device__ __forceinline__ void copies_done() {
    __builtin_amdgcn_s_waitcnt((N & 0xF) | ((N & 0x30) << 10) | 0x0F70);  // vmcnt(N)
    asm volatile("" ::: "memory");
}

// One tile's weights of one super-block in a lane's registers: read asks LDS for the lane's quant bytes (kReads reads, there
// behind arrived), scales makes of them what operand<H>(t), the operand of MFMA 4 H + t, needs besides.
struct TileQ4 {
    static constexpr int kBytes = 16 * DFL_Q4_K_BYTES, kReads = 3;
    struct At {
        uint32_t hdr, q;
        __device__ __forceinline__ At(uint32_t tile, int n, int g) : hdr(tile + n * DFL_Q4_K_BYTES), q(hdr + 32 * g) {}
    };
    u32x4_t hdr, q0, q1;
    half2_t S, Cs, m;
    template <int OFF>
    __device__ __forceinline__ void read(const At &at) {
        hdr = lds_read<u32x4_t, OFF>(at.hdr);
        q0 = lds_read<u32x4_t, OFF + 16>(at.q);
        q1 = lds_read<u32x4_t, OFF + 32>(at.q);
    }
    __device__ __forceinline__ void arrived() { asm volatile("" : "+v"(hdr), "+v"(q0), "+v"(q1)); }
    __device__ __forceinline__ void scales(int g, uint32_t sc_sel, bool negate_min) {
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
    __device__ __forceinline__ half8_t minima() const { return q4k_min_operand(m); }
};

struct TileQ6 {
    static constexpr int kBytes = kQ6TileBytes, kReads = 6;
    struct At {
        uint32_t ql, ql1, qh, qh1, sc, d;
        __device__ __forceinline__ At(uint32_t tile, int n, int g)
            : ql(tile + q6t_ql_piece(n, 2 * g)), ql1(tile + q6t_ql_piece(n, 2 * g + 1)), qh(tile + q6t_qh_piece(n, g & 2)),
              qh1(tile + q6t_qh_piece(n, (g & 2) + 1)), sc(tile + kQ6TSc + n * 16 + 4 * (g & 2)), d(tile + kQ6TD + n * 2) {}
    };
    u32x4_t qa, qb, ha, hb;
    u32x2_t sc;
    uint32_t d16;
    _Float16 s[4];
    int odd2;
    template <int OFF>
    __device__ __forceinline__ void read(const At &at) {
        qa = lds_read<u32x4_t, OFF>(at.ql);
        qb = lds_read<u32x4_t, OFF>(at.ql1);
        ha = lds_read<u32x4_t, OFF>(at.qh);
        hb = lds_read<u32x4_t, OFF>(at.qh1);
        sc = lds_read<u32x2_t, OFF>(at.sc);
        d16 = lds_read<uint32_t, OFF>(at.d);
    }
    __device__ __forceinline__ void arrived() { asm volatile("" : "+v"(qa), "+v"(qb), "+v"(ha), "+v"(hb), "+v"(sc), "+v"(d16)); }
    __device__ __forceinline__ void scales(int g, uint32_t, bool) {
        const int odd = g & 1;
        const float d = __half2float(__ushort_as_half(static_cast<uint16_t>(d16)));
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
    __device__ __forceinline__ half8_t minima() const { return splat8(static_cast<_Float16>(0.0f)); }  // (named, never asked for)
};

// this wave's reads from LDS are done, and everybody has come this far
__device__ __forceinline__ void landed_for_all() {
    __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// Dispatch index -> linear tile index: the hardware deals consecutive workgroups to the eight XCDs in turn, so dispatch
// indices i, i + 8, i + 16, ... share an L2; they get consecutive tiles.  Returns -1 past the end.
__device__ __forceinline__ int rows_linear(int dispatch, int count) {
    const int per = (count + 7) >> 3, at = dispatch >> 3, l = (dispatch & 7) * per + at;
    return at < per && l < count ? l : -1;
}

enum { kEpiY = 0, kEpiSwiglu = 1, kEpiSplit = 2 };

// LDS of a tile: three halves of a super-block of its activations (4 KB per row block), two super-blocks of their sub-block
// sums where the minima go by them, one of every wave's weights.
template <typename Tile, bool kTwin, int RB, int W>
struct RowsLds {
    static constexpr int kHalf = RB * 4096, kSums = kTwin ? 0 : RB * 1024, kW = 2 * Tile::kBytes;
    static constexpr int sums = 3 * kHalf, w = sums + 2 * kSums, total = w + W * kW;
};

// kTwin: the minima / offsets through a twin MFMA per activation fragment into a second accumulator (the whole-K kernel's
// arithmetic for Q6_K and short K); else one MFMA per super-block over the sub-block sums.
// kCut: K is cut somewhere.  RB: 16-row blocks of the tile.
template <typename Tile, bool kTwin, bool kCut, int RB, int kEpi, int kList>
__global__ void __launch_bounds__(64 * (kList ? kList : kRowsWaves), 2) gemm_rows_kernel(RowsArgs a) {
    constexpr int W = kList ? kList : kRowsWaves;  // waves, 32 columns each
    constexpr bool kPair = kEpi == kEpiSwiglu, kSplit = kEpi == kEpiSplit, kTotal = kCut && !kSplit;
    constexpr int NSEG = kPair ? 2 : 1, kSegTiles = 2 * W / NSEG;
    typedef RowsLds<Tile, kTwin, RB, W> Lds;
    static_assert(8 / W * Lds::total <= 160 * 1024, "a CU's LDS");
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
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
        __builtin_amdgcn_global_load_lds((gptr_t)(src + static_cast<uint32_t>(lane * 16)), (lptr_t)(dst), 16, 0, 0);
    };
    // A wave makes the same number of copies in every half of a super-block (where the pieces do not come out even, some copy
    // what another copies too), so that a constant says how many may still be under way.
    auto copy_x = [&](auto rows, int half, int slot, int j) {  // half-super-block `half` of `rows` row blocks, this wave's piece j
        constexpr int R = decltype(rows)::value;
        const int p = min(wave + W * j, R * 4 - 1), blk = min(p >> 2, blocks_left - 1);  // (blocks past the end repeat the last one)
        copy(xf0 + blk * xf_stride + static_cast<size_t>(half) * 4096 + (p & 3) * 1024, lds + slot * Lds::kHalf + p * 1024);
    };
    auto copy_s = [&](auto rows, int b) {
        constexpr int R = decltype(rows)::value;
        static_assert(RB <= W, "a wave copies one block's sums");
        const int blk = min(wave, R - 1);
        copy(xs0 + min(blk, blocks_left - 1) * xs_stride + static_cast<size_t>(b) * 1024, lds + Lds::sums + (b & 1) * Lds::kSums + blk * 1024);
    };
    // (a wave-load less than a whole one starts early enough to be one)
    constexpr int kWRun = kPair ? Tile::kBytes : 2 * Tile::kBytes, kWLoads = (kWRun + 1023) / 1024, kWCopies = NSEG * kWLoads;
    auto copy_w = [&](int b, int i) {
        const int s = i / kWLoads, at = min(i % kWLoads * 1024, kWRun - 1024);
        copy(wbase[s] + static_cast<size_t>(b) * 16 * Tile::kBytes + wave * kWRun + at, lds + Lds::w + wave * Lds::kW + s * Tile::kBytes + at);
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

    const int live = min(blocks_left, RB);
    Tile tile[2];
    const uint32_t lds0 = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((lptr_t)lds));
    const typename Tile::At w_at(lds0 + Lds::w + wave * Lds::kW, n, g);
    // The products of a super-block stand in the order step (the minima, then MFMA 0 to 7 of a tile), row block.  A product's
    // fragment is read kRing products ahead, the weights of a step are unpacked under the products of the one before, and the
    // copies stand between the products (a wave that issues many at once waits at the issue and computes nothing meanwhile).
    // A barrier says that a half has landed for everybody and that everybody has read the one before it; it comes
    // when the ring still holds kTail fragments, whose products then cover the first reads of the new half.  So what runs
    // from one such barrier to the same one a super-block later begins with the last kTail products of the super-block before.
    auto product = [&](auto row, const half8_t &x, const half8_t (&o)[4]) {
        constexpr int r = decltype(row)::value, z = kTwin ? r : 0;
        acc[r][0] = __builtin_amdgcn_mfma_f32_16x16x32_f16(x, o[0], acc[r][0], 0, 0, 0);
        acc[r][1] = __builtin_amdgcn_mfma_f32_16x16x32_f16(x, o[1], acc[r][1], 0, 0, 0);
        if constexpr (kTwin) {
            sub[z][0] = __builtin_amdgcn_mfma_f32_16x16x32_f16(x, o[2], sub[z][0], 0, 0, 0);
            sub[z][1] = __builtin_amdgcn_mfma_f32_16x16x32_f16(x, o[3], sub[z][1], 0, 0, 0);
        }
    };
    auto operands = [&](auto st, half8_t (&o)[4]) {  // the weights of a step, and their twins
        constexpr int step = decltype(st)::value - (kTwin ? 0 : 1);
#pragma unroll
        for (int j = 0; j < 2; j++) {
            if constexpr (step < 0) {
                o[j] = tile[j].minima();
            } else {
                o[j] = tile[j].template operand<step / 4>(step % 4, magic);
                if constexpr (kTwin) o[2 + j] = tile[j].template twin<step / 4>(step % 4);
            }
        }
    };
    auto range_result = [&](int r, int j) -> float4_t {
        if constexpr (kTwin) return acc[r][j] - sub[kTwin ? r : 0][j];
        return acc[r][j];
    };
    auto store_y = [&](float *y, int r, int j, float4_t v) __attribute__((always_inline)) {
        if (r >= live) return;
        const int64_t row0 = static_cast<int64_t>(block0 + r) * 16 + 4 * g;
        const int col = (tile0[0] + 2 * wave + j) * 16 + n;
        if (col < a.n_out) {
#pragma unroll
            for (int i = 0; i < 4; i++)
                if (kList || kSplit || row0 + i < a.n_rows) y[(row0 + i) * a.n_out + col] = v[i];
        }
    };
    auto fold = [&](int s) __attribute__((always_inline)) {  // the range that ends here joins the total of segment s (kSplit: goes to memory by itself)
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

    auto walk_k = [&](auto rows) __attribute__((always_inline)) {
        constexpr int R = decltype(rows)::value, kFirst = kTwin ? 0 : 1, kSteps = 8 + kFirst, N = kSteps * R, kMid = (4 + kFirst) * R;
        constexpr int kRing = kTwin ? 4 : R == 1 || R == 3 ? 3 : R == 5 || R == 7 ? R : 6;  // (divides N: a fragment's place is its product's index)
        constexpr int kTail = kRing - kRing / 2, kTail0 = (N - kTail) / R, kTailSteps = kSteps - kTail0;
        constexpr int kX = (R * 4 + W - 1) / W, kEarly = kWCopies + kX, kLate = kFirst + kX;  // copies in the first part and in the second
        constexpr int kSwitch = kMid - kTail, kEnd = N - kTail;  // the barriers stand ahead of these products
        // The next weights are read ahead of this one: into the registers of the present ones where all of those are unpacked by
        // then (the last step's are while the step before it begins), else into others.
        constexpr bool kInPlace = R > 2;
        constexpr int kReadW = kInPlace && kEnd - 1 - kRing < (kSteps - 2) * R ? (kSteps - 2) * R : kEnd - 1 - kRing;
        static_assert(N % kRing == 0 && kReadW >= kSwitch && kReadW < kEnd, "shape of the pipeline");
        half8_t ring[kRing], tail[kTailSteps][4];
        // fragments asked for ahead of the wait of product i
        struct Reads {
            static constexpr int upto(int i) { return i < kSwitch ? (i + kRing < kMid ? i + kRing : kMid) : i + kRing < N ? i + kRing : N; }
            static constexpr int later(int i) {
                return upto(i) - i - 1 + (i >= kReadW && i < upto(kReadW) ? 2 * Tile::kReads : 0);
            }
        };
        auto body = [&](int b, int ahead, int slot) __attribute__((always_inline)) {
            const int slot1 = slot == 2 ? 0 : slot + 1, slot2 = slot1 == 2 ? 0 : slot1 + 1;
            const uint32_t at_s = lds0 + Lds::sums + (b & 1) * Lds::kSums + lane * 16;
            const uint32_t at0 = lds0 + slot * Lds::kHalf + lane * 16, at1 = lds0 + slot1 * Lds::kHalf + lane * 16;
            auto read = [&](auto i) {
                constexpr int I = decltype(i)::value, step = I / R - kFirst, r = I % R;
                if constexpr (step < 0)
                    ring[I % kRing] = lds_read<half8_t, r * 1024>(at_s);
                else if constexpr (step < 4)
                    ring[I % kRing] = lds_read<half8_t, r * 4096 + step * 1024>(at0);
                else
                    ring[I % kRing] = lds_read<half8_t, r * 4096 + (step - 4) * 1024>(at1);
            };
            // first part: the next super-block's weights, then its first half's activations; second: its sums and its second half's
            auto copies = [&](auto i) {
                constexpr int I = decltype(i)::value;
                if constexpr (I < kSwitch) {
                    constexpr int at = I + kTail;
                    static_for<at * kEarly / kMid, (at + 1) * kEarly / kMid>([&](auto c) {
                        constexpr int C = decltype(c)::value;
                        if constexpr (C < kWCopies)
                            copy_w(ahead, C);
                        else
                            copy_x(rows, 2 * ahead, slot2, C - kWCopies);
                    });
                } else {
                    constexpr int at = I - kSwitch;
                    static_for<at * kLate / (N - kMid), (at + 1) * kLate / (N - kMid)>([&](auto c) {
                        constexpr int C = decltype(c)::value;
                        if constexpr (C < kFirst)
                            copy_s(rows, ahead);
                        else
                            copy_x(rows, 2 * ahead + 1, slot, C - kFirst);
                    });
                }
            };
            half8_t op[4], op_next[4];
            Tile next[2];
            static_for<0, kTail>([&](auto t) {  // what is left of the super-block before
                constexpr int I = decltype(t)::value - kTail, P = N + I;
                static_for<(I == -kTail ? 0 : Reads::upto(I - 1)), Reads::upto(I)>(read);
                copies(std::integral_constant<int, I>());
                product(std::integral_constant<int, P % R>(), ring[P % kRing], tail[P / R - kTail0]);
                if constexpr (I == -kTail) {
#pragma unroll
                    for (int j = 0; j < 2; j++) tile[j].scales(g, sc_sel, !kTwin);
                    operands(std::integral_constant<int, 0>(), op);
                }
            });
            if constexpr (kCut) {
                // (no register waits for LDS where the code branches: the compiler may copy one there)
                __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
#pragma unroll
                for (int i = 0; i < kRing; i++) asm volatile("" : "+v"(ring[i]));
                if (b > b_begin) {
#pragma unroll
                    for (int s = 0; s < NSEG; s++) {
                        if constexpr (kSplit) {  // (the range's own number is needed before it moves on)
                            if (b == cut[s].next) {
                                fold(s);
                                (void)cut[s].at(b, a);
                            }
                        } else if (cut[s].at(b, a)) {
                            fold(s);
                        }
                    }
                }
            }
            static_for<0, kEnd>([&](auto i) {
                constexpr int I = decltype(i)::value, step = I / R, r = I % R;
                if constexpr (r == 0 && step + 1 < kSteps && !(kInPlace && I > kReadW)) operands(std::integral_constant<int, step + 1>(), op_next);
                if constexpr (I == kSwitch) {  // the second half is in LDS for everybody, and everybody has read the first
                    copies_done<kEarly>();
                    landed_for_all();
                }
                static_for<Reads::upto(I - 1), Reads::upto(I)>(read);
                if constexpr (I == kReadW) {  // (the weights were the first copies of this super-block)
                    copies_done<kX + (I - kSwitch) * kLate / (N - kMid)>();
                    if constexpr (kInPlace) {
                        static_for<kTail0, kSteps>([&](auto st) { operands(st, tail[decltype(st)::value - kTail0]); });
#pragma unroll
                        for (int q = 0; q < kTailSteps; q++)
#pragma unroll
                            for (int j = 0; j < (kTwin ? 4 : 2); j++) asm volatile("" : "+v"(tail[q][j]));
                    }
                    (kInPlace ? tile : next)[0].template read<0>(w_at);
                    (kInPlace ? tile : next)[1].template read<Tile::kBytes>(w_at);
                }
                copies(i);
                lds_arrived<Reads::later(I)>(ring[I % kRing]);
                if constexpr (kInPlace && step >= kTail0 && I >= kReadW)
                    product(std::integral_constant<int, r>(), ring[I % kRing], tail[step - kTail0]);
                else
                    product(std::integral_constant<int, r>(), ring[I % kRing], op);
                if constexpr (r == R - 1) {
#pragma unroll
                    for (int j = 0; j < 4; j++) op[j] = op_next[j];
                }
            });
            if constexpr (!kInPlace) static_for<kTail0, kSteps>([&](auto st) { operands(st, tail[decltype(st)::value - kTail0]); });
            copies_done<kX>();  // all but the second half's activations
            landed_for_all();
#pragma unroll
            for (int i = 0; i < kRing; i++) asm volatile("" : "+v"(ring[i]));
#pragma unroll
            for (int j = 0; j < 2; j++) {
                (kInPlace ? tile : next)[j].arrived();
                if (!kInPlace) tile[j] = next[j];
            }
        };
#pragma unroll
        for (int i = 0; i < kWCopies; i++) copy_w(b_begin, i);
        if constexpr (!kTwin) copy_s(rows, b_begin);
#pragma unroll
        for (int h = 0; h < 2; h++)
#pragma unroll
            for (int j = 0; j < kX; j++) copy_x(rows, 2 * b_begin + h, h, j);
        copies_done<kX>();  // (all but the second half)
        tile[0].template read<0>(w_at);
        tile[1].template read<Tile::kBytes>(w_at);
        landed_for_all();
        tile[0].arrived();
        tile[1].arrived();
        const half8_t none = splat8(static_cast<_Float16>(0.0f));  // (nothing is left of the super-block before the first)
#pragma unroll
        for (int i = 0; i < kRing; i++) ring[i] = none;
#pragma unroll
        for (int i = 0; i < kTailSteps; i++)
#pragma unroll
            for (int j = 0; j < 4; j++) tail[i][j] = none;
        int slot = 0;
        for (int b = b_begin; b < b_end; b++) {
            body(b, min(b + 1, b_end - 1), slot);  // (the last one copies itself again, to where nobody reads any more)
            slot = slot == 0 ? 2 : slot - 1;
        }
        static_for<N - kTail, N>([&](auto i) {
            constexpr int P = decltype(i)::value;
            product(std::integral_constant<int, P % R>(), ring[P % kRing], tail[P / R - kTail0]);
        });
        if constexpr (kSplit) fold(0);
        copies_done<0>();  // (the epilogue has other uses for LDS, and the next workgroup too)
    };
    // An expert's few rows are computed alone, by code of their own; a tail of no more than half the tile's blocks as half a tile.
    // What the instances of a list earn against 1, 2, 4 and 8 alone (a layer of a mixture's prompt, 128 experts top-8, rows,
    // that : this): 2048 697 : 673 us, 1500 550 : 536, 600 300 : 295; 32 top-4, 1000 rows 320 : 314.
    if constexpr (kList) {
        switch (live) {
            case 1: walk_k(std::integral_constant<int, 1>()); break;
            case 2: walk_k(std::integral_constant<int, 2>()); break;
            case 3: walk_k(std::integral_constant<int, 3>()); break;
            default:
                if constexpr (RB > 4) {
                    switch (live) {
                        case 4: walk_k(std::integral_constant<int, 4>()); break;
                        case 5: walk_k(std::integral_constant<int, 5>()); break;
                        case 6: walk_k(std::integral_constant<int, 6>()); break;
                        case 7: walk_k(std::integral_constant<int, 7>()); break;
                        default: walk_k(std::integral_constant<int, RB>()); break;
                    }
                } else {
                    walk_k(std::integral_constant<int, RB>());
                }
                break;
        }
        static_assert(!kList || RB == kList, "a list's tiles");
    } else {
        constexpr int kHalf = RB > 2 ? (RB + 1) / 2 : RB;
        if (live <= kHalf)
            walk_k(std::integral_constant<int, kHalf>());
        else if constexpr (kHalf < RB)
            walk_k(std::integral_constant<int, RB>());
    }
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

}  // namespace

dfl_rows_plan dfl_gemm_rows_plan(const dflash_ctx *ctx, int32_t w_type, int64_t n_in, int64_t n_out, int64_t pair_ffn, bool row_major) {
    dfl_rows_plan p = {};
    if (w_type != DFLASH_TYPE_Q4_K_TILED && w_type != DFLASH_TYPE_Q6_K_TILED) return p;
    if (n_in <= 0 || n_in % DFL_QK_K || n_out <= 0 || n_out >= (1 << 24) || n_in >= (1 << 24)) return p;
    if (pair_ffn && (n_out != 2 * pair_ffn || pair_ffn % DFL_QK_K || w_type != DFLASH_TYPE_Q4_K_TILED)) return p;
    if (ctx->lds_bytes < 160 * 1024) return p;
    const int nb = static_cast<int>(n_in / DFL_QK_K);
    const int kind = row_major && w_type == DFLASH_TYPE_Q4_K_TILED ? DFL_XF_NONE : dfl_whole_kind(ctx, w_type, n_in, n_out, pair_ffn);
    if (kind != DFL_XF_NONE) {
        p.kind = kind;
        p.whole = 1;
        p.sums = dfl_whole_by_sums(ctx, w_type, n_in, n_out, pair_ffn);
        p.total = nb;
        p.n_cut = nb < 16 ? nb : 16;  // the whole-K kernel's slices
        return p;
    }
    if (w_type != DFLASH_TYPE_Q4_K_TILED) return p;
    if (pair_ffn && dfl_gemm_dense_pair_takes(ctx, w_type, n_in, pair_ffn)) {  // (one sum over the whole K)
        p.kind = DFL_XF_Q4K;
        p.sums = 1;
        p.total = nb;
        p.n_cut = 1;
        return p;
    }
    int total = 0, n_wg = 0;
    if (!dfl_q4k_tiled_split(ctx, n_in, n_out, &total, &n_wg)) return p;
    p.kind = DFL_XF_Q4K;
    p.sums = 1;
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
template <typename Tile, bool kTwin, bool kCut, int RB, int kEpi, int kList>
int32_t rows_launch(dflash_ctx *ctx, const RowsArgs &a, int64_t tiles, hipStream_t st) {
    const auto fn = gemm_rows_kernel<Tile, kTwin, kCut, RB, kEpi, kList>;
    constexpr int W = kList ? kList : kRowsWaves;
    const size_t lds = RowsLds<Tile, kTwin, RB, W>::total;
    if (const int32_t rc = dfl_raise_lds_limit(ctx, reinterpret_cast<const void *>(fn), lds)) return rc;
    if (tiles < 1 || tiles > 0x0fffffff) return dfl_fail(ctx, DFLASH_ERR_BAD_SHAPE, "gemm_rows: %lld tiles", static_cast<long long>(tiles));
    dfl_timed timer(ctx, st, DFL_T_GEMM);
    fn<<<static_cast<unsigned>((tiles + 7) / 8 * 8), 64 * W, lds, st>>>(a);
    DFL_HIP_CHECK(ctx, hipGetLastError());
    return DFLASH_OK;
}

// Row blocks per tile: the largest tile (the fewest unpackings per product) unless a smaller one leaves less of the last
// round of the chip idle: cost = rounds x (row blocks of a tile + what a tile costs besides).
int rows_pick_rb(const dflash_ctx *ctx, int n_blocks, int n_ct, int most, int64_t *cost_of = nullptr) {
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
    if (cost_of) *cost_of = best;
    return rb;
}

// The same where the workgroups of a tile share K: what larger tiles leave idle goes to more shares, so the cost is that
// of the longest share, and the weights are read by fewer row tiles.  The tile by whole rounds (2 blocks) : this one.  Q4_K,
// 100 rows, 5120 -> 6144, 4096 -> 5120 and 17408 -> 5120 on average 28.1 : 23.8 us (6 and 3 blocks); 200 rows, 4096 -> 5120 26.5 :
// 23.2 (4).  Q6_K, 300 rows, 4096 -> 2048 27.4 : 20.2 (4).
int rows_pick_split_rb(const dflash_ctx *ctx, int n_blocks, int n_ct, int most, int ranges, int64_t *cost_of = nullptr) {
    int rb = 2;
    int64_t best = -1;
    for (int r = most; r >= 2; r--) {
        const int64_t tiles = static_cast<int64_t>(n_ct) * ((n_blocks + r - 1) / r);
        const int64_t n_split = std::min<int64_t>(ranges, ctx->n_cu / tiles);
        if (n_split < 2) continue;
        const int64_t cost = (ranges + n_split - 1) / n_split * (4 * r + 5);
        if (best < 0 || cost < best) {
            best = cost;
            rb = r;
        }
    }
    if (cost_of) *cost_of = best;
    return rb;
}

// What decides on a product's launch besides its rows: the most row blocks of a tile (a twin product has second accumulators) and the ranges K falls into.
int rows_most(const dfl_rows_plan &p) { return p.sums ? 8 : 4; }
int rows_columns(int64_t n_out, int64_t pair_ffn) { return static_cast<int>(pair_ffn ? pair_ffn / 128 : (n_out + 255) / 256); }
int rows_ranges(const dfl_rows_plan &p, int nb) {
    return p.by_group ? std::max(1, static_cast<int>(static_cast<int64_t>(nb) * p.n_cut / p.total)) : p.n_cut;
}

template <typename Tile, bool kTwin, int kEpi>
int32_t rows_dispatch(dflash_ctx *ctx, const RowsArgs &a, int rb, int64_t tiles, hipStream_t st) {
    switch (rb) {
        case 2: return rows_launch<Tile, kTwin, true, 2, kEpi, 0>(ctx, a, tiles, st);
        case 3: return rows_launch<Tile, kTwin, true, 3, kEpi, 0>(ctx, a, tiles, st);
        case 4: return rows_launch<Tile, kTwin, true, 4, kEpi, 0>(ctx, a, tiles, st);
        default: break;
    }
    if constexpr (!kTwin) {
        switch (rb) {
            case 5: return rows_launch<Tile, kTwin, true, 5, kEpi, 0>(ctx, a, tiles, st);
            case 6: return rows_launch<Tile, kTwin, true, 6, kEpi, 0>(ctx, a, tiles, st);
            case 7: return rows_launch<Tile, kTwin, true, 7, kEpi, 0>(ctx, a, tiles, st);
            case 8: return rows_launch<Tile, kTwin, true, 8, kEpi, 0>(ctx, a, tiles, st);
            default: break;
        }
    }
    return dfl_fail(ctx, DFLASH_ERR_UNSUPPORTED, "gemm_rows: %d row blocks per tile", rb);
}
}  // namespace

double dfl_gemm_rows_cost(const dflash_ctx *ctx, const dfl_rows_plan &p, int64_t n_in, int64_t n_out, int32_t n_rows, int64_t pair_ffn) {
    const int n_blocks = (n_rows + 15) / 16, n_ct = rows_columns(n_out, pair_ffn), nb = static_cast<int>(n_in / DFL_QK_K), ranges = rows_ranges(p, nb);
    if (n_blocks < 1 || n_ct < 1) return 0.0;
    const double twin = p.sums ? 1.0 : 2.0;  // (two MFMAs a product)
    int64_t cost = 0;
    const int rb = rows_pick_rb(ctx, n_blocks, n_ct, rows_most(p), &cost);
    if (!pair_ffn && ranges > 1 && 2ll * n_ct * ((n_blocks + rb - 1) / rb) <= ctx->n_cu) {
        rows_pick_split_rb(ctx, n_blocks, n_ct, rows_most(p), ranges, &cost);
        return twin * nb * static_cast<double>(cost) / ranges;
    }
    return twin * nb * static_cast<double>(cost);
}

int32_t dfl_gemm_rows(dflash_ctx *ctx, const dfl_rows_plan &p, int32_t w_type, const void *w, const void *xf, void *xs, bool make_sums, float *y,
                      int64_t n_in, int64_t n_out, int32_t n_rows, int64_t pair_ffn, void *y_xf, void *y_xs, int y_kind, hipStream_t st) {
    if (p.kind == DFL_XF_NONE || !w || !xf || n_rows < 1 || (p.sums && !xs) || (pair_ffn ? !y_xf : !y))
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
    a.n_ct = rows_columns(n_out, pair_ffn);
    const bool q6 = w_type == DFLASH_TYPE_Q6_K_TILED;
    const int most = rows_most(p);
    int rb = rows_pick_rb(ctx, a.n_blocks, a.n_ct, most);
    a.n_rt = (a.n_blocks + rb - 1) / rb;
    int64_t tiles = static_cast<int64_t>(a.n_ct) * a.n_rt;
    auto sums = [&]() -> int32_t { return p.sums && make_sums ? dfl_xf_sums(ctx, xf, n_in, a.n_blocks, xs, st) : DFLASH_OK; };
    if (pair_ffn) {
        if (const int32_t rc = sums()) return rc;
        return p.sums ? rows_dispatch<TileQ4, false, kEpiSwiglu>(ctx, a, rb, tiles, st) : rows_dispatch<TileQ4, true, kEpiSwiglu>(ctx, a, rb, tiles, st);
    }
    // Tiles for less than half the chip: K is shared by several workgroups, each range between two cuts on its own (as
    // many as there are at least in every tile group), where the workspace holds the partial products.
    const int ranges = rows_ranges(p, a.nb);
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
        // (the split of that table with tiles of two blocks; with the tiles it has now, 2048 -> 5120 and 4096 -> 2048 in Q6_K on
        // average, 7 / 9 / 12 blocks: 13.7 : 18.2, 17.2 : 19.7, 22.2 : 22.7, the same line)
        // so: twelve blocks for matrices of 80 super-blocks x column tiles or more, four for smaller ones, none where the
        // weights are not held.
        const int whole_most = a.nb * a.n_ct >= 80 ? 12 : 4;
        if (p.whole && a.n_blocks <= whole_most && dfl_whole_holds_weights(ctx, w_type, n_in, n_out))
            return dfl_gemm_whole_blocks(ctx, w_type, w, xf, y, n_in, n_out, n_rows, 0, nullptr, 0, st, true);
        size_t off = 0;
        float *part = dfl_ws_take<float>(ctx, &off, static_cast<size_t>(most_ranges) * a.n_blocks * 16 * n_out * sizeof(float));
        if (part) {
            rb = rows_pick_split_rb(ctx, a.n_blocks, a.n_ct, most, ranges);
            a.n_rt = (a.n_blocks + rb - 1) / rb;
            tiles = static_cast<int64_t>(a.n_ct) * a.n_rt;
            a.n_split = std::min<int>(ranges, static_cast<int>(ctx->n_cu / tiles));
            a.y = part;
            tiles *= a.n_split;
            int32_t rc = sums();
            if (!rc)
                rc = q6       ? rows_dispatch<TileQ6, true, kEpiSplit>(ctx, a, rb, tiles, st)
                     : p.sums ? rows_dispatch<TileQ4, false, kEpiSplit>(ctx, a, rb, tiles, st)
                              : rows_dispatch<TileQ4, true, kEpiSplit>(ctx, a, rb, tiles, st);
            if (rc) return rc;
            rows_reduce_kernel<<<dim3(static_cast<unsigned>((n_out + 1023) / 1024), n_rows), 256, 0, st>>>(a, part, y);
            DFL_HIP_CHECK(ctx, hipGetLastError());
            return DFLASH_OK;
        }
    }
    if (const int32_t rc = sums()) return rc;
    return q6       ? rows_dispatch<TileQ6, true, kEpiY>(ctx, a, rb, tiles, st)
           : p.sums ? rows_dispatch<TileQ4, false, kEpiY>(ctx, a, rb, tiles, st)
                    : rows_dispatch<TileQ4, true, kEpiY>(ctx, a, rb, tiles, st);
}

int32_t dfl_gemm_rows_experts(dflash_ctx *ctx, const void *w, const void *w_extra, const void *w_up, const void *w_up_extra, size_t w_stride,
                              const void *xf, const void *xs, const int32_t *tiles, const int32_t *n_tiles, int32_t max_tiles,
                              int32_t tile_blocks, float *y, int64_t n_in, int64_t n_out, void *y_xf, void *y_xs, hipStream_t st) {
    if (!w || !w_extra || !xf || !xs || !tiles || !n_tiles || max_tiles < 1 || n_in <= 0 || n_in % DFL_QK_K || n_out <= 0 || n_out % DFL_QK_K ||
        (w_up ? (!w_up_extra || !y_xf || !y_xs) : !y) || (tile_blocks != 4 && tile_blocks != 8) || ctx->lds_bytes < 160 * 1024)
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
    a.n_ct = static_cast<int>(n_out / ((w_up ? 16 : 32) * tile_blocks));  // (as many waves as a tile has row blocks at most)
    const int64_t tiles_max = static_cast<int64_t>(max_tiles) * a.n_ct;
    if (tile_blocks == 8)
        return w_up ? rows_launch<TileQ4, false, false, 8, kEpiSwiglu, 8>(ctx, a, tiles_max, st) : rows_launch<TileQ4, false, false, 8, kEpiY, 8>(ctx, a, tiles_max, st);
    return w_up ? rows_launch<TileQ4, false, false, 4, kEpiSwiglu, 4>(ctx, a, tiles_max, st) : rows_launch<TileQ4, false, false, 4, kEpiY, 4>(ctx, a, tiles_max, st);
}
