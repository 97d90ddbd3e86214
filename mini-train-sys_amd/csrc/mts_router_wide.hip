// The router projection of more than 16 experts: logits[t,e] = sum_h x[t,h] * w_r[e,h] with fp32 weights and fp32 sums, and
// its backward, on the fp32 matrix instruction; 16-bit activations are widened on their way into LDS, so there is no fp32
// copy of x and no cast of dx.  (Up to 16 experts the weights sit in LDS and the projection is a stream over x: see
// mts_router_linear.hip.)
//
// What bounds it: 2*T*H*E FLOP each way at the instruction's 157 TFLOP/s (7 us for 8192 x 1024 x 64, where x is 17 MB, 4 us),
// so what matters is that every SIMD has a share: forward, 32 rows x 64 experts per block with k dealt to its eight waves;
// dW_r, whose outputs fill 16 blocks only, the rows cut into chunks and the partial sums added in chunk order; dx in the same launch, so that
// the blocks of either fill the CUs that the other leaves.  Loads never depend on a branch (mts_f32_tiles.h).
// 8192 x 1024, 64 experts: 15.8 us forward, 29 + 5.5 backward; 22 and 19 + 17 + 6 with branches at the loads, four waves, 2-byte stores
// of dx and a launch each.  16 384 x 2048, 128 experts: 124 -> 95 and 210 -> 188.
//
// Backward of bf16 rows, from 1024 on (split_bwd_kernel): the fp32 operands as three bf16 terms each, which the bf16 instruction multiplies at 16 times the rate,
// three products for dW_r and six for dx.  Two waves a SIMD and what they wait for bound it then, so operands go from memory into fragments without
// LDS, except w_r's terms, which many rows share.  The launch and the sum of its partial dW_r, us: 8192 x 1024, 64 experts 35.3 -> 24.1; 8192 x 768, 24 23.7 -> 16.5;
// 16 384 x 2048, 128 173 -> 116, 32 experts 78 -> 43.  Error against fp64: dW_r 1.6e-7 (3.0e-7), 3.6e-7 (8.1e-7) at 16 384 x 2048, 128; dx its rounding.  The forward pass so
// split, fragments from memory: 14.6 -> 15.0 us and 83 -> 91 (32 experts 42 -> 38), as every 32 rows read and split w_r anew: not taken.  dW_r with three or four
// steps in flight 10.3 -> 13.7 and 15.0 us alone: more code than a short kernel can fetch.
#include "mts_cast_block.h"
#include "mts_f32_tiles.h"
#include "mts_router_row.h"
#include "mts_split3.h"

#include <type_traits>

namespace {

using namespace mts_f32;

constexpr int kThreads = 256, kLogitsThreads = 512;
constexpr int kBwdLds = 2 * (64 * 20 + 16 * 72);   // floats: the two buffers of dx

// bf16 activations: the fp32 operand as three bf16 terms (mts_split3.h), split in registers as they come from memory; x needs no splitting, so that three
// bf16 products make one that nothing is left out of.  The operand is split at a multiple of its size, a power of two that the sums are divided by at the end:
// down to the smallest numbers that there are, all terms are then ordinary ones, and what a product loses under the smallest number lies below the sum's own.
// Split as they come, values below 2^-60 had to be left to the fp32 instruction, and a softmax over logits 28 apart leaves such gradients behind a mean over
// 8192 tokens: both gradients of 8192 x 1024, 64 experts, took 81 us for 24 at logits of standard deviation 5 and 87 at 10 (16 384 x 2048, 128: 559 and 564 for
// 122); 24 and 124 at any now.  dW_r against fp64 there 1.55e-7 and 1.40e-7 (the fp32 instruction 1.96e-7 and 1.48e-7; 24 experts at 10: 1.81e-7 and 1.71e-7).
// Terms and products under 2^-126 are worth less than 2^-150 at 2^24 times their size.  Sums of fewer than 2^27 products below 2^100 stay in range: dlogits up
// to 2^36, weights up to 2^16 and rows up to 2^40; a gradient of a sum over wide rows passes 4, and one that is scaled passes 2^16.
constexpr float kScale = 0x1p24f;
constexpr uint16_t kLargestDl = 2 * ((127 + 60) << 7), kLargestOther = 2 * ((127 + 40) << 7);   // 2^60 and 2^40 in the order of sizes()
// two bf16 values without their signs, as numbers in the order of their size, infinities and NaN behind all others
__device__ __forceinline__ mts_split3::u16x2 sizes(uint32_t pair) { return __builtin_bit_cast(mts_split3::u16x2, pair) << 1; }
// in every lane of the wave
__device__ __forceinline__ bool below(mts_split3::u16x2 largest, uint16_t bound) { return !__ballot(max(largest[0], largest[1]) >= bound); }

struct Split8 {
    bf16x8 term[3];
    bool holds;   // every one of the scaled values is the sum of its terms, and sums of products stay in range, in every lane of the wave
};
__device__ __forceinline__ Split8 split8(const float (&value)[8], uint16_t bound) {
    Split8 s;
    float v[8];
    mts_split3::u16x2 largest = {};
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = value[j] * kScale;
#pragma unroll
    for (int q = 0; q < 3; ++q) {
        u32x4 h;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            h[i] = mts_split3::round2(v[2 * i], v[2 * i + 1]);
            if (q < 2) v[2 * i] -= __uint_as_float(h[i] << 16), v[2 * i + 1] -= __uint_as_float(h[i] & 0xffff0000u);
            if (q == 0) largest = __builtin_elementwise_max(largest, sizes(h[i]));
        }
        s.term[q] = __builtin_bit_cast(bf16x8, h);
    }
    s.holds = below(largest, bound);
    return s;
}

// 32 rows x 64 experts; wave w multiplies k-step w of every 64-wide k-tile, the eight sums meet in LDS.  Two waves of a SIMD: one reads its
// fragments while the other multiplies (four waves of two k-steps each: 19.9 us for 8192 x 1024 x 64 where this takes 15.8).
template <typename XT>
struct WideTile {
    static constexpr int BM = 32, BN = 64, TKS = 64, WAVES = kLogitsThreads / MTS_WAVE, STEPS = TKS / 8 / WAVES;
    typedef RowTile<XT, BM, TKS, true, kLogitsThreads> AT;
    typedef RowTile<float, BN, TKS, true, kLogitsThreads> BT;
    static constexpr int TILES = 2 * (AT::SIZE + BT::SIZE), SUMS = WAVES * BM * BN, LDS = TILES > SUMS ? TILES : SUMS;   // floats
    static_assert(BM * BN / 4 == kLogitsThreads, "four sums a thread");
    static __device__ __forceinline__ int row() { return threadIdx.x / (BN / 4); }
    static __device__ __forceinline__ int first_expert() { return threadIdx.x % (BN / 4) * 4; }

    // logits of row row0 + row(), experts e0 + first_expert() .. + 3
    static __device__ __forceinline__ f32x4 logits(const XT* __restrict__ x, const float* __restrict__ w, int64_t T, int H, int E, int64_t row0, int e0, float* lds) {
        float(*As)[AT::SIZE] = reinterpret_cast<float(*)[AT::SIZE]>(lds);
        float(*Bs)[BT::SIZE] = reinterpret_cast<float(*)[BT::SIZE]>(lds + 2 * AT::SIZE);
        AT a;
        BT b;
#pragma unroll
        for (int q = 0; q < AT::LOADS; ++q) {
            const int64_t r = row0 + AT::row(q);
            a.ptr[q] = x + (r < T ? r : T - 1) * H;
        }
#pragma unroll
        for (int q = 0; q < BT::LOADS; ++q) {
            const int e = e0 + BT::row(q);
            b.ptr[q] = w + (int64_t)(e < E ? e : E - 1) * H;
        }
        const int wave = threadIdx.x / MTS_WAVE, lane = threadIdx.x % MTS_WAVE;
        f32x16 acc[1][2] = {};
        auto fetch = [&](int set, int t) {
            a.fetch(set, t * TKS, H);
            b.fetch(set, t * TKS, H);
        };
        run_k_tiles<AT, BT, TKS, STEPS, 1, 2, true>(H, a, b, As, Bs, acc, [](int) { return 0; }, [](int nf) { return nf * 32; }, fetch, wave * STEPS);
        // a lane holds runs of four experts of row lane % 32; the groups of four of a row are dealt by the row
        const int ml = lane % 32;
        float* mine = lds + wave * BM * BN + ml * BN;
#pragma unroll
        for (int nf = 0; nf < 2; ++nf)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const f32x4 v = {acc[0][nf][4 * j], acc[0][nf][4 * j + 1], acc[0][nf][4 * j + 2], acc[0][nf][4 * j + 3]};
                *reinterpret_cast<f32x4*>(mine + (((nf * 8 + 2 * j + lane / 32) ^ (ml & 15)) << 2)) = v;
            }
        __syncthreads();
        const float* part = lds + row() * BN + ((first_expert() / 4 ^ (row() & 15)) << 2);
        f32x4 sum = *reinterpret_cast<const f32x4*>(part);
#pragma unroll
        for (int k = 1; k < WAVES; ++k) {   // in wave order
            const f32x4 v = *reinterpret_cast<const f32x4*>(part + k * BM * BN);
#pragma unroll
            for (int j = 0; j < 4; ++j) sum[j] += v[j];
        }
        return sum;
    }
    static __device__ __forceinline__ void store(f32x4 sum, float* __restrict__ logits, int64_t r, int64_t T, int E, int e) {
        if (r >= T) return;
        float* out = logits + r * E + e;
        if (E % 4 == 0) {
            if (e < E) *reinterpret_cast<f32x4*>(out) = sum;
        } else {
#pragma unroll
            for (int j = 0; j < 4; ++j)
                if (e + j < E) out[j] = sum[j];
        }
    }
};
template <typename XT>
__global__ __launch_bounds__(kLogitsThreads) void wide_logits_kernel(const XT* __restrict__ x, const float* __restrict__ w, int64_t T, int H, int E,
                                                                     float* __restrict__ logits) {
    typedef WideTile<XT> Tile;
    __shared__ __attribute__((aligned(16))) float lds[Tile::LDS];
    const int64_t row0 = (int64_t)blockIdx.x * Tile::BM;
    const int e0 = blockIdx.y * Tile::BN;
    const f32x4 sum = Tile::logits(x, w, T, H, E, row0, e0, lds);
    Tile::store(sum, logits, row0 + Tile::row(), T, E, e0 + Tile::first_expert());
}

// The same chained to the post-process, for up to 64 experts: a block holds all logits of its rows, so that its first waves go on with
// G lanes a row, as the post-process kernel does (the same results), and leave its routes per expert, which are the counters of the routing
// metadata's chunks.
template <typename XT, int G>
__global__ __launch_bounds__(kLogitsThreads) void wide_head_kernel(const XT* __restrict__ x, const float* __restrict__ w, int64_t T, int H, int E, int K, int normalize,
                                                                   float* __restrict__ logits, float* __restrict__ weights, int32_t* __restrict__ indices,
                                                                   void* __restrict__ weights_act, int act_dtype, float* __restrict__ partial,
                                                                   int32_t* __restrict__ partial_counts, int32_t* __restrict__ cnt, MtsCastJob copy) {
    using namespace mts_router;
    if constexpr (sizeof(XT) == 2) {
        if (blockIdx.x >= copy.own_blocks) return mts_cast::cast_block<XT, kLogitsThreads>(copy.cast, blockIdx.x - copy.own_blocks);
    }
    typedef WideTile<XT> Tile;
    constexpr int EP = 8, WAVES = Tile::BM * G / MTS_WAVE, LROW = 72;   // a row's lanes and the rows of a wave fall on different banks
    __shared__ __attribute__((aligned(16))) float lds[Tile::LDS];
    __shared__ __attribute__((aligned(16))) float rows[Tile::BM][LROW];
    __shared__ float red[WAVES][EP * G + 2];
    __shared__ int32_t cred[WAVES][EP * G];
    const int64_t row0 = (int64_t)blockIdx.x * Tile::BM;
    const f32x4 sum = Tile::logits(x, w, T, H, E, row0, 0, lds);
    *reinterpret_cast<f32x4*>(&rows[Tile::row()][Tile::first_expert()]) = sum;
    Tile::store(sum, logits, row0 + Tile::row(), T, E, Tile::first_expert());
    __syncthreads();
    const int wave = threadIdx.x / MTS_WAVE;
    if (wave < WAVES) {
        const int g = threadIdx.x % G, rl = threadIdx.x / G;
        RowState<EP, G> r;
#pragma unroll
        for (int j = 0; j < EP; ++j) r.l[j] = j * G + g < E ? rows[rl][j * G + g] : -INFINITY;
        softmax_row<EP, G>(r);
        RowTotals<EP, G> totals;
        totals.take(r, row0 + rl < T, row0 + rl, E, K, normalize, g, weights, indices, weights_act, act_dtype);
        totals.to_lds(red[wave], cred[wave]);
    }
    __syncthreads();
    const int i = threadIdx.x;
    if (i < E + 2) partial[(int64_t)blockIdx.x * (E + 2) + i] = block_column<EP, G, WAVES>(red, i, E);
    if (i < E) {
        int32_t v = 0;
#pragma unroll
        for (int k = 0; k < WAVES; ++k) v += cred[k][i];
        partial_counts[(int64_t)blockIdx.x * E + i] = v;
        cnt[(int64_t)blockIdx.x * E + i] = v;
    }
}

// dx[t,h] = sum_e dlogits[t,e] * w_r[e,h], 64 x 64 per block
template <typename XT, bool VEC>
__device__ __forceinline__ void wide_dx_block(const float* __restrict__ dl, const float* __restrict__ w, int64_t T, int H, int E, XT* __restrict__ dx,
                                              unsigned block, float* lds) {
    constexpr int BM = 64, BN = 64, TKS = 16;
    typedef RowTile<float, BM, TKS, VEC> AT;
    typedef KTile<float, BN, TKS, true> BT;
    constexpr int LDO = BN + 16 / (int)sizeof(XT), PER16 = 16 / (int)sizeof(XT);
    float(*As)[AT::SIZE] = reinterpret_cast<float(*)[AT::SIZE]>(lds);
    float(*Bs)[BT::SIZE] = reinterpret_cast<float(*)[BT::SIZE]>(lds + 2 * AT::SIZE);
    XT* staged = reinterpret_cast<XT*>(lds);
    static_assert(2 * (AT::SIZE + BT::SIZE) <= kBwdLds && BM * LDO * sizeof(XT) <= kBwdLds * sizeof(float), "LDS of a block");
    const int n_tiles = (H + BN - 1) / BN;
    const int64_t row0 = (int64_t)(block / n_tiles) * BM;
    const int n0 = block % n_tiles * BN;
    AT a;
    BT b;
#pragma unroll
    for (int q = 0; q < AT::LOADS; ++q) {
        const int64_t r = row0 + AT::row(q);
        a.ptr[q] = dl + (r < T ? r : T - 1) * E;
    }
    b.base = w + n0, b.ld = H, b.cols = H - n0;
    const int wave = threadIdx.x / MTS_WAVE, lane = threadIdx.x % MTS_WAVE, wm = wave / 2, wn = wave % 2;
    f32x16 acc[1][1] = {};
    auto fetch = [&](int set, int t) {
        a.fetch(set, t * TKS, E);
        int64_t rows[BT::LOADS];
#pragma unroll
        for (int q = 0; q < BT::LOADS; ++q) rows[q] = t * TKS + BT::k(q) < E ? t * TKS + BT::k(q) : E - 1;
        b.fetch(set, rows);
    };
    run_k_tiles<AT, BT, TKS, TKS / 8, 1, 1, true>(E, a, b, As, Bs, acc, [&](int) { return wm * 32; }, [&](int) { return wn * 32; }, fetch);
    // through LDS (the k loop ends with a barrier) into stores of 16 bytes
    typedef __attribute__((ext_vector_type(4))) XT quad;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const quad v = {(XT)acc[0][0][4 * j], (XT)acc[0][0][4 * j + 1], (XT)acc[0][0][4 * j + 2], (XT)acc[0][0][4 * j + 3]};
        *reinterpret_cast<quad*>(staged + (wm * 32 + lane % 32) * LDO + wn * 32 + 8 * j + 4 * (lane / 32)) = v;
    }
    __syncthreads();
#pragma unroll
    for (int i = threadIdx.x; i < BM * BN / PER16; i += kThreads) {
        const int m = i / (BN / PER16), c = i % (BN / PER16) * PER16;
        const int64_t r = row0 + m;
        if (r >= T || n0 + c >= H) continue;
        const XT* from = staged + m * LDO + c;
        XT* to = dx + r * H + n0 + c;
        if (H % PER16 == 0) *reinterpret_cast<u32x4*>(to) = *reinterpret_cast<const u32x4*>(from);
        else {   // rows start on four elements
            *reinterpret_cast<quad*>(to) = *reinterpret_cast<const quad*>(from);
            if (PER16 > 4 && n0 + c + 4 < H) *reinterpret_cast<quad*>(to + PER16 - 4) = *reinterpret_cast<const quad*>(from + PER16 - 4);
        }
    }
}

// partial dW_r[e,h] over one chunk of rows, 64 x 64 per block
template <typename XT, bool VEC>
__device__ __forceinline__ void wide_dw_block(const float* __restrict__ dl, const XT* __restrict__ x, int64_t T, int H, int E, int64_t rows_per_chunk,
                                              float* __restrict__ part, unsigned tile, unsigned chunk, float* lds) {
    constexpr int BM = 64, BN = 64, TKS = 16;
    typedef KTile<float, BM, TKS, VEC> PT;
    typedef KTile<XT, BN, TKS, true> QT;
    float(*Ps)[PT::SIZE] = reinterpret_cast<float(*)[PT::SIZE]>(lds);
    float(*Qs)[QT::SIZE] = reinterpret_cast<float(*)[QT::SIZE]>(lds + 2 * PT::SIZE);
    static_assert(2 * (PT::SIZE + QT::SIZE) <= kBwdLds, "LDS of a block");
    const unsigned n_tiles = (unsigned)((H + BN - 1) / BN);
    const int m0 = tile / n_tiles * BM, n0 = tile % n_tiles * BN;
    const int64_t r0 = (int64_t)chunk * rows_per_chunk, r1 = r0 + rows_per_chunk < T ? r0 + rows_per_chunk : T;
    PT a;
    QT b;
    a.base = dl + m0, a.ld = E, a.cols = E - m0;
    b.base = x + n0, b.ld = H, b.cols = H - n0;
    const int wave = threadIdx.x / MTS_WAVE, lane = threadIdx.x % MTS_WAVE, wm = wave / 2, wn = wave % 2;
    f32x16 acc[1][1] = {};
    auto fetch = [&](int set, int t) {
        int64_t pr[PT::LOADS], qr[QT::LOADS];
#pragma unroll
        for (int q = 0; q < PT::LOADS; ++q) pr[q] = r0 + t * TKS + PT::k(q) < r1 ? r0 + t * TKS + PT::k(q) : r1 - 1;
#pragma unroll
        for (int q = 0; q < QT::LOADS; ++q) qr[q] = r0 + t * TKS + QT::k(q) < r1 ? r0 + t * TKS + QT::k(q) : r1 - 1;
        a.fetch(set, pr);
        b.fetch(set, qr);
    };
    run_k_tiles<PT, QT, TKS, TKS / 8, 1, 1>((int)(r1 - r0), a, b, Ps, Qs, acc, [&](int) { return wm * 32; }, [&](int) { return wn * 32; }, fetch);
    float* out = part + (int64_t)chunk * E * H;
    const int n = n0 + wn * 32 + lane % 32;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const int m = m0 + wm * 32 + 8 * (i / 4) + 4 * (lane / 32) + i % 4;
        if (m < E && n < H) out[(int64_t)m * H + n] = acc[0][0][i];
    }
}

// Both gradients, the longer blocks of dW_r first.
template <typename XT, bool VEC>
__global__ __launch_bounds__(kThreads) void wide_bwd_kernel(const float* __restrict__ dl, const XT* __restrict__ x, const float* __restrict__ w, int64_t T, int H,
                                                            int E, int64_t rows_per_chunk, unsigned dw_tiles, unsigned chunks, XT* __restrict__ dx,
                                                            float* __restrict__ part) {
    __shared__ __attribute__((aligned(16))) float lds[kBwdLds];
    const unsigned dw_blocks = dw_tiles * chunks;
    if (blockIdx.x < dw_blocks) wide_dw_block<XT, VEC>(dl, x, T, H, E, rows_per_chunk, part, blockIdx.x % dw_tiles, blockIdx.x / dw_tiles, lds);
    else wide_dx_block<XT, VEC>(dl, w, T, H, E, dx, blockIdx.x - dw_blocks, lds);
}

// Both gradients for bf16 rows, up to 128 experts, on the split.
constexpr int kSplitCols = 128;   // columns of a dW_r block
constexpr int kSplitDwLds = 4 * 16 * MTS_WAVE * 4;   // floats: the sums of four waves

// partial dW_r over one chunk of rows, 32 experts x 128 columns per block, steps of 16 rows dealt to the waves.  A lane loads an expert and four columns of
// eight rows: with the columns of a fragment four apart these are the fragments, without LDS.  (64 experts a block would split and convert half as
// often, in more registers than there are.)
__device__ __forceinline__ void split_dw_block(const float* __restrict__ dl, const bf16_t* __restrict__ x, int64_t T, int H, int E, int64_t rows_per_chunk,
                                               float* __restrict__ part, unsigned tile, unsigned chunk, float* lds) {
    typedef __attribute__((ext_vector_type(2))) uint32_t Columns;
    const unsigned n_tiles = (unsigned)((H + kSplitCols - 1) / kSplitCols);
    const int wave = threadIdx.x / MTS_WAVE, lane = threadIdx.x % MTS_WAVE;
    const int e0 = (int)(tile / n_tiles) * 32, h = (int)(tile % n_tiles) * kSplitCols + lane % 32 * 4;
    const int64_t r0 = (int64_t)chunk * rows_per_chunk;
    const int rows = (int)(r0 + rows_per_chunk < T ? rows_per_chunk : T - r0), steps = (rows + 15) / 16;
    const float* dp = dl + r0 * E + min(e0 + lane % 32, E - 1);
    const bf16_t* xp = x + r0 * H + min(h, H - 4);
    float d[2][8];
    Columns c[2][8];
    auto fetch = [&](int set, int s) {
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const int64_t r = min(s * 16 + lane / 32 * 8 + j, rows - 1);
            d[set][j] = dp[r * E];
            c[set][j] = *reinterpret_cast<const Columns*>(xp + r * H);
        }
    };
    f32x16 acc[4] = {};
    auto multiply = [&](int set, int s) {   // false: not this step
        if (s * 16 + 16 > rows) {   // the last step: zeros on both sides
#pragma unroll
            for (int j = 0; j < 8; ++j)
                if (s * 16 + lane / 32 * 8 + j >= rows) d[set][j] = 0.f, c[set][j] = Columns{};
        }
        mts_split3::u16x2 largest = sizes(c[set][0][0]);
#pragma unroll
        for (int i = 1; i < 16; ++i) largest = __builtin_elementwise_max(largest, sizes(c[set][i / 2][i % 2]));
        bf16x8 xv[4];
#pragma unroll
        for (int p = 0; p < 4; ++p) {
            u32x4 u;
#pragma unroll
            for (int i = 0; i < 4; ++i) u[i] = __builtin_amdgcn_perm(c[set][2 * i + 1][p / 2], c[set][2 * i][p / 2], p % 2 ? 0x07060302u : 0x05040100u);
            xv[p] = __builtin_bit_cast(bf16x8, u);
        }
        const Split8 t = split8(d[set], kLargestDl);
        if (!below(largest, kLargestOther) || !t.holds) return false;
#pragma unroll
        for (int q = 2; q >= 0; --q)
#pragma unroll
            for (int p = 0; p < 4; ++p) acc[p] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(t.term[q], xv[p], acc[p], 0, 0, 0);
        return true;
    };
    int s = wave;
    if (s < steps) fetch(0, s);
    for (bool holds = true; holds && s < steps;) {
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            fetch(1 - u, s + 4);
            __builtin_amdgcn_sched_barrier(0);   // the loads stay in front
            if (!(holds = multiply(u, s)) || (s += 4) >= steps) break;
        }
    }
#pragma unroll
    for (int p = 0; p < 4; ++p) acc[p] *= 1.f / kScale;
#pragma unroll 1
    for (; s < steps; s += 4)   // from a step on that holds a value which is too large: by the fp32 instruction, whose k is lane / 32
#pragma unroll 1
        for (int j = 0; j < 8; ++j) {
            const int64_t r = s * 16 + lane / 32 * 8 + j;
            const bool in = r < rows;
            const float dv = in ? dp[r * E] : 0.f;
            const Columns cv = in ? *reinterpret_cast<const Columns*>(xp + r * H) : Columns{};
#pragma unroll
            for (int p = 0; p < 4; ++p) {
                const float xf = __uint_as_float(p % 2 ? cv[p / 2] & 0xffff0000u : cv[p / 2] << 16);
                acc[p] = __builtin_amdgcn_mfma_f32_32x32x2f32(dv, xf, acc[p], 0, 0, 0);
            }
        }
    // the waves' sums in wave order; wave w adds and stores rows 8w .. 8w + 7
    f32x4* sums = reinterpret_cast<f32x4*>(lds);
    float* out = part + (int64_t)chunk * E * H;
#pragma unroll
    for (int i = 0; i < 16; ++i) sums[(wave * 16 + i) * MTS_WAVE + lane] = f32x4{acc[0][i], acc[1][i], acc[2][i], acc[3][i]};
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        f32x4 v = sums[(4 * wave + i) * MTS_WAVE + lane];
#pragma unroll
        for (int k = 1; k < 4; ++k) v += sums[(k * 16 + 4 * wave + i) * MTS_WAVE + lane];
        const int m = e0 + 8 * wave + 4 * (lane / 32) + i;
        if (m < E && h < H) *reinterpret_cast<f32x4*>(out + (int64_t)m * H + h) = v;
    }
}

// dx: a block keeps the terms of w_r for COLS columns and all experts in LDS and takes 32 rows a wave at a time, whose dlogits are split in registers.  The
// columns of a fragment are dealt so that a lane ends with 16 consecutive ones.
template <int KS>
struct SplitDx {
    static constexpr int COLS = KS > 4 ? 64 : 128, LD = KS * 16 + 8, PLANE = COLS * LD;   // bf16; rows of 16 bytes more than a multiple of 64: reads of eight lanes on all banks
    static constexpr int LDS = 3 * PLANE / 2 + 4;   // floats, and the flag
    static constexpr int column(int m) { return 16 * (m >> 2 & 1) + 4 * (m >> 3) + (m & 3); }

    static __device__ __forceinline__ void block(const float* __restrict__ dl, const float* __restrict__ w, int64_t T, int H, int E, bf16_t* __restrict__ dx, unsigned block,
                                                 unsigned row_blocks, float* lds) {
        bf16_t* terms = reinterpret_cast<bf16_t*>(lds);
        int* special = reinterpret_cast<int*>(lds + 3 * PLANE / 2);
        const int n_tiles = (H + COLS - 1) / COLS, n0 = (int)(block % n_tiles) * COLS;
        const int wave = threadIdx.x / MTS_WAVE, lane = threadIdx.x % MTS_WAVE;
        if (threadIdx.x == 0) *special = 0;
        const int64_t step = (int64_t)row_blocks * 128;
        int64_t row0 = ((int64_t)(block / n_tiles) * 4 + wave) * 32;
        f32x4 raw[KS][2];
        auto fetch = [&](int64_t r) {
            const float* dp = dl + (r < T ? r : T - 1) * E;
#pragma unroll
            for (int s = 0; s < KS; ++s)
#pragma unroll
                for (int h = 0; h < 2; ++h) raw[s][h] = *reinterpret_cast<const f32x4*>(dp + min(16 * s + lane / 32 * 8, E - 8) + 4 * h);
        };
        fetch(row0 + lane % 32);
        constexpr int PIECES = COLS * KS * 2 / kThreads;   // eight experts of a column
        float v[PIECES][8];
#pragma unroll
        for (int i = 0; i < PIECES; ++i) {
            const int at = i * kThreads + threadIdx.x, col = min(n0 + at % COLS, H - 1);
#pragma unroll
            for (int j = 0; j < 8; ++j) v[i][j] = w[(int64_t)min(at / COLS * 8 + j, E - 1) * H + col];
        }
        __builtin_amdgcn_sched_barrier(0);   // the loads stay together in front
        __syncthreads();
        bool holds = true;
#pragma unroll
        for (int i = 0; i < PIECES; ++i) {
            const int at = i * kThreads + threadIdx.x, c = at % COLS, k0 = at / COLS * 8;
            if (k0 >= E) {
#pragma unroll
                for (int j = 0; j < 8; ++j) v[i][j] = 0.f;
            }
            const Split8 s = split8(v[i], kLargestOther);
            holds &= s.holds;
#pragma unroll
            for (int q = 0; q < 3; ++q) *reinterpret_cast<bf16x8*>(terms + q * PLANE + c * LD + k0) = s.term[q];
        }
        if (!holds && lane == 0) *special = 1;
        __syncthreads();
        const bool plain = *special == 0;
        const int cm = column(lane % 32);
        for (; row0 < T; row0 += step) {
            const int64_t r = row0 + lane % 32;
            const float* dp = dl + (r < T ? r : T - 1) * E;
            Split8 d[KS];
            bool all = plain;
#pragma unroll
            for (int s = 0; s < KS; ++s) {
                float v[8];
#pragma unroll
                for (int j = 0; j < 8; ++j) v[j] = 16 * s + lane / 32 * 8 < E ? raw[s][j / 4][j % 4] : 0.f;
                d[s] = split8(v, kLargestDl);
                all &= d[s].holds;
            }
            fetch(r + step);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int nf = 0; nf < COLS / 32; ++nf) {
                f32x16 acc = {};
                if (all) {
#pragma unroll
                    for (int s = 0; s < KS; ++s) {
                        bf16x8 a[3];
#pragma unroll
                        for (int q = 0; q < 3; ++q) a[q] = *reinterpret_cast<const bf16x8*>(terms + q * PLANE + (nf * 32 + cm) * LD + 16 * s + lane / 32 * 8);
                        constexpr int kTerms[6][2] = {{2, 0}, {0, 2}, {1, 1}, {1, 0}, {0, 1}, {0, 0}};   // small ones first
#pragma unroll
                        for (int t = 0; t < 6; ++t) acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[kTerms[t][0]], d[s].term[kTerms[t][1]], acc, 0, 0, 0);
                    }
                    acc *= 1.f / kScale / kScale;
                } else {   // by the fp32 instruction, whose k is lane / 32
                    const float* wp = w + min(n0 + nf * 32 + cm, H - 1);
#pragma unroll 1
                    for (int k = lane / 32; k < (E + 1) / 2 * 2; k += 2)
                        acc = __builtin_amdgcn_mfma_f32_32x32x2f32(k < E ? wp[(int64_t)k * H] : 0.f, k < E ? dp[k] : 0.f, acc, 0, 0, 0);
                }
                const int h = n0 + nf * 32 + 16 * (lane / 32);
#pragma unroll
                for (int g = 0; g < 2; ++g) {
                    bf16x8 v;
#pragma unroll
                    for (int j = 0; j < 8; ++j) v[j] = (bf16_t)acc[8 * g + j];
                    if (r < T && h + 8 * g < H) *reinterpret_cast<bf16x8*>(dx + r * H + h + 8 * g) = v;
                }
            }
        }
    }
};

// KS: steps of 16 experts
template <int KS>
__global__ __launch_bounds__(kThreads, 2) void split_bwd_kernel(const float* __restrict__ dl, const bf16_t* __restrict__ x, const float* __restrict__ w, int64_t T, int H,
                                                                int E, int64_t rows_per_chunk, unsigned dw_tiles, unsigned chunks, unsigned row_blocks,
                                                                bf16_t* __restrict__ dx, float* __restrict__ part) {
    constexpr int LDS = SplitDx<KS>::LDS > kSplitDwLds ? SplitDx<KS>::LDS : kSplitDwLds;
    __shared__ __attribute__((aligned(16))) float lds[LDS];
    const unsigned dw_blocks = dw_tiles * chunks;
    if (blockIdx.x < dw_blocks) split_dw_block(dl, x, T, H, E, rows_per_chunk, part, blockIdx.x % dw_tiles, blockIdx.x / dw_tiles, lds);
    else SplitDx<KS>::block(dl, w, T, H, E, dx, blockIdx.x - dw_blocks, row_blocks, lds);
}

// Whole pieces of eight experts and columns are what the loads take, and the terms of more than 128 experts do not fit.  Fewer rows leave the blocks a chain
// of latencies either way: 256 of 768 and 24 experts 4.8 us / 4.8 here, 613 and 32 experts 5.2 / 5.6, 993 and 24 5.8 / 5.6; 2048 of 1024 and 64 13.9 / 8.7.
bool split_bwd_takes(int64_t T, int H, int E, int act_dtype) {
    return act_dtype == MTS_BF16 && H % 8 == 0 && E % 8 == 0 && E <= 128 && T >= 1024;
}
struct SplitGrid {
    int64_t rows;
    unsigned dw_tiles, chunks, col_tiles, row_blocks;
};
// A block of each kind per CU; chunks of 128 rows or more.
SplitGrid split_grid(int64_t T, int H, int E) {
    SplitGrid g;
    g.dw_tiles = (unsigned)((E + 31) / 32 * ((H + kSplitCols - 1) / kSplitCols));
    int64_t count = (256 + g.dw_tiles - 1) / g.dw_tiles;
    const int64_t most = (T + 127) / 128;
    if (count > most) count = most;
    g.rows = ((T + count - 1) / count + 15) / 16 * 16;
    g.chunks = (unsigned)((T + g.rows - 1) / g.rows);
    const int cols = E > 64 ? SplitDx<8>::COLS : SplitDx<4>::COLS;
    g.col_tiles = (unsigned)((H + cols - 1) / cols);
    const int64_t want = (256 + g.col_tiles - 1) / g.col_tiles, need = (T + 127) / 128;
    g.row_blocks = (unsigned)(want < need ? want : need);
    return g;
}

// Rows are cut into as many chunks as make about two blocks per CU, of at least 64 rows.
struct WideChunks {
    int64_t rows;
    int count;
};
WideChunks wide_chunks(int64_t T, int H, int E) {
    const int64_t tiles = (int64_t)((E + 63) / 64) * ((H + 63) / 64);
    int64_t count = (512 + tiles - 1) / tiles;
    const int64_t most = (T + 63) / 64;
    if (count > most) count = most;
    const int64_t rows = ((T + count - 1) / count + 15) / 16 * 16;
    return {rows, (int)((T + rows - 1) / rows)};
}

int wide_check(const void* x, const float* w_r, int64_t T, int H, int E, int act_dtype) {
    if (!x || !w_r) return MTS_ERR_NULL;
    if (!mts_router_wide_supported(H, E) || T <= 0 || (T + 63) / 64 * ((H + 63) / 64) >= (1LL << 31) - (1 << 20)) return MTS_ERR_SHAPE;
    if (act_dtype != MTS_BF16 && act_dtype != MTS_F16 && act_dtype != MTS_F32) return MTS_ERR_DTYPE;
    if (!mts_aligned16(x) || !mts_aligned16(w_r)) return MTS_ERR_ALIGN;
    return MTS_OK;
}

}  // namespace

extern "C" int mts_router_wide_supported(int H, int E) { return H >= 4 && H % 4 == 0 && E >= 1 && E <= MTS_MAX_EXPERTS ? 1 : 0; }

extern "C" int mts_router_wide_fwd(const void* x, const float* w_r, int64_t T, int H, int E, int act_dtype, float* logits, void* stream) {
    const int rc = wide_check(x, w_r, T, H, E, act_dtype);
    if (rc) return rc;
    if (!logits) return MTS_ERR_NULL;
    const dim3 grid((unsigned)((T + 31) / 32), (unsigned)((E + 63) / 64));
    hipStream_t s = (hipStream_t)stream;
    if (act_dtype == MTS_BF16) wide_logits_kernel<bf16_t><<<grid, kLogitsThreads, 0, s>>>((const bf16_t*)x, w_r, T, H, E, logits);
    else if (act_dtype == MTS_F16) wide_logits_kernel<mts_f16_t><<<grid, kLogitsThreads, 0, s>>>((const mts_f16_t*)x, w_r, T, H, E, logits);
    else wide_logits_kernel<float><<<grid, kLogitsThreads, 0, s>>>((const float*)x, w_r, T, H, E, logits);
    MTS_CHECK_LAUNCH();
    return MTS_OK;
}

int mts_launch_wide_head(const void* x, const float* w_r, int64_t T, int H, int E, int K, int normalize, int act_dtype, float* logits, float* weights, int32_t* indices,
                         void* weights_act, float* partial, int32_t* partial_counts, int32_t* cnt, const MtsCast* cast, hipStream_t s) {
    const int rc = wide_check(x, w_r, T, H, E, act_dtype);
    if (rc) return rc;
    if (!logits || !weights || !indices) return MTS_ERR_NULL;
    if (E > 64 || K < 1 || K > E || K > MTS_MAX_TOP_K) return MTS_ERR_SHAPE;
    if (!mts_aligned16(logits)) return MTS_ERR_ALIGN;
    const unsigned blocks = (unsigned)((T + MTS_WIDE_HEAD_ROWS - 1) / MTS_WIDE_HEAD_ROWS);
    const dim3 grid((unsigned)(blocks + mts_cast::blocks(cast, kLogitsThreads)));
    const MtsCastJob copy = mts_cast::job(cast, blocks);
    auto launch = [&](auto* kind) {
        typedef typename std::remove_pointer<decltype(kind)>::type XT;
        static_assert(WideTile<XT>::BM == MTS_WIDE_HEAD_ROWS, "rows of a chunk");
        // as many lanes a row as the post-process kernel takes for as many experts
        if (E > 32) wide_head_kernel<XT, 8><<<grid, kLogitsThreads, 0, s>>>((const XT*)x, w_r, T, H, E, K, normalize, logits, weights, indices, weights_act, act_dtype, partial, partial_counts, cnt, copy);
        else wide_head_kernel<XT, 4><<<grid, kLogitsThreads, 0, s>>>((const XT*)x, w_r, T, H, E, K, normalize, logits, weights, indices, weights_act, act_dtype, partial, partial_counts, cnt, copy);
    };
    if (act_dtype == MTS_BF16) launch((bf16_t*)nullptr);
    else if (act_dtype == MTS_F16) launch((mts_f16_t*)nullptr);
    else launch((float*)nullptr);
    MTS_CHECK_LAUNCH();
    return MTS_OK;
}

extern "C" int64_t mts_router_wide_bwd_workspace_bytes(int64_t T, int H, int E) {
    if (T <= 0 || H <= 0 || E <= 0) return 0;
    const int64_t chunks = wide_chunks(T, H, E).count, split = split_bwd_takes(T, H, E, MTS_BF16) ? split_grid(T, H, E).chunks : 0;
    return (chunks > split ? chunks : split) * E * H * (int64_t)sizeof(float);
}

extern "C" int mts_router_wide_bwd(const float* dlogits, const void* x, const float* w_r, int64_t T, int H, int E, int act_dtype, void* dx,
                                   float* d_w_r, void* workspace, int64_t workspace_bytes, void* stream) {
    const int rc = wide_check(x, w_r, T, H, E, act_dtype);
    if (rc) return rc;
    if (!dlogits || !dx || !d_w_r || !workspace) return MTS_ERR_NULL;
    if (workspace_bytes < mts_router_wide_bwd_workspace_bytes(T, H, E)) return MTS_ERR_WORKSPACE;
    if (!mts_aligned16(dlogits) || !mts_aligned16(dx) || !mts_aligned16(d_w_r) || !mts_aligned16(workspace)) return MTS_ERR_ALIGN;
    hipStream_t s = (hipStream_t)stream;
    if (split_bwd_takes(T, H, E, act_dtype)) {
        const SplitGrid g = split_grid(T, H, E);
        const unsigned blocks = g.dw_tiles * g.chunks + g.col_tiles * g.row_blocks;
        auto launch = [&](auto steps) {
            split_bwd_kernel<decltype(steps)::value><<<blocks, kThreads, 0, s>>>(dlogits, (const bf16_t*)x, w_r, T, H, E, g.rows, g.dw_tiles, g.chunks, g.row_blocks,
                                                                                 (bf16_t*)dx, (float*)workspace);
        };
        if (E <= 32) launch(std::integral_constant<int, 2>());
        else if (E <= 64) launch(std::integral_constant<int, 4>());
        else launch(std::integral_constant<int, 8>());
        MTS_CHECK_LAUNCH();
        return mts_launch_router_dw_reduce((const float*)workspace, (int)g.chunks, (int64_t)E * H, d_w_r, s);
    }
    const bool vec = E % 4 == 0;
    const WideChunks c = wide_chunks(T, H, E);
    const unsigned dw_tiles = (unsigned)((H + 63) / 64 * ((E + 63) / 64));
    const dim3 grid((unsigned)(dw_tiles * c.count + (T + 63) / 64 * ((H + 63) / 64)));
    float* part = (float*)workspace;
    auto launch = [&](auto* kind) {
        typedef typename std::remove_pointer<decltype(kind)>::type XT;
        if (vec) wide_bwd_kernel<XT, true><<<grid, kThreads, 0, s>>>(dlogits, (const XT*)x, w_r, T, H, E, c.rows, dw_tiles, (unsigned)c.count, (XT*)dx, part);
        else wide_bwd_kernel<XT, false><<<grid, kThreads, 0, s>>>(dlogits, (const XT*)x, w_r, T, H, E, c.rows, dw_tiles, (unsigned)c.count, (XT*)dx, part);
    };
    if (act_dtype == MTS_BF16) launch((bf16_t*)nullptr);
    else if (act_dtype == MTS_F16) launch((mts_f16_t*)nullptr);
    else launch((float*)nullptr);
    MTS_CHECK_LAUNCH();
    return mts_launch_router_dw_reduce(part, c.count, (int64_t)E * H, d_w_r, s);
}
