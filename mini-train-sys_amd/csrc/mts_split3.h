// Tiles of fp32 products on the bf16 matrix instruction (v_mfma_f32_32x32x16_bf16): loaders that split fp32 values into three
// bf16 planes on their way into LDS, fragment reads and the k loop of a block of four waves.
//
// x0 = bf16(x), x1 = bf16(x - x0), x2 = x - x0 - x1, each rounded to nearest: the differences are exact, x1 is at most 2^-9 of x
// and x2 at most 2^-18, and x2 fits 8 bits, so x = x0 + x1 + x2 (the splitting of Henry, Tang and Heinecke, "Leveraging the bfloat16
// Artificial Intelligence Datatype For Higher-Precision Computations", 2019).  Values in [2^-60, 2^50) and zero are split so.  Below, a
// product could lose bits under the smallest number there is; above, a sum could leave the range of fp32 where the values' own does
// not, because x0 may be rounded up: sums of fewer than 2^27 products below 2^100 cannot.  Any other value goes into the planes as its
// own bits with a marker, and its k-tile and the ones behind it are multiplied by the fp32 instruction from the values put together again.
#pragma once

#include "mts_common.h"

namespace mts_split3 {

constexpr int kLoaders = 256;            // threads that load and split: the second half of a block
constexpr int kThreads = 2 * kLoaders;
constexpr int TK = 16;                   // k extent of an LDS tile
constexpr int kDepth = 2;                // k-tiles in flight in registers, and LDS tiles

typedef volatile __attribute__((address_space(3))) int LdsWord;

constexpr uint32_t kSmallest = 0x21800000u;   // 2^-60
constexpr uint32_t kBeyond = 0x58800000u;     // 2^50
constexpr uint32_t kMarker = 0x7fffu;         // third plane of a value kept as its bits: a NaN, which no split gives

// Sums of so few terms are left to the fp32 instruction, which rounds once for each: six bf16 products a term and the three left out come to more
// than that.  Relative error against fp64 (norm, and the worst of 512 x 512 sums over the sum of the terms' sizes), fp32 instruction / six products:
// 1 term 2.5e-8 / 3.5e-8, 0.6e-7 / 1.5e-7; 2 terms 3.1e-8 / 3.3e-8, 1.1e-7 / 1.2e-7; 3 terms 3.6e-8 / 3.3e-8, 1.5e-7 / 1.2e-7; 16 terms 7.4e-8 / 3.4e-8,
// 2.3e-7 / 1.0e-7; 17 terms (the second k-tile) 7.5e-8 / 6.3e-8, 2.2e-7 / 2.1e-7; 1024 terms 5.7e-7 / 4.9e-7, 2.5e-7 / 2.4e-7.  All nine products: 1 term
// 3.4e-8, 1.2e-7, and a fifth more time.
constexpr int kFewTerms = 2;

// The loads of the loops below are unconditional: a load that a lane or a pass may skip makes the compiler wait for all loads in flight at the
// next use of any.  What lies outside an operand is read from its last element instead, and set to zero where it would be added.

// elements p[first .. first + 3] of `count` (VEC: both are multiples of four, and p is aligned to four elements)
template <bool VEC>
__device__ __forceinline__ f32x4 load4(const float* p, int first, int count) {
    if constexpr (VEC) return *reinterpret_cast<const f32x4*>(p + (first < count ? first : count - 4));
    f32x4 v;
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] = p[first + j < count ? first + j : count - 1];
    return v;
}

typedef __attribute__((ext_vector_type(2))) uint16_t u16x2;

__device__ __forceinline__ bool splits_exactly(float x) {
    const uint32_t u = __float_as_uint(x) & 0x7fffffffu;
    return (u >= kSmallest && u < kBeyond) || u == 0;
}
// The first plane as numbers that order a value by its size, from the smallest that splits on: kRange and above where one does not
// (zero among them: whoever asks looks again).
constexpr uint16_t kRange = (uint16_t)((kBeyond - kSmallest) >> 15);
__device__ __forceinline__ u16x2 range_keys(uint32_t pair) {
    const uint32_t two = 0x00020002u, shift = 0x00010001u * (uint16_t)(0u - (kSmallest >> 15));
    uint32_t key;
    asm("v_pk_mad_u16 %0, %1, %2, %3" : "=v"(key) : "v"(pair), "s"(two), "v"(shift));   // 2 * bits - smallest
    return __builtin_bit_cast(u16x2, key);
}

// two values rounded to bf16, in one register (from a conversion of its own the compiler would make one more for every half taken out)
__device__ __forceinline__ uint32_t round2(float a, float b) {
    uint32_t h;
    asm("v_cvt_pk_bf16_f32 %0, %1, %2" : "=v"(h) : "v"(a), "v"(b));
    return h;
}
__device__ __forceinline__ u16x2 store_planes(f32x4 v, bf16_t* at, int plane) {
    u16x2 keys = {};
#pragma unroll
    for (int q = 0; q < 3; ++q) {
        const uint2 h = {round2(v[0], v[1]), round2(v[2], v[3])};
        *reinterpret_cast<uint2*>(at + q * plane) = h;
        if (q == 0) keys = __builtin_elementwise_max(range_keys(h.x), range_keys(h.y));
        if (q < 2) v -= f32x4{__uint_as_float(h.x << 16), __uint_as_float(h.x & 0xffff0000u), __uint_as_float(h.y << 16), __uint_as_float(h.y & 0xffff0000u)};
    }
    return keys;
}
// the pairs of values of which the split does not hold one, over what store_planes wrote
__device__ __forceinline__ bool store_bits(f32x4 v, bf16_t* at, int plane) {
    bool any = false;
#pragma unroll
    for (int j = 0; j < 4; j += 2)
        if (!splits_exactly(v[j]) || !splits_exactly(v[j + 1])) {
            const uint32_t a = __float_as_uint(v[j]), b = __float_as_uint(v[j + 1]);
            *reinterpret_cast<uint32_t*>(at + j) = a >> 16 | (b & 0xffff0000u);
            *reinterpret_cast<uint32_t*>(at + plane + j) = (a & 0xffffu) | b << 16;
            *reinterpret_cast<uint32_t*>(at + 2 * plane + j) = kMarker * 0x10001u;
            any = true;
        }
    return any;
}
__device__ __forceinline__ float put_together(const bf16_t* at, int plane) {
    const uint32_t b0 = __builtin_bit_cast(uint16_t, at[0]), b1 = __builtin_bit_cast(uint16_t, at[plane]), b2 = __builtin_bit_cast(uint16_t, at[2 * plane]);
    const float sum = bf16_bits_to_f32(b0) + (bf16_bits_to_f32(b1) + bf16_bits_to_f32(b2));
    return b2 == kMarker ? __uint_as_float(b0 << 16 | b1) : sum;
}

// what both kinds of tile do with the values of a k-tile: true where one of them is kept as its bits
template <int LOADS, class At>
__device__ __forceinline__ bool commit_planes(const f32x4 (&reg)[LOADS], bf16_t* lds, int plane, At at) {
    u16x2 keys = {};
#pragma unroll
    for (int p = 0; p < LOADS; ++p) keys = __builtin_elementwise_max(keys, store_planes(reg[p], lds + at(p), plane));
    const uint16_t key = max(keys[0], keys[1]);
    bool any = false;
    if (__ballot(key >= kRange)) {
#pragma unroll
        for (int p = 0; p < LOADS; ++p) any |= store_bits(reg[p], lds + at(p), plane);
    }
    return any;
}

// [ROWS][TK] tile of k-contiguous rows.  A row is 32 bytes of a plane; its two 16-byte chunks change places every eight rows, so that
// the fragment reads of a wave (32 rows, one chunk each) meet every bank equally often.
template <int ROWS, bool VEC>
struct RowPlanes {
    static constexpr int TPR = TK / 4, LOADS = ROWS * TPR / kLoaders, PLANE = ROWS * TK, SIZE = 3 * PLANE;
    const float* ptr[LOADS];   // this thread's rows
    f32x4 reg[kDepth][LOADS];
    __device__ __forceinline__ static int thread() { return threadIdx.x % kLoaders; }
    __device__ __forceinline__ static int row(int p) { return thread() / TPR + p * (kLoaders / TPR); }
    __device__ __forceinline__ void fetch(int set, int k0, int Kdim) {
#pragma unroll
        for (int p = 0; p < LOADS; ++p) reg[set][p] = load4<VEC>(ptr[p], k0 + thread() % TPR * 4, Kdim);
    }
    // the first `count` of the tile's k are added
    __device__ __forceinline__ bool commit(int set, bf16_t* lds, int count) {
        if (count < TK) {
#pragma unroll
            for (int p = 0; p < LOADS; ++p)
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    if (thread() % TPR * 4 + j >= count) reg[set][p][j] = 0.f;
        }
        return commit_planes(reg[set], lds, PLANE, [&](int p) { return at(row(p), thread() % TPR * 4); });
    }
    __device__ __forceinline__ static int at(int r, int k) { return r * TK + (((k / 8) ^ (r >> 3 & 1)) << 3) + k % 8; }
    // k = 8 * (lane / 32) + 0..7 of row `r0 + lane % 32`
    __device__ __forceinline__ static bf16x8 frag(const bf16_t* plane, int r0) {
        const int lane = threadIdx.x % MTS_WAVE, r = r0 + lane % 32;
        return *reinterpret_cast<const bf16x8*>(plane + at(r, lane / 32 * 8));
    }
};

// [TK][COLS] tile of k-major rows, read with the transposing LDS load: within 16 lanes, lane l addresses four columns of
// row l / 4 and receives four rows of column l.  The chunks of a row are dealt so that four neighbouring rows, which such a group
// reads together, lie in different banks.
template <int COLS, bool VEC>
struct KPlanes {
    static constexpr int PER_ROW = COLS / 4, LOADS = COLS * TK / 4 / kLoaders, PLANE = TK * COLS, SIZE = 3 * PLANE;
    static_assert(COLS == 64 || COLS == 128, "the deal of the chunks");
    const float* base;       // element (k = 0, the tile's first column)
    int64_t ld;
    int cols;                // columns from there on that exist
    f32x4 reg[kDepth][LOADS];
    __device__ __forceinline__ static int thread() { return threadIdx.x % kLoaders; }
    __device__ __forceinline__ static int deal(int k) { return COLS == 128 ? (k & 3) << 2 : (k >> 1 & 1) << 2; }
    __device__ __forceinline__ static int k(int p) { return thread() / PER_ROW + p * (kLoaders / PER_ROW); }
    __device__ __forceinline__ static int col() { return (thread() % PER_ROW) * 4; }
    // rows[p] = memory row of k-row k(p)
    __device__ __forceinline__ void fetch(int set, const int64_t (&rows)[LOADS]) {
#pragma unroll
        for (int p = 0; p < LOADS; ++p) reg[set][p] = load4<VEC>(base + rows[p] * ld, col(), cols);
    }
    __device__ __forceinline__ bool commit(int set, bf16_t* lds, int count) {
        if (count < TK) {
#pragma unroll
            for (int p = 0; p < LOADS; ++p)
                if (k(p) >= count) reg[set][p] = f32x4{};
        }
        return commit_planes(reg[set], lds, PLANE, [&](int p) { return at(col(), k(p)); });
    }
    __device__ __forceinline__ static int at(int c, int k) { return k * COLS + (((c / 8) ^ deal(k)) << 3) + c % 8; }
    // k = 8 * (lane / 32) + 0..7 of column `c0 + lane % 32`
    __device__ __forceinline__ static bf16x8 frag(const bf16_t* plane, int c0) {
        typedef __attribute__((ext_vector_type(4))) short s16x4;
        typedef __attribute__((ext_vector_type(8))) short s16x8;
        const int lane = threadIdx.x % MTS_WAVE, c = c0 + 16 * (lane / 16 % 2) + 4 * (lane % 4);
        s16x4 h[2];
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            const int r = 8 * (lane / 32) + 4 * q + lane % 16 / 4;
            const bf16_t* src = plane + at(c, r);
            h[q] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)(src));
        }
        const s16x8 v = {h[0][0], h[0][1], h[0][2], h[0][3], h[1][0], h[1][1], h[1][2], h[1][3]};
        return __builtin_bit_cast(bf16x8, v);
    }
};

// one k-tile: MF x NF fragments of 32x32 per wave; a_at / b_at give the first row / column of a fragment in the tile
template <class AT, class BT, int MF, int NF, class AAt, class BAt>
__device__ __forceinline__ void mma_tile(const bf16_t* As, const bf16_t* Bs, f32x16 (&acc)[MF][NF], AAt a_at, BAt b_at) {
    bf16x8 b[NF][3];
#pragma unroll
    for (int nf = 0; nf < NF; ++nf)
#pragma unroll
        for (int q = 0; q < 3; ++q) b[nf][q] = BT::frag(Bs + q * BT::PLANE, b_at(nf));
#pragma unroll
    for (int mf = 0; mf < MF; ++mf) {
        bf16x8 a[3];
#pragma unroll
        for (int q = 0; q < 3; ++q) a[q] = AT::frag(As + q * AT::PLANE, a_at(mf));
        constexpr int kTerms[6][2] = {{2, 0}, {0, 2}, {1, 1}, {1, 0}, {0, 1}, {0, 0}};   // small ones first
#pragma unroll
        for (int t = 0; t < 6; ++t)
#pragma unroll
            for (int nf = 0; nf < NF; ++nf)
                acc[mf][nf] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[kTerms[t][0]], b[nf][kTerms[t][1]], acc[mf][nf], 0, 0, 0);
    }
}

// the same by the fp32 instruction, whose k is lane / 32
template <class AT, class BT, int MF, int NF, class AAt, class BAt>
__device__ __forceinline__ void mma_tile_f32(const bf16_t* As, const bf16_t* Bs, f32x16 (&acc)[MF][NF], AAt a_at, BAt b_at) {
    const int lane = threadIdx.x % MTS_WAVE;
#pragma unroll 1
    for (int k = lane / 32; k < TK; k += 2) {
        float b[NF];
#pragma unroll
        for (int nf = 0; nf < NF; ++nf) b[nf] = put_together(Bs + BT::at(b_at(nf) + lane % 32, k), BT::PLANE);
#pragma unroll
        for (int mf = 0; mf < MF; ++mf) {
            const float a = put_together(As + AT::at(a_at(mf) + lane % 32, k), AT::PLANE);
#pragma unroll
            for (int nf = 0; nf < NF; ++nf) acc[mf][nf] = __builtin_amdgcn_mfma_f32_32x32x2f32(a, b[nf], acc[mf][nf], 0, 0, 0);
        }
    }
}

// The k loop, through two LDS tiles: the second half of the block loads and splits k-tile t + 1 while the first half multiplies
// k-tile t.  fetch(set, t) starts the loads of k-tile t into a register set; it is called for every t in order, and for the last
// one again behind that.  special: a word of
// LDS, the first k-tile (counted from 1) that holds a value the split does not.
template <class AT, class BT, class Fetch>
__device__ __forceinline__ void load_k_tiles(int Kdim, AT& a, BT& b, bf16_t* As, bf16_t* Bs, LdsWord* special, Fetch fetch) {
    const int tiles = (Kdim + TK - 1) / TK;
    if (tiles > 0) {
#pragma unroll
        for (int d = 0; d < kDepth; ++d) fetch(d, d < tiles ? d : tiles - 1);
    }
    __syncthreads();   // the word is cleared
    auto step = [&](int set, int t) {   // set and LDS tile are t % 2
        const bool sa = a.commit(set, As + set * AT::SIZE, Kdim - t * TK), sb = b.commit(set, Bs + set * BT::SIZE, Kdim - t * TK);
        if ((sa | sb) && *special == 0) *special = t + 1;
        fetch(set, t + kDepth < tiles ? t + kDepth : tiles - 1);
        __syncthreads();
    };
    int t = 0;
    for (; t + 1 < tiles; t += kDepth) {
        step(0, t);
        step(1, t + 1);
    }
    if (t < tiles) step(0, t);
    __syncthreads();
}
template <class AT, class BT, int MF, int NF, class AAt, class BAt>
__device__ __forceinline__ void multiply_k_tiles(int Kdim, const bf16_t* As, const bf16_t* Bs, LdsWord* special, f32x16 (&acc)[MF][NF], AAt a_at,
                                                 BAt b_at) {
    const int tiles = (Kdim + TK - 1) / TK;
    __syncthreads();
    int t = 0;
    __syncthreads();   // k-tile 0 has landed
    for (; t < tiles && Kdim > kFewTerms; ++t) {
        const int first = __builtin_amdgcn_readfirstlane(*special);
        if (first && t + 1 >= first) break;
        mma_tile<AT, BT>(As + t % 2 * AT::SIZE, Bs + t % 2 * BT::SIZE, acc, a_at, b_at);
        __syncthreads();
    }
    for (; t < tiles; ++t) {
        mma_tile_f32<AT, BT>(As + t % 2 * AT::SIZE, Bs + t % 2 * BT::SIZE, acc, a_at, b_at);
        __syncthreads();
    }
}

}  // namespace mts_split3
