// Tiles of fp32 products on v_mfma_f32_32x32x2_f32 for the router projection of many experts (mts_router_wide.hip):
// loaders, fragment reads and the k loop of a block of THREADS threads.
//
// The k index an operand register stands for is free as long as both operands agree: lanes 0..31 hold k = 8s+0..3 and lanes
// 32..63 k = 8s+4..7 of four consecutive instructions, so an operand whose rows are k-contiguous is read as one 16-byte
// LDS load per four instructions, and one whose memory rows are k ("k-major": the weights in the backward pass, both
// operands of the weight gradient) as four 4-byte loads, with no transposed copy of anything.
#pragma once

#include "mts_common.h"

namespace mts_f32 {

template <typename XT>
struct Vec4 {
    typedef __attribute__((ext_vector_type(4))) XT type;
};

// Elements p[first .. first + 3] of `count` (VEC: both are multiples of four, and p is aligned to four elements).  Unconditional: a load that a
// lane or a pass may skip makes the compiler wait for all loads in flight at the next use of any.  What lies outside is read from the last
// element instead: along k it is set to zero on its way into LDS, along rows and columns it reaches outputs that nobody stores.
// They stay as they are until they go to LDS: a conversion here would wait for the load.
template <bool VEC, typename XT>
__device__ __forceinline__ typename Vec4<XT>::type load4(const XT* p, int first, int count) {
    if constexpr (VEC) return *reinterpret_cast<const typename Vec4<XT>::type*>(p + (first < count ? first : count - 4));
    typename Vec4<XT>::type v;
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] = p[first + j < count ? first + j : count - 1];
    return v;
}
template <typename V>
__device__ __forceinline__ f32x4 widen4(V v) {
    return f32x4{(float)v[0], (float)v[1], (float)v[2], (float)v[3]};
}

// [ROWS][TKS] tile of k-contiguous rows of XT, floats in LDS.  Rows are TKS + 4 floats apart: the 16-byte fragment reads of 16 lanes then
// start on 16 different groups of four banks.
template <typename XT, int ROWS, int TKS, bool VEC, int THREADS = 256>
struct RowTile {
    static constexpr int LD = TKS + 4, TPR = TKS / 4, LOADS = ROWS * TPR / THREADS, SIZE = ROWS * LD;
    static_assert(LOADS * THREADS == ROWS * TPR, "every thread loads as much");
    const XT* ptr[LOADS];   // this thread's rows
    typename Vec4<XT>::type reg[2][LOADS];
    __device__ __forceinline__ static int row(int p) { return threadIdx.x / TPR + p * (THREADS / TPR); }
    __device__ __forceinline__ void fetch(int set, int k0, int Kdim) {
#pragma unroll
        for (int p = 0; p < LOADS; ++p) reg[set][p] = load4<VEC>(ptr[p], k0 + (threadIdx.x % TPR) * 4, Kdim);
    }
    // the first `count` of the tile's k are added
    __device__ __forceinline__ void commit(int set, float* lds, int count) {
        if (count < TKS) {
#pragma unroll
            for (int p = 0; p < LOADS; ++p)
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    if ((int)(threadIdx.x % TPR) * 4 + j >= count) reg[set][p][j] = (XT)0.f;
        }
#pragma unroll
        for (int p = 0; p < LOADS; ++p) *reinterpret_cast<f32x4*>(lds + row(p) * LD + (threadIdx.x % TPR) * 4) = widen4(reg[set][p]);
    }
    // k = 8s + 4 * (lane / 32) + 0..3 of row `r0 + lane % 32`
    __device__ __forceinline__ static f32x4 frag(const float* lds, int r0, int s) {
        const int lane = threadIdx.x % MTS_WAVE;
        return *reinterpret_cast<const f32x4*>(lds + (r0 + lane % 32) * LD + s * 8 + (lane / 32) * 4);
    }
};

// [TKS][COLS] tile of k-major rows of XT.  The row length in LDS puts k and k+4, which the two halves of a wave read together,
// 32 banks apart.
template <typename XT, int COLS, int TKS, bool VEC, int THREADS = 256>
struct KTile {
    static constexpr int LD = COLS + 8, LOADS = COLS * TKS / 4 / THREADS, SIZE = TKS * LD, PER_ROW = COLS / 4;
    const XT* base;          // element (k = 0, the tile's first column)
    int64_t ld;
    int cols;                // columns from there on that exist
    typename Vec4<XT>::type reg[2][LOADS];
    __device__ __forceinline__ static int k(int p) { return threadIdx.x / PER_ROW + p * (THREADS / PER_ROW); }
    __device__ __forceinline__ static int col() { return (threadIdx.x % PER_ROW) * 4; }
    // rows[p] = memory row of k-row k(p)
    __device__ __forceinline__ void fetch(int set, const int64_t (&rows)[LOADS]) {
#pragma unroll
        for (int p = 0; p < LOADS; ++p) reg[set][p] = load4<VEC>(base + rows[p] * ld, col(), cols);
    }
    __device__ __forceinline__ void commit(int set, float* lds, int count) {
        if (count < TKS) {
#pragma unroll
            for (int p = 0; p < LOADS; ++p)
                if (k(p) >= count) reg[set][p] = typename Vec4<XT>::type{};
        }
#pragma unroll
        for (int p = 0; p < LOADS; ++p) *reinterpret_cast<f32x4*>(lds + k(p) * LD + col()) = widen4(reg[set][p]);
    }
    __device__ __forceinline__ static f32x4 frag(const float* lds, int c0, int s) {
        const int lane = threadIdx.x % MTS_WAVE;
        const float* q = lds + (s * 8 + (lane / 32) * 4) * LD + c0 + lane % 32;
        return f32x4{q[0], q[LD], q[2 * LD], q[3 * LD]};
    }
};

// SWAP: a lane then holds columns of one row instead of rows of one column.
// STEPS k-steps from s0 on (8 of k each) of one k-tile: MF x NF fragments of 32x32 per wave; a_at / b_at give the first row / column of a fragment in the tile
template <class AT, class BT, int STEPS, int MF, int NF, bool SWAP = false, class AAt, class BAt>
__device__ __forceinline__ void mma_tile32(const float* As, const float* Bs, f32x16 (&acc)[MF][NF], AAt a_at, BAt b_at, int s0 = 0) {
#pragma unroll
    for (int s = 0; s < STEPS; ++s) {
        f32x4 a[MF], b[NF];
#pragma unroll
        for (int i = 0; i < MF; ++i) a[i] = AT::frag(As, a_at(i), s0 + s);
#pragma unroll
        for (int i = 0; i < NF; ++i) b[i] = BT::frag(Bs, b_at(i), s0 + s);
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int mf = 0; mf < MF; ++mf)
#pragma unroll
                for (int nf = 0; nf < NF; ++nf)
                    acc[mf][nf] = SWAP ? __builtin_amdgcn_mfma_f32_32x32x2f32(b[nf][j], a[mf][j], acc[mf][nf], 0, 0, 0)
                                       : __builtin_amdgcn_mfma_f32_32x32x2f32(a[mf][j], b[nf][j], acc[mf][nf], 0, 0, 0);
    }
}

// The k loop: two LDS buffers, and two k-tiles in flight in registers behind them (a tile's loads have two tiles' matrix
// work to arrive in).  fetch(set, t) starts the loads of k-tile t; it is called for every t in order, and for the last one again behind that.
template <class AT, class BT, int TKS, int STEPS, int MF, int NF, bool SWAP = false, class AAt, class BAt, class Fetch>
__device__ __forceinline__ void run_k_tiles(int Kdim, AT& a, BT& b, float (*As)[AT::SIZE], float (*Bs)[BT::SIZE], f32x16 (&acc)[MF][NF],
                                            AAt a_at, BAt b_at, Fetch fetch, int s0 = 0) {
    const int tiles = (Kdim + TKS - 1) / TKS;
    if (tiles <= 0) return;
    fetch(0, 0);
    fetch(1, tiles > 1 ? 1 : 0);
    a.commit(0, As[0], Kdim);
    b.commit(0, Bs[0], Kdim);
    __syncthreads();
    auto step = [&](int u, int t) {   // buffer and set are t % 2; the tile behind this one goes to the other buffer
        fetch(u, t + 2 < tiles ? t + 2 : tiles - 1);
        mma_tile32<AT, BT, STEPS, MF, NF, SWAP>(As[u], Bs[u], acc, a_at, b_at, s0);
        a.commit(1 - u, As[1 - u], Kdim - (t + 1) * TKS);
        b.commit(1 - u, Bs[1 - u], Kdim - (t + 1) * TKS);
        __syncthreads();
    };
    int t = 0;
    for (; t + 1 < tiles; t += 2) {
        step(0, t);
        step(1, t + 1);
    }
    if (t < tiles) step(0, t);
}

}  // namespace mts_f32
