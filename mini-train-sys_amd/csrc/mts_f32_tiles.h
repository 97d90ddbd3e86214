// Tiles of fp32 products on v_mfma_f32_32x32x2_f32 for the router projection of many experts (mts_router_wide.hip):
// loaders, fragment reads and the k loop of a block of four waves.
//
// The k index an operand register stands for is free as long as both operands agree: lanes 0..31 hold k = 8s+0..3 and lanes
// 32..63 k = 8s+4..7 of four consecutive instructions, so an operand whose rows are k-contiguous is read as one 16-byte
// LDS load per four instructions, and one whose memory rows are k ("k-major": the weights in the backward pass, both
// operands of the weight gradient) as four 4-byte loads, with no transposed copy of anything.
#pragma once

#include "mts_common.h"

namespace mts_f32 {

constexpr int kTileThreads = 256;

template <typename XT>
struct Vec4 {
    typedef __attribute__((ext_vector_type(4))) XT type;
};

// four consecutive elements at p, of which the first `count` exist (VEC: p is aligned to four elements and count is 0 or >= 4).
// They stay as they are until they go to LDS: a conversion here would wait for the load.
template <bool VEC, typename XT>
__device__ __forceinline__ typename Vec4<XT>::type load4(const XT* p, int count) {
    typename Vec4<XT>::type v = {};
    if constexpr (VEC) {
        if (count > 0) v = *reinterpret_cast<const typename Vec4<XT>::type*>(p);
    } else {
#pragma unroll
        for (int j = 0; j < 4; ++j)
            if (j < count) v[j] = p[j];
    }
    return v;
}
template <typename V>
__device__ __forceinline__ f32x4 widen4(V v) {
    return f32x4{(float)v[0], (float)v[1], (float)v[2], (float)v[3]};
}

// [ROWS][TKS] tile of k-contiguous rows of XT, floats in LDS.  Rows are TKS + 4 floats apart: the 16-byte fragment reads of 16 lanes then
// start on 16 different groups of four banks.
template <typename XT, int ROWS, int TKS, bool VEC>
struct RowTile {
    static constexpr int LD = TKS + 4, TPR = TKS / 4, LOADS = ROWS * TPR / kTileThreads, SIZE = ROWS * LD;
    const XT* ptr[LOADS];   // this thread's rows, NULL: zeros
    typename Vec4<XT>::type reg[2][LOADS];
    __device__ __forceinline__ static int row(int p) { return threadIdx.x / TPR + p * (kTileThreads / TPR); }
    __device__ __forceinline__ void fetch(int set, int k0, int Kdim) {
        const int k = k0 + (threadIdx.x % TPR) * 4;
#pragma unroll
        for (int p = 0; p < LOADS; ++p) reg[set][p] = load4<VEC>(ptr[p] + k, ptr[p] ? Kdim - k : 0);
    }
    __device__ __forceinline__ void commit(int set, float* lds) const {
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
template <typename XT, int COLS, int TKS, bool VEC>
struct KTile {
    static constexpr int LD = COLS + 8, LOADS = COLS * TKS / 4 / kTileThreads, SIZE = TKS * LD, PER_ROW = COLS / 4;
    const XT* base;          // element (k = 0, this thread's first column)
    int64_t ld;
    int cols;                // columns from there on that exist
    typename Vec4<XT>::type reg[2][LOADS];
    __device__ __forceinline__ static int k(int p) { return threadIdx.x / PER_ROW + p * (kTileThreads / PER_ROW); }
    __device__ __forceinline__ static int col() { return (threadIdx.x % PER_ROW) * 4; }
    // rows[p] = memory row of k-row k(p), or < 0: zeros
    __device__ __forceinline__ void fetch(int set, const int64_t (&rows)[LOADS]) {
#pragma unroll
        for (int p = 0; p < LOADS; ++p) reg[set][p] = load4<VEC>(base + rows[p] * ld, rows[p] >= 0 ? cols : 0);
    }
    __device__ __forceinline__ void commit(int set, float* lds) const {
#pragma unroll
        for (int p = 0; p < LOADS; ++p) *reinterpret_cast<f32x4*>(lds + k(p) * LD + col()) = widen4(reg[set][p]);
    }
    __device__ __forceinline__ static f32x4 frag(const float* lds, int c0, int s) {
        const int lane = threadIdx.x % MTS_WAVE;
        const float* q = lds + (s * 8 + (lane / 32) * 4) * LD + c0 + lane % 32;
        return f32x4{q[0], q[LD], q[2 * LD], q[3 * LD]};
    }
};

// STEPS k-steps from s0 on (8 of k each) of one k-tile: MF x NF fragments of 32x32 per wave; a_at / b_at give the first row / column of a fragment in the tile
template <class AT, class BT, int STEPS, int MF, int NF, class AAt, class BAt>
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
                    acc[mf][nf] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[mf][j], b[nf][j], acc[mf][nf], 0, 0, 0);
    }
}

// The k loop: two LDS buffers, and two k-tiles in flight in registers behind them (a tile's loads have two tiles' matrix
// work to arrive in).  fetch(set, t) starts the loads of k-tile t; it is called once for every t in order.
template <class AT, class BT, int STEPS, int MF, int NF, class AAt, class BAt, class Fetch>
__device__ __forceinline__ void run_k_tiles(int tiles, AT& a, BT& b, float (*As)[AT::SIZE], float (*Bs)[BT::SIZE], f32x16 (&acc)[MF][NF],
                                            AAt a_at, BAt b_at, Fetch fetch, int s0 = 0) {
    if (tiles <= 0) return;
    fetch(0, 0);
    if (tiles > 1) fetch(1, 1);
    a.commit(0, As[0]);
    b.commit(0, Bs[0]);
    __syncthreads();
    for (int t0 = 0; t0 < tiles; t0 += 2) {
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const int t = t0 + u;
            if (t >= tiles) break;
            if (t + 2 < tiles) fetch(u, t + 2);
            mma_tile32<AT, BT, STEPS, MF, NF>(As[u], Bs[u], acc, a_at, b_at, s0);
            if (t + 1 < tiles) {
                a.commit(1 - u, As[1 - u]);
                b.commit(1 - u, Bs[1 - u]);
            }
            __syncthreads();
        }
    }
}

}  // namespace mts_f32
