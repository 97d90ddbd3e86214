// fp32 variant of the grouped expert GEMMs: activations, weights and results in fp32.  Same contracts and epilogues as the
// 16-bit kernels.
//
// An fp32 value is the exact sum of three bf16 ones (x = x0 + x1 + x2, each the rest rounded to nearest: mts_split3.h), a
// product of two bf16 values is exact in fp32, and the bf16 matrix instruction adds in fp32 at 16 times the rate of the fp32
// one.  A product is therefore taken as x0*y0 + x0*y1 + x1*y0 + x1*y1 + x0*y2 + x2*y0; the three terms left out are below
// 2^-26 of it, a quarter of an fp32 rounding, and a sum of three and more products still comes out closer than from the fp32
// instruction, which rounds more often.  Shorter sums (the weight gradient of an expert with one or two rows) are left to
// that instruction, and so are k-tiles that hold a value whose split is not exact (infinite, NaN, below 2^-60 or
// from 2^50 on, but not zero).
//
// What bounds it: on paper the matrix pipes (six instructions of 32 cycles for a 32 x 32 x 16 product: 417 TFLOP/s at 2.4 GHz, 2.7 times the fp32
// instruction), in fact the vector unit that splits: a value costs about 8 vector instructions, each 4.9 cycles of a SIMD, and a wave alone
// issues one in 8.  Hence half of a block's waves load and split while the other half multiply (in step, a block's two phases would add
// up), tiles as large as two blocks of a CU can be (128 x 128, 16 of k, two LDS tiles: each value is split once per 128 outputs), and
// loads that never depend on a branch.  2048 tokens, 768/1024, 8 experts, top-2, us before (fp32 instruction) and now: gate/up 178 -> 112, down
// 90 -> 60, dO*W2 95 -> 90, dX 167 -> 96, dW1 146 -> 87, dW2 76 -> 57; 8192 tokens: 588 -> 397, 282 -> 172, 298 -> 227, 498 -> 324, 512 -> 303, 266 -> 177.
// Relative error against fp64 over all five results of the operator: 4.1e-7..1.02e-6 where the fp32 instruction had 4.3e-7..1.18e-6,
// smaller for each at every size; by the length of the sum: mts_split3.h.
#include "mts_ds_block.h"
#include "mts_split3.h"

#include <type_traits>

namespace {

using namespace mts_split3;

constexpr int kXcds = 8;

// Tiles of 128 x 128 where about 160 of them come together: below that the CUs they leave idle cost more than the smaller tiles'
// splitting of every value twice as often.  us, 64 x 64 / 128 x 128 tiles, top-2, 8 experts of 768/1024: gate/up 32 / 39 at 256 tokens (128 tiles),
// 47 / 42 at 512 (192); down 45 / 49 at 1024 (120), 76 / 60 at 2048 (216); dX 81 / 85 and 129 / 95 there.  Weight gradients, whose tiles do not
// depend on the rows: dW1 15.2 / 14.5 at 64 tokens, 114 / 87 at 2048.
bool large_tiles(int64_t rows, int64_t cols, int units) { return (rows + 64 * (int64_t)units) * cols >= 160 * 128 * 128; }

enum Epi32 { E32_PLAIN = 0, E32_SWIGLU = 1, E32_DY1 = 2 };

struct Rows32 {
    const float* A;
    int lda;
    const int32_t* a_gather;
    const float* B;      // [E][b_rows][Kdim], or k-major: [E][Kdim][N]
    int b_rows;
    int N, Kdim;
    const int32_t* expert_start;
    int E;
    float* C;
    float* C2;
    const float* pre_act;
    const float* route_w;
    const int32_t* s_scatter;
    float* ds_part;
    int np;
    int n_tiles;
};

__device__ __forceinline__ float sigmoid32(float x) { return 1.0f / (1.0f + expf(-x)); }

// The m-tiles of all experts in expert order, 64 experts per round: their number, and expert and rows of tile `tile`
// (every lane of the wave gets the same answer; tile < 0: only the number is wanted).
template <int BM>
__device__ __forceinline__ int find_m_tile(const int32_t* __restrict__ expert_start, int E, int tile, int& e_out, int& row0, int& rend) {
    const int lane = threadIdx.x % MTS_WAVE;
    int seen = 0;
    for (int e0 = 0; e0 < E; e0 += MTS_WAVE) {
        const int e = e0 + lane;
        const int s0 = e < E ? expert_start[e] : 0, s1 = e < E ? expert_start[e + 1] : 0;
        const int nt = (s1 - s0 + BM - 1) / BM;
        const int upto = wave_scan(nt);
        const uint64_t mine = __ballot(tile >= seen + upto - nt && tile < seen + upto);
        if (mine) {
            const int l = __ffsll((unsigned long long)mine) - 1;
            e_out = e0 + l;
            row0 = __builtin_amdgcn_readlane(s0, l) + (tile - seen - __builtin_amdgcn_readlane(upto - nt, l)) * BM;
            rend = __builtin_amdgcn_readlane(s1, l);
        }
        seen += __builtin_amdgcn_readlane(upto, MTS_WAVE - 1);
    }
    return seen;
}

// BN counts the columns of the B tile (SwiGLU: gate and up columns side by side, half the outputs)
template <int BM, int BN, int EPI, bool BKM, bool VEC>
struct RowsTile {
    static constexpr int WAVES_M = 2, WAVES_N = 2;
    typedef RowPlanes<BM, VEC> ATile;
    typedef typename std::conditional<BKM, KPlanes<BN, VEC>, RowPlanes<BN, VEC>>::type BTile;
    struct Lds {
        __attribute__((aligned(16))) bf16_t As[2 * ATile::SIZE];
        __attribute__((aligned(16))) bf16_t Bs[2 * BTile::SIZE];
        float ds_sum[EPI == E32_DY1 ? WAVES_N : 1][BM];
        float row_weight[EPI == E32_PLAIN ? 1 : BM];
        int special;
    };
};

// the work of block `block`
template <int BM, int BN, int EPI, bool BKM, bool VEC>
__device__ __forceinline__ void rows_block(const Rows32& p, int block, typename RowsTile<BM, BN, EPI, BKM, VEC>::Lds& lds) {
    typedef RowsTile<BM, BN, EPI, BKM, VEC> Tile;
    typedef typename Tile::ATile ATile;
    typedef typename Tile::BTile BTile;
    constexpr int WAVES_M = Tile::WAVES_M, WAVES_N = Tile::WAVES_N;
    constexpr int MF = BM / WAVES_M / 32, NF = BN / WAVES_N / 32;
    constexpr int OUT_N = EPI == E32_SWIGLU ? BN / 2 : BN, SLOT = 64, SLOTS = OUT_N / SLOT, HALF = NF > 1 ? NF / 2 : 1;
    static_assert(OUT_N % SLOT == 0, "partial row sums cover 64 columns each");
    bf16_t *As = lds.As, *Bs = lds.Bs;
    auto& ds_sum = lds.ds_sum;
    auto& row_weight = lds.row_weight;
    int& special = lds.special;

    // block b runs on XCD b % 8: every XCD takes an equal contiguous run of the tiles, columns fastest, so that an expert's
    // weights stream through one L2 and the blocks that share activation rows are neighbours in time
    int e = 0, row0 = 0, rend = 0;
    const int total = find_m_tile<BM>(p.expert_start, p.E, -1, e, row0, rend) * p.n_tiles;
    const int per_xcd = (total + kXcds - 1) / kXcds, slot = block / kXcds;
    const int tile = (block % kXcds) * per_xcd + slot;
    if (slot >= per_xcd || tile >= total) return;
    find_m_tile<BM>(p.expert_start, p.E, tile / p.n_tiles, e, row0, rend);
    const int ny = tile % p.n_tiles, n0 = ny * OUT_N;

    if constexpr (EPI != E32_PLAIN) {   // the k loop's barriers stand between these and the epilogue
        const int r = row0 + threadIdx.x;
        if (threadIdx.x < BM) row_weight[threadIdx.x] = p.route_w && r < rend ? p.route_w[p.s_scatter[r]] : 1.f;
    }
    if (threadIdx.x == 0) special = 0;
    f32x16 acc[MF][NF] = {};
    const int wave = threadIdx.x / MTS_WAVE, wm = wave / WAVES_N, wn = wave % WAVES_N, lane = threadIdx.x % MTS_WAVE;
    auto a_at = [&](int mf) { return wm * (BM / WAVES_M) + mf * 32; };
    auto b_at = [&](int nf) { return EPI == E32_SWIGLU ? nf / HALF * OUT_N + wn * (OUT_N / WAVES_N) + nf % HALF * 32 : wn * (BN / WAVES_N) + nf * 32; };
    if (threadIdx.x >= kLoaders) {
        ATile a;
#pragma unroll
        for (int q = 0; q < ATile::LOADS; ++q) {
            const int r = row0 + ATile::row(q) < rend ? row0 + ATile::row(q) : rend - 1;
            a.ptr[q] = p.A + (int64_t)(p.a_gather ? p.a_gather[r] : r) * p.lda;
        }
        const float* Be = p.B + (int64_t)e * p.b_rows * p.Kdim;
        BTile b;
        if constexpr (BKM) {
            b.base = Be + n0;
            b.ld = p.N;
            b.cols = p.N - n0;
        } else {
#pragma unroll
            for (int q = 0; q < BTile::LOADS; ++q) {
                const int r = BTile::row(q), half = r / OUT_N, n = n0 + r % OUT_N < p.N ? n0 + r % OUT_N : p.N - 1;
                b.ptr[q] = Be + (int64_t)(half * p.N + n) * p.Kdim;
            }
        }
        auto fetch = [&](int set, int t) {
            a.fetch(set, t * TK, p.Kdim);
            if constexpr (BKM) {
                int64_t rows[BTile::LOADS];
#pragma unroll
                for (int q = 0; q < BTile::LOADS; ++q) rows[q] = t * TK + BTile::k(q) < p.Kdim ? t * TK + BTile::k(q) : p.Kdim - 1;
                b.fetch(set, rows);
            } else b.fetch(set, t * TK, p.Kdim);
        };
        load_k_tiles(p.Kdim, a, b, As, Bs, (LdsWord*)&special, fetch);
    } else multiply_k_tiles<ATile, BTile>(p.Kdim, As, Bs, (LdsWord*)&special, acc, a_at, b_at);

    if (threadIdx.x < kLoaders) {
#pragma unroll
        for (int mf = 0; mf < MF; ++mf)
#pragma unroll
            for (int i4 = 0; i4 < 16; i4 += 4) {
                const int r0 = a_at(mf) + 8 * (i4 / 4) + 4 * (lane / 32);   // the lane's four rows from here on
                float g[NF][4], u[NF][4];
                if constexpr (EPI == E32_DY1) {   // all loads of the four rows ahead of their use; the ones that do not exist read others
#pragma unroll
                    for (int nf = 0; nf < NF; ++nf)
#pragma unroll
                        for (int j = 0; j < 4; ++j) {
                            const int row = row0 + r0 + j < rend ? row0 + r0 + j : rend - 1, n = n0 + b_at(nf) + lane % 32;
                            const float* src = p.pre_act + (int64_t)row * (2 * p.N) + (n < p.N ? n : 0);
                            g[nf][j] = src[0], u[nf][j] = src[p.N];
                        }
                }
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const int r = r0 + j, row = row0 + r, i = i4 + j;
                    const bool rok = row < rend;
                    if constexpr (EPI == E32_PLAIN) {
#pragma unroll
                        for (int nf = 0; nf < NF; ++nf) {
                            const int n = n0 + b_at(nf) + lane % 32;
                            if (rok && n < p.N) p.C[(int64_t)row * p.N + n] = acc[mf][nf][i];
                        }
                    } else if constexpr (EPI == E32_SWIGLU) {
                        const float s = row_weight[r];   // post_act may carry the routing weight
#pragma unroll
                        for (int nf = 0; nf < NF / 2; ++nf) {
                            const int n = n0 + b_at(nf) + lane % 32;
                            const float gate = acc[mf][nf][i], up = acc[mf][nf + NF / 2][i];
                            const float y = gate * sigmoid32(gate) * up * s;
                            if (!rok || n >= p.N) continue;
                            p.C[(int64_t)row * (2 * p.N) + n] = gate;
                            p.C[(int64_t)row * (2 * p.N) + p.N + n] = up;
                            p.C2[(int64_t)row * p.N + n] = y;
                        }
                    } else {
                        const float s = row_weight[r];
                        float dsp = 0.f;
#pragma unroll
                        for (int nf = 0; nf < NF; ++nf) {
                            const int n = n0 + b_at(nf) + lane % 32;
                            const int64_t o = (int64_t)row * (2 * p.N) + n;
                            const float v = acc[mf][nf][i];
                            const float sig = sigmoid32(g[nf][j]);
                            const float silu = g[nf][j] * sig;
                            const float y1 = silu * u[nf][j];
                            const float da = v * s, dg = da * (silu * (1.0f - sig) + sig) * u[nf][j];
                            if (!rok || n >= p.N) continue;
                            dsp += v * y1;
                            if (p.C2) p.C2[(int64_t)row * p.N + n] = s * y1;
                            p.C[o] = dg;
                            p.C[o + p.N] = da * silu;
                        }
#pragma unroll
                        for (int o = 16; o > 0; o >>= 1) dsp += __shfl_xor(dsp, o, 32);
                        if (lane % 32 == 0) ds_sum[wn][r] = dsp;
                    }
                }
            }
    }
    if constexpr (EPI == E32_DY1) {   // row sums over 64 columns each: of one wave, or of the two that share them
        constexpr int PER = WAVES_N / SLOTS;
        __syncthreads();
        for (int i = threadIdx.x; i < BM * SLOTS; i += kThreads) {
            const int r = i % BM, slot = i / BM, at = ny * SLOTS + slot;
            if (row0 + r < rend && at < p.np) {
                float v = ds_sum[slot * PER][r];
#pragma unroll
                for (int q = 1; q < PER; ++q) v += ds_sum[slot * PER + q][r];
                p.ds_part[(int64_t)(row0 + r) * p.np + at] = v;
            }
        }
    }
}

template <int BM, int BN, int EPI, bool BKM, bool VEC>
__global__ __launch_bounds__(kThreads, 4) void rows_gemm_f32_kernel(Rows32 p) {
    __shared__ typename RowsTile<BM, BN, EPI, BKM, VEC>::Lds lds;
    rows_block<BM, BN, EPI, BKM, VEC>(p, blockIdx.x, lds);
}

struct Dw32 {
    const float* P;
    const int32_t* p_gather;
    const float* Q;
    const int32_t* q_gather;
    int M, N;
    const int32_t* expert_start;
    int E;
    void* C;
    int m_tiles, n_tiles;
};

// The expert with the `n`-th most rows: the longest sums start first.  More experts than a wave has lanes: as they come.
__device__ __forceinline__ int longest_expert(const int32_t* __restrict__ expert_start, int E, int n) {
    if (E > MTS_WAVE) return n;
    const int lane = threadIdx.x % MTS_WAVE;
    const int rows = lane < E ? expert_start[lane + 1] - expert_start[lane] : -1;
    int before = 0;
    for (int f = 0; f < E; ++f) {
        const int other = __builtin_amdgcn_readlane(rows, f);
        before += other > rows || (other == rows && f < lane) ? 1 : 0;
    }
    return __ffsll((unsigned long long)__ballot(lane < E && before == n)) - 1;
}

template <int BM, int BN, bool VEC>
struct DwTile {
    typedef KPlanes<BM, VEC> PT;
    typedef KPlanes<BN, VEC> QT;
    struct Lds {
        __attribute__((aligned(16))) bf16_t Ps[2 * PT::SIZE];
        __attribute__((aligned(16))) bf16_t Qs[2 * QT::SIZE];
        int special;
    };
};

// BM x BN outputs; the reduction runs over the expert's rows, both operands k-major
template <int BM, int BN, typename OutT, bool VEC>
__device__ __forceinline__ void dw_block(const Dw32& p, int block, typename DwTile<BM, BN, VEC>::Lds& lds) {
    constexpr int MF = BM / 64, NF = BN / 64;
    typedef typename DwTile<BM, BN, VEC>::PT PT;
    typedef typename DwTile<BM, BN, VEC>::QT QT;
    bf16_t *Ps = lds.Ps, *Qs = lds.Qs;
    int& special = lds.special;
    // an XCD takes an equal contiguous run of every expert's tiles, columns fastest: an equal share of the work however
    // uneven the experts are, and about an eighth of P through its L2
    const int per_expert = p.m_tiles * p.n_tiles, per_xcd = (per_expert + kXcds - 1) / kXcds;
    const int slot = block / kXcds;
    const int tile = (block % kXcds) * per_xcd + slot % per_xcd;
    if (tile >= per_expert || slot / per_xcd >= p.E) return;
    const int e = longest_expert(p.expert_start, p.E, slot / per_xcd);
    const int m0 = tile / p.n_tiles * BM, n0 = tile % p.n_tiles * BN;
    const int rbeg = p.expert_start[e], rend = p.expert_start[e + 1];

    if (threadIdx.x == 0) special = 0;
    const int wave = threadIdx.x / MTS_WAVE, wm = wave / 2, wn = wave % 2, lane = threadIdx.x % MTS_WAVE;
    auto a_at = [&](int mf) { return wm * (BM / 2) + mf * 32; };
    auto b_at = [&](int nf) { return wn * (BN / 2) + nf * 32; };
    f32x16 acc[MF][NF] = {};
    if (threadIdx.x >= kLoaders) {
        PT a;
        QT b;
        a.base = p.P + m0, a.ld = p.M, a.cols = p.M - m0;
        b.base = p.Q + n0, b.ld = p.N, b.cols = p.N - n0;
        // Memory rows of the k-tiles, read two tiles ahead: loads return in order, so a row read one tile ahead would be waited
        // for together with the data of the tile in front of it.  An operand that is not gathered reads some index and drops it.
        int pi[2][PT::LOADS], qi[2][QT::LOADS];
        auto locate = [&](int set, int r0) {
#pragma unroll
            for (int q = 0; q < PT::LOADS; ++q) pi[set][q] = *(p.p_gather ? p.p_gather + min(r0 + PT::k(q), rend - 1) : p.expert_start);
#pragma unroll
            for (int q = 0; q < QT::LOADS; ++q) qi[set][q] = *(p.q_gather ? p.q_gather + min(r0 + QT::k(q), rend - 1) : p.expert_start);
        };
        if (rbeg < rend) {
            locate(0, rbeg);
            locate(1, rbeg + TK);
        }
        auto fetch = [&](int set, int t) {   // set is t % 2
            const int r0 = rbeg + t * TK;
            int64_t pr[PT::LOADS], qr[QT::LOADS];
#pragma unroll
            for (int q = 0; q < PT::LOADS; ++q) pr[q] = p.p_gather ? pi[set][q] : min(r0 + PT::k(q), rend - 1);
#pragma unroll
            for (int q = 0; q < QT::LOADS; ++q) qr[q] = p.q_gather ? qi[set][q] : min(r0 + QT::k(q), rend - 1);
            a.fetch(set, pr);
            b.fetch(set, qr);
            locate(set, r0 + 2 * TK);
        };
        load_k_tiles(rend - rbeg, a, b, Ps, Qs, (LdsWord*)&special, fetch);
        return;
    }
    multiply_k_tiles<PT, QT>(rend - rbeg, Ps, Qs, (LdsWord*)&special, acc, a_at, b_at);

    OutT* C = reinterpret_cast<OutT*>(p.C) + (int64_t)e * p.M * p.N;
#pragma unroll
    for (int mf = 0; mf < MF; ++mf)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const int m = m0 + a_at(mf) + 8 * (i / 4) + 4 * (lane / 32) + i % 4;
#pragma unroll
            for (int nf = 0; nf < NF; ++nf) {
                const int n = n0 + b_at(nf) + lane % 32;
                if (m < p.M && n < p.N) C[(int64_t)m * p.N + n] = (OutT)acc[mf][nf][i];
            }
        }
}

template <int BM, int BN, typename OutT, bool VEC>
__global__ __launch_bounds__(kThreads, 4) void dw_gemm_f32_kernel(Dw32 p) {
    __shared__ typename DwTile<BM, BN, VEC>::Lds lds;
    dw_block<BM, BN, OutT, VEC>(p, blockIdx.x, lds);
}

// the experts with more than `rows` rows; more experts than a wave has lanes: all of them where one has
__device__ __forceinline__ int longer_experts(const int32_t* __restrict__ expert_start, int E, int rows) {
    int longer = 0;
    for (int e0 = 0; e0 < E; e0 += MTS_WAVE) {
        const int e = e0 + threadIdx.x % MTS_WAVE;
        longer += (int)__popcll(__ballot(e < E && expert_start[min(e, E - 1) + 1] - expert_start[min(e, E - 1)] > rows));
    }
    return E > MTS_WAVE && longer ? E : longer;
}

// dX, dW1, dW2 and the routing weights' gradient in one launch: blocks of one part take the CUs as those in front leave them, and nothing is forked onto
// other streams and joined again (four events, for which the host takes 20 us and the stream some 5 each).  In front of dX, whose sums have 2I terms, come the
// weight gradients of experts with more than two thirds as many rows, the longest first; behind it those of the others.  Whole operators, us, as launches
// side by side and so: 64 tokens of 256/256 210 / 125; 256 of 768/1024 202 / 171; 2048 477 / 456, a few experts popular 476 / 470; 4096 of 1024/1024 1066 /
// 1045 and 1052 / 1048; 8192 of 768/1024 1493 / 1465 and 1490 / 1488.  With all of dX in front 4096 tokens and popular experts took 1060 for 1019, with all of
// it behind 2048 even ones 478 for 442; with both weight gradients of an expert side by side 2048 tokens of 16 popular experts 530 for 498.
struct Bwd32 {
    Rows32 dx;
    Dw32 dw1, dw2;
    int n_dx, n_dw1, n_dw2, per_dw1, per_dw2;   // blocks, multiples of the XCDs; blocks an expert and XCD
    const float* ds_part;
    const int32_t* s_reverse;
    int64_t entries;
    int np, n_ds;
    float* d_weights;
};
template <int DX, int DW>
__global__ __launch_bounds__(kThreads, 4) void bwd_joint_f32_kernel(Bwd32 q) {
    __shared__ union {
        typename RowsTile<DX, DX, E32_PLAIN, true, true>::Lds dx;
        typename DwTile<DW, DW, true>::Lds dw;
    } lds;
    const int front = longer_experts(q.dx.expert_start, q.dx.E, 2 * q.dx.Kdim / 3) * kXcds, front1 = front * q.per_dw1, front2 = front * q.per_dw2;
    int b = blockIdx.x;
    if (b < front1) return dw_block<DW, DW, float, true>(q.dw1, b, lds.dw);
    b -= front1;
    if (b < front2) return dw_block<DW, DW, float, true>(q.dw2, b, lds.dw);
    b -= front2;
    if (b < q.n_dx) return rows_block<DX, DX, E32_PLAIN, true, true>(q.dx, b, lds.dx);
    b -= q.n_dx;
    if (b < q.n_dw1 - front1) return dw_block<DW, DW, float, true>(q.dw1, front1 + b, lds.dw);
    b -= q.n_dw1 - front1;
    if (b < q.n_dw2 - front2) return dw_block<DW, DW, float, true>(q.dw2, front2 + b, lds.dw);
    b -= q.n_dw2 - front2;
    mts_ds::sum_block<float, kThreads>(q.ds_part, q.s_reverse, q.entries, q.np, q.d_weights, b, q.n_ds);
}

int64_t dw_blocks(const Dw32& p) { return ((int64_t)p.m_tiles * p.n_tiles + kXcds - 1) / kXcds * kXcds * p.E; }

int64_t m_tiles32(int64_t rows, int E, int bm) {
    const int64_t a = (rows + bm - 1) / bm + E - 1;
    return a < rows ? a : rows;
}

template <int BM, int BN, int EPI, bool BKM>
int launch_rows_tile(Rows32 p, int64_t rows, bool vec, hipStream_t s) {
    constexpr int OUT_N = EPI == E32_SWIGLU ? BN / 2 : BN;
    p.n_tiles = (p.N + OUT_N - 1) / OUT_N;
    const int64_t blocks = (m_tiles32(rows, p.E, BM) * p.n_tiles + kXcds - 1) / kXcds * kXcds;
    if (blocks >= (1LL << 31)) return MTS_ERR_SHAPE;
    const dim3 grid((unsigned)blocks);
    if (vec) rows_gemm_f32_kernel<BM, BN, EPI, BKM, true><<<grid, kThreads, 0, s>>>(p);
    else rows_gemm_f32_kernel<BM, BN, EPI, BKM, false><<<grid, kThreads, 0, s>>>(p);
    MTS_CHECK_LAUNCH();
    return MTS_OK;
}

template <int EPI, bool BKM>
int launch_rows(const Rows32& p, int64_t rows, bool vec, hipStream_t s) {
    constexpr int SMALL_N = EPI == E32_SWIGLU ? 128 : 64;
    if (large_tiles(rows, EPI == E32_SWIGLU ? 2 * p.N : p.N, p.E)) return launch_rows_tile<128, 128, EPI, BKM>(p, rows, vec, s);
    return launch_rows_tile<64, SMALL_N, EPI, BKM>(p, rows, vec, s);
}

}  // namespace

// entry points used by the dispatchers in mts_gemm.hip when act_dtype == MTS_F32; b_kmajor: B is [E][Kdim][N]
int mts_f32_rows(int epi, const float* A, int lda, const int32_t* a_gather, const float* B, int b_rows, int b_kmajor,
                 int N, int Kdim, const int32_t* expert_start, int E, int64_t TK, float* C, float* C2,
                 const float* pre_act, const float* route_w, const int32_t* s_scatter, float* ds_part,
                 int np, hipStream_t s) {
    Rows32 p = {A, lda, a_gather, B, b_rows, N, Kdim, expert_start, E, C, C2, pre_act, route_w, s_scatter, ds_part, np, 0};
    // rows that are whole 16-byte groups; others are loaded four bytes at a time
    const bool vec = lda % 4 == 0 && Kdim % 4 == 0 && (!b_kmajor || N % 4 == 0) && mts_aligned16(A) && mts_aligned16(B);
    if (epi == E32_SWIGLU) return launch_rows<E32_SWIGLU, false>(p, TK, vec, s);
    if (epi == E32_PLAIN) return b_kmajor ? launch_rows<E32_PLAIN, true>(p, TK, vec, s) : launch_rows<E32_PLAIN, false>(p, TK, vec, s);
    return b_kmajor ? launch_rows<E32_DY1, true>(p, TK, vec, s) : launch_rows<E32_DY1, false>(p, TK, vec, s);
}

int mts_f32_dw(const float* P, const int32_t* p_gather, const float* Q, const int32_t* q_gather, int M,
               int N, const int32_t* expert_start, int E, int grad_dtype, void* C, hipStream_t s) {
    const bool large = large_tiles((int64_t)E * M, N, 0);
    const int bt = large ? 128 : 64;
    Dw32 p = {P, p_gather, Q, q_gather, M, N, expert_start, E, C, (M + bt - 1) / bt, (N + bt - 1) / bt};
    const bool vec = M % 4 == 0 && N % 4 == 0 && mts_aligned16(P) && mts_aligned16(Q);
    const int64_t blocks = dw_blocks(p);
    if (blocks >= (1LL << 31)) return MTS_ERR_SHAPE;
    const dim3 grid((unsigned)blocks);
    auto launch = [&](auto* kind) {
        typedef typename std::remove_pointer<decltype(kind)>::type OutT;
        if (large && vec) dw_gemm_f32_kernel<128, 128, OutT, true><<<grid, kThreads, 0, s>>>(p);
        else if (large) dw_gemm_f32_kernel<128, 128, OutT, false><<<grid, kThreads, 0, s>>>(p);
        else if (vec) dw_gemm_f32_kernel<64, 64, OutT, true><<<grid, kThreads, 0, s>>>(p);
        else dw_gemm_f32_kernel<64, 64, OutT, false><<<grid, kThreads, 0, s>>>(p);
    };
    if (grad_dtype == MTS_F32) launch((float*)nullptr);
    else if (grad_dtype == MTS_BF16) launch((bf16_t*)nullptr);
    else if (grad_dtype == MTS_F16) launch((mts_f16_t*)nullptr);
    else return MTS_ERR_DTYPE;
    MTS_CHECK_LAUNCH();
    return MTS_OK;
}

extern "C" int mts_moe_bwd_joint_f32_supported(int H, int I) { return H >= 4 && I >= 4 && H % 4 == 0 && I % 4 == 0; }

extern "C" int mts_moe_bwd_joint_f32(const float* d_out, const float* weighted_act, const float* d_pre_act, const float* x, const float* w1, const int32_t* x_gather,
                                     const int32_t* expert_start, const int32_t* s_reverse, const float* ds_partial, int64_t T, int K, int E, int H, int I,
                                     float* dx_expanded, float* d_w1, float* d_w2, float* d_weights, void* stream) {
    if (!d_out || !weighted_act || !d_pre_act || !x || !w1 || !x_gather || !expert_start || !s_reverse || !ds_partial || !dx_expanded || !d_w1 || !d_w2 || !d_weights)
        return MTS_ERR_NULL;
    if (T <= 0 || K < 1 || T * K > 0x7fffffffLL || E < 1 || E > MTS_MAX_MOE_EXPERTS || !mts_moe_bwd_joint_f32_supported(H, I)) return MTS_ERR_SHAPE;
    if (!mts_aligned16(d_out) || !mts_aligned16(weighted_act) || !mts_aligned16(d_pre_act) || !mts_aligned16(x) || !mts_aligned16(w1)) return MTS_ERR_ALIGN;
    const int64_t TK = T * K;
    const bool large_dx = large_tiles(TK, H, E), large_dw = large_tiles((int64_t)E * 2 * I, H, 0);   // dW2's tiles follow dW1's
    const int bx = large_dx ? 128 : 64, bw = large_dw ? 128 : 64;
    Bwd32 q = {};
    q.dx = {d_pre_act, 2 * I, nullptr, w1, H, H, 2 * I, expert_start, E, dx_expanded, nullptr, nullptr, nullptr, nullptr, nullptr, 0, (H + bx - 1) / bx};
    q.dw1 = {d_pre_act, nullptr, x, x_gather, 2 * I, H, expert_start, E, d_w1, (2 * I + bw - 1) / bw, (H + bw - 1) / bw};
    q.dw2 = {d_out, x_gather, weighted_act, nullptr, H, I, expert_start, E, d_w2, (H + bw - 1) / bw, (I + bw - 1) / bw};
    const int64_t n_dx = (m_tiles32(TK, E, bx) * q.dx.n_tiles + kXcds - 1) / kXcds * kXcds, n_dw1 = dw_blocks(q.dw1), n_dw2 = dw_blocks(q.dw2);
    const int64_t want = (TK + kThreads - 1) / kThreads;
    q.n_ds = (int)(want < 64 ? want : 64);
    const int64_t blocks = n_dx + n_dw1 + n_dw2 + q.n_ds;
    if (blocks >= (1LL << 31)) return MTS_ERR_SHAPE;
    q.n_dx = (int)n_dx, q.n_dw1 = (int)n_dw1, q.n_dw2 = (int)n_dw2, q.per_dw1 = (int)(n_dw1 / E / kXcds), q.per_dw2 = (int)(n_dw2 / E / kXcds);
    q.ds_part = ds_partial, q.s_reverse = s_reverse, q.entries = TK, q.np = mts_moe_ds_partials(I), q.d_weights = d_weights;
    const dim3 grid((unsigned)blocks);
    hipStream_t s = (hipStream_t)stream;
    if (large_dx && large_dw) bwd_joint_f32_kernel<128, 128><<<grid, kThreads, 0, s>>>(q);
    else if (large_dx) bwd_joint_f32_kernel<128, 64><<<grid, kThreads, 0, s>>>(q);
    else if (large_dw) bwd_joint_f32_kernel<64, 128><<<grid, kThreads, 0, s>>>(q);
    else bwd_joint_f32_kernel<64, 64><<<grid, kThreads, 0, s>>>(q);
    MTS_CHECK_LAUNCH();
    return MTS_OK;
}
