// fp32 variant of the grouped expert GEMMs: activations, weights and accumulation all in fp32, on the fp32 matrix
// instruction (v_mfma_f32_32x32x2_f32, full fp32 products and sums).  Same contracts and epilogues as the 16-bit kernels.
//
// What bounds it: the instruction's rate, 157 TFLOP/s on the card (64 cycles for 4096 FLOP), a sixteenth of the bf16 rate,
// so nothing here needs direct-to-LDS loads or specialised waves: tiles of 64 x 64 outputs per block of four waves, 16 of k
// at a time through two LDS buffers, two more k-tiles in flight in registers, and up to eight blocks per CU.  A tile reads
// one byte of L2 per 16 FLOP; tiles of 128 rows are no faster at 16 000 rows (101 TFLOP/s over all GEMMs either way) and
// 12 % slower at 4096, where they leave the CUs unevenly filled.  2048 tokens, 768/1024, 8 experts, top-2: forward and
// backward of the operator 1776 -> 727 us, 80 TFLOP/s (plain FMA from 64x64 tiles before: 33 TFLOP/s).
#include "mts_f32_tiles.h"

#include <type_traits>

namespace {

using namespace mts_f32;

constexpr int BM = 64;   // rows of a tile, and of P columns in the weight gradients
constexpr int kThreads = kTileThreads;
constexpr int kXcds = 8;
constexpr int TKS = 16;  // k extent of an LDS tile

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
__device__ __forceinline__ int find_m_tile(const int32_t* __restrict__ expert_start, int E, int tile, int& e_out, int& row0, int& rend) {
    const int lane = threadIdx.x % MTS_WAVE;
    int seen = 0;
    for (int e0 = 0; e0 < E; e0 += MTS_WAVE) {
        const int e = e0 + lane;
        const int s0 = e < E ? expert_start[e] : 0, s1 = e < E ? expert_start[e + 1] : 0;
        const int nt = (s1 - s0 + BM - 1) / BM;
        int upto = nt;
#pragma unroll
        for (int o = 1; o < MTS_WAVE; o <<= 1) {
            const int t = __shfl_up(upto, o, MTS_WAVE);
            if (lane >= o) upto += t;
        }
        const uint64_t mine = __ballot(tile >= seen + upto - nt && tile < seen + upto);
        if (mine) {
            const int l = __ffsll((unsigned long long)mine) - 1;
            e_out = e0 + l;
            row0 = __shfl(s0, l, MTS_WAVE) + (tile - seen - __shfl(upto - nt, l, MTS_WAVE)) * BM;
            rend = __shfl(s1, l, MTS_WAVE);
        }
        seen += __shfl(upto, MTS_WAVE - 1, MTS_WAVE);
    }
    return seen;
}

// BN counts the columns of the B tile (SwiGLU: gate and up columns side by side, half the outputs)
template <int BN, int EPI, bool BKM, bool VEC>
__global__ __launch_bounds__(kThreads) void rows_gemm_f32_kernel(Rows32 p) {
    constexpr int WAVES_M = 2, WAVES_N = 2;
    constexpr int MF = BM / WAVES_M / 32, NF = BN / WAVES_N / 32;
    constexpr int OUT_N = EPI == E32_SWIGLU ? BN / 2 : BN;
    typedef RowTile<float, BM, TKS, VEC> ATile;
    typedef typename std::conditional<BKM, KTile<float, BN, TKS, VEC>, RowTile<float, BN, TKS, VEC>>::type BTile;
    __shared__ __attribute__((aligned(16))) float As[2][ATile::SIZE];
    __shared__ __attribute__((aligned(16))) float Bs[2][BTile::SIZE];
    __shared__ float ds_sum[EPI == E32_DY1 ? WAVES_N : 1][BM];

    // block b runs on XCD b % 8: every XCD takes an equal contiguous run of the tiles, columns fastest, so that an expert's
    // weights stream through one L2 and the blocks that share activation rows are neighbours in time
    int e = 0, row0 = 0, rend = 0;
    const int total = find_m_tile(p.expert_start, p.E, -1, e, row0, rend) * p.n_tiles;
    const int per_xcd = (total + kXcds - 1) / kXcds, slot = blockIdx.x / kXcds;
    const int tile = (blockIdx.x % kXcds) * per_xcd + slot;
    if (slot >= per_xcd || tile >= total) return;
    find_m_tile(p.expert_start, p.E, tile / p.n_tiles, e, row0, rend);
    const int ny = tile % p.n_tiles, n0 = ny * OUT_N;

    ATile a;
#pragma unroll
    for (int q = 0; q < ATile::LOADS; ++q) {
        const int r = row0 + ATile::row(q);
        a.ptr[q] = r < rend ? p.A + (int64_t)(p.a_gather ? p.a_gather[r] : r) * p.lda : nullptr;
    }
    const float* Be = p.B + (int64_t)e * p.b_rows * p.Kdim;
    BTile b;
    if constexpr (BKM) {
        b.base = Be + n0 + BTile::col();
        b.ld = p.N;
        b.cols = p.N - n0 - BTile::col();
    } else {
#pragma unroll
        for (int q = 0; q < BTile::LOADS; ++q) {
            const int r = BTile::row(q), half = r / OUT_N, n = n0 + r % OUT_N;
            b.ptr[q] = n < p.N ? Be + (int64_t)(half * p.N + n) * p.Kdim : nullptr;
        }
    }
    auto fetch = [&](int set, int t) {
        a.fetch(set, t * TKS, p.Kdim);
        if constexpr (BKM) {
            int64_t rows[BTile::LOADS];
#pragma unroll
            for (int q = 0; q < BTile::LOADS; ++q) rows[q] = t * TKS + BTile::k(q) < p.Kdim ? t * TKS + BTile::k(q) : -1;
            b.fetch(set, rows);
        } else b.fetch(set, t * TKS, p.Kdim);
    };

    const int wave = threadIdx.x / MTS_WAVE, wm = wave / WAVES_N, wn = wave % WAVES_N, lane = threadIdx.x % MTS_WAVE;
    auto a_at = [&](int mf) { return wm * (BM / WAVES_M) + mf * 32; };
    auto b_at = [&](int nf) { return EPI == E32_SWIGLU ? nf / (NF / 2) * OUT_N + wn * (OUT_N / WAVES_N) + nf % (NF / 2) * 32 : wn * (BN / WAVES_N) + nf * 32; };
    f32x16 acc[MF][NF] = {};
    const int tiles = (p.Kdim + TKS - 1) / TKS;
    run_k_tiles<ATile, BTile, TKS / 8, MF, NF>(tiles, a, b, As, Bs, acc, a_at, b_at, fetch);

#pragma unroll
    for (int mf = 0; mf < MF; ++mf)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const int r = a_at(mf) + 8 * (i / 4) + 4 * (lane / 32) + i % 4;
            const int row = row0 + r;
            const bool rok = row < rend;
            if constexpr (EPI == E32_PLAIN) {
#pragma unroll
                for (int nf = 0; nf < NF; ++nf) {
                    const int n = n0 + b_at(nf) + lane % 32;
                    if (rok && n < p.N) p.C[(int64_t)row * p.N + n] = acc[mf][nf][i];
                }
            } else if constexpr (EPI == E32_SWIGLU) {
                const float s = (rok && p.route_w) ? p.route_w[p.s_scatter[row]] : 1.f;   // post_act may carry the routing weight
#pragma unroll
                for (int nf = 0; nf < NF / 2; ++nf) {
                    const int n = n0 + b_at(nf) + lane % 32;
                    if (!rok || n >= p.N) continue;
                    const float g = acc[mf][nf][i], u = acc[mf][nf + NF / 2][i];
                    p.C[(int64_t)row * (2 * p.N) + n] = g;
                    p.C[(int64_t)row * (2 * p.N) + p.N + n] = u;
                    p.C2[(int64_t)row * p.N + n] = g * sigmoid32(g) * u * s;
                }
            } else {
                const float s = rok ? p.route_w[p.s_scatter[row]] : 0.f;
                float dsp = 0.f;
#pragma unroll
                for (int nf = 0; nf < NF; ++nf) {
                    const int n = n0 + b_at(nf) + lane % 32;
                    if (!rok || n >= p.N) continue;
                    const int64_t o = (int64_t)row * (2 * p.N) + n;
                    const float g = p.pre_act[o], u = p.pre_act[o + p.N];
                    const float v = acc[mf][nf][i];
                    const float sig = sigmoid32(g);
                    const float silu = g * sig;
                    const float y1 = silu * u;
                    dsp += v * y1;
                    if (p.C2) p.C2[(int64_t)row * p.N + n] = s * y1;
                    const float da = v * s;
                    p.C[o] = da * (silu * (1.0f - sig) + sig) * u;
                    p.C[o + p.N] = da * silu;
                }
#pragma unroll
                for (int o = 16; o > 0; o >>= 1) dsp += __shfl_xor(dsp, o, 32);
                if (lane % 32 == 0) ds_sum[wn][r] = dsp;
            }
        }
    if constexpr (EPI == E32_DY1) {   // row sums over the tile's 64 columns
        __syncthreads();
        for (int r = threadIdx.x; r < BM; r += kThreads)
            if (row0 + r < rend) {
                float v = ds_sum[0][r];
#pragma unroll
                for (int q = 1; q < WAVES_N; ++q) v += ds_sum[q][r];
                p.ds_part[(int64_t)(row0 + r) * p.np + ny] = v;
            }
    }
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

// 64 x 64 outputs; the reduction runs over the expert's rows, both operands k-major
template <typename OutT, bool VEC>
__global__ __launch_bounds__(kThreads) void dw_gemm_f32_kernel(Dw32 p) {
    constexpr int BN = 64, MF = BM / 64, NF = 1;
    typedef KTile<float, BM, TKS, VEC> PT;
    typedef KTile<float, BN, TKS, VEC> QT;
    __shared__ __attribute__((aligned(16))) float Ps[2][PT::SIZE];
    __shared__ __attribute__((aligned(16))) float Qs[2][QT::SIZE];
    // an XCD takes an equal contiguous run of every expert's tiles, columns fastest: an equal share of the work however
    // uneven the experts are, and about an eighth of P through its L2
    const int per_expert = p.m_tiles * p.n_tiles, per_xcd = (per_expert + kXcds - 1) / kXcds;
    const int slot = blockIdx.x / kXcds, e = slot / per_xcd;
    const int tile = (blockIdx.x % kXcds) * per_xcd + slot % per_xcd;
    if (tile >= per_expert || e >= p.E) return;
    const int m0 = tile / p.n_tiles * BM, n0 = tile % p.n_tiles * BN;
    const int rbeg = p.expert_start[e], rend = p.expert_start[e + 1];

    PT a;
    QT b;
    a.base = p.P + m0 + PT::col(), a.ld = p.M, a.cols = p.M - m0 - PT::col();
    b.base = p.Q + n0 + QT::col(), b.ld = p.N, b.cols = p.N - n0 - QT::col();
    int64_t pr[PT::LOADS], qr[QT::LOADS];   // memory rows of the k-tile to fetch next: read a tile ahead of its data
    auto locate = [&](int r0) {
#pragma unroll
        for (int q = 0; q < PT::LOADS; ++q) {
            const int r = r0 + PT::k(q);
            pr[q] = r < rend ? (p.p_gather ? p.p_gather[r] : r) : -1;
        }
#pragma unroll
        for (int q = 0; q < QT::LOADS; ++q) {
            const int r = r0 + QT::k(q);
            qr[q] = r < rend ? (p.q_gather ? p.q_gather[r] : r) : -1;
        }
    };
    const int wave = threadIdx.x / MTS_WAVE, wm = wave / 2, wn = wave % 2, lane = threadIdx.x % MTS_WAVE;
    auto a_at = [&](int mf) { return wm * (BM / 2) + mf * 32; };
    auto b_at = [&](int) { return wn * (BN / 2); };
    f32x16 acc[MF][NF] = {};
    locate(rbeg);
    auto fetch = [&](int set, int t) {
        a.fetch(set, pr);
        b.fetch(set, qr);
        locate(rbeg + (t + 1) * TKS);
    };
    const int tiles = (rend - rbeg + TKS - 1) / TKS;
    run_k_tiles<PT, QT, TKS / 8, MF, NF>(tiles, a, b, Ps, Qs, acc, a_at, b_at, fetch);

    OutT* C = reinterpret_cast<OutT*>(p.C) + (int64_t)e * p.M * p.N;
    const int n = n0 + b_at(0) + lane % 32;
#pragma unroll
    for (int mf = 0; mf < MF; ++mf)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const int m = m0 + a_at(mf) + 8 * (i / 4) + 4 * (lane / 32) + i % 4;
            if (m < p.M && n < p.N) C[(int64_t)m * p.N + n] = (OutT)acc[mf][0][i];
        }
}

int64_t m_tiles32(int64_t TK, int E) {
    const int64_t a = (TK + BM - 1) / BM + E - 1;
    return a < TK ? a : TK;
}

template <int EPI, bool BKM>
int launch_rows(Rows32 p, int64_t TK, bool vec, hipStream_t s) {
    constexpr int BN = EPI == E32_SWIGLU ? 128 : 64, OUT_N = 64;
    p.n_tiles = (p.N + OUT_N - 1) / OUT_N;
    const int64_t blocks = (m_tiles32(TK, p.E) * p.n_tiles + kXcds - 1) / kXcds * kXcds;
    if (blocks >= (1LL << 31)) return MTS_ERR_SHAPE;
    const dim3 grid((unsigned)blocks);
    if (vec) rows_gemm_f32_kernel<BN, EPI, BKM, true><<<grid, kThreads, 0, s>>>(p);
    else rows_gemm_f32_kernel<BN, EPI, BKM, false><<<grid, kThreads, 0, s>>>(p);
    MTS_CHECK_LAUNCH();
    return MTS_OK;
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
    Dw32 p = {P, p_gather, Q, q_gather, M, N, expert_start, E, C, (M + BM - 1) / BM, (N + 63) / 64};
    const bool vec = M % 4 == 0 && N % 4 == 0 && mts_aligned16(P) && mts_aligned16(Q);
    const int64_t blocks = ((int64_t)p.m_tiles * p.n_tiles + kXcds - 1) / kXcds * kXcds * E;
    if (blocks >= (1LL << 31)) return MTS_ERR_SHAPE;
    const dim3 grid((unsigned)blocks);
    auto launch = [&](auto* kind) {
        typedef typename std::remove_pointer<decltype(kind)>::type OutT;
        if (vec) dw_gemm_f32_kernel<OutT, true><<<grid, kThreads, 0, s>>>(p);
        else dw_gemm_f32_kernel<OutT, false><<<grid, kThreads, 0, s>>>(p);
    };
    if (grad_dtype == MTS_F32) launch((float*)nullptr);
    else if (grad_dtype == MTS_BF16) launch((bf16_t*)nullptr);
    else if (grad_dtype == MTS_F16) launch((mts_f16_t*)nullptr);
    else return MTS_ERR_DTYPE;
    MTS_CHECK_LAUNCH();
    return MTS_OK;
}
