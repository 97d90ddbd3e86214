// Forward expert GEMMs for few rows per expert (decoding, short sequences): y = W a, bound by reading the weights once.
//
// The 256 x 256 tiles of mts_gemm.hip leave most of the chip idle here (16 tokens, 8 experts of 768/1024: 64 and 24 blocks
// for 25 and 12.6 MB of weights, 1.5 and 0.9 TB/s).  Here a block owns 32 output columns (of gate and of up) for 16 * MT
// rows, its four waves split k and add their sums in LDS, and fragments go from memory to registers without LDS: a weight
// is used by one wave only.  The products are 16 x 16 x 32: a load then takes 64 consecutive bytes of 16 rows, where the
// 32 x 32 x 16 form takes 32 bytes of 32 and waits for the tags of twice to four times the lines.  All loads of up to DEPTH
// steps of 64 k are in flight before the first product.  fp32 weights are rounded on the way, as the cast in front of the
// large tiles does.  16 tokens, top-2 of 8 experts: gate/up 17.3 -> 11.6 us, down 14.6 -> 5.5; with fp32 weights 17.9 and 8.3,
// and no cast (20 us) in front.
#include "mts_few_block.h"

namespace {

using namespace mts_few;

struct FewRows {
    const void *A, *W;
    const int32_t *gather, *expert_start;   // gather NULL: rows of A are the sorted rows themselves
    int64_t a_rows;
    int E, N, K, n_tiles, m_tiles;
    void *C, *C2;
    const void* route_w;
    const int32_t* s_scatter;
};

// The m-th tile of `rows` rows, counted over the experts: expert and rows, or false behind the last one.  64 experts at a time.
__device__ __forceinline__ bool find_tile(const int32_t* start, int E, int m, int rows, int& expert, int& row0, int& end) {
    const int lane = threadIdx.x % MTS_WAVE;
    for (int e0 = 0; e0 < E; e0 += MTS_WAVE) {
        const int e = min(e0 + lane, E - 1);
        const int s = start[e], t = e0 + lane < E ? start[e + 1] : s;
        const int own = (t - s + rows - 1) / rows;
        const int upto = wave_scan(own);
        const uint64_t behind = __ballot(upto > m);
        if (behind) {
            const int l = __ffsll((unsigned long long)behind) - 1;
            expert = e0 + l;
            row0 = __builtin_amdgcn_readlane(s, l) + (m - __builtin_amdgcn_readlane(upto - own, l)) * rows;
            end = __builtin_amdgcn_readlane(t, l);
            return true;
        }
        m -= __builtin_amdgcn_readlane(upto, MTS_WAVE - 1);
    }
    return false;
}

template <typename ET, typename WT, bool SWIGLU, int MT>
__global__ __launch_bounds__(kThreads) void few_rows_kernel(FewRows p) {
    typedef typename Few<ET>::quad quad;
    constexpr int F = SWIGLU ? 2 : 1;                                // gate and up
    constexpr int STEP_REGS = 8 * (2 * F * (int)(sizeof(WT) / sizeof(ET)) + MT);
    constexpr int DEPTH = STEP_REGS > 64 ? 2 : (STEP_REGS > 32 ? 3 : 4);   // steps of 64 k in flight
    __shared__ f32x4 sums[kWaves][F][2][MT][MTS_WAVE];
    // the row tiles of one column range run on one XCD, one after the other: its weights come from that L2
    const int j = blockIdx.x / 8, nt = (j / p.m_tiles) * 8 + blockIdx.x % 8;
    int e, row0, end;
    if (nt >= p.n_tiles || !find_tile(p.expert_start, p.E, j % p.m_tiles, 16 * MT, e, row0, end)) return;
    const int lane = threadIdx.x % MTS_WAVE, wave = threadIdx.x / MTS_WAVE, n0 = nt * kCols;
    const uint32_t K = (uint32_t)p.K;
    const int w_rows = F * p.N;
    const __amdgpu_buffer_rsrc_t rw = operand((const WT*)p.W + (int64_t)e * w_rows * p.K, (int64_t)w_rows * p.K * sizeof(WT));
    const __amdgpu_buffer_rsrc_t ra = operand(p.A, p.a_rows * p.K * 2);
    bool col_in[2], row_in[MT];
    uint32_t wk[F][2], ak[MT];
#pragma unroll
    for (int c = 0; c < 2; ++c) {
        const int n = n0 + 16 * c + lane % 16;
        col_in[c] = n < p.N;
#pragma unroll
        for (int f = 0; f < F; ++f) wk[f][c] = (uint32_t)(f * p.N + n) * K;
    }
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
        const int row = row0 + 16 * mt + lane % 16;
        row_in[mt] = row < end;
        ak[mt] = (uint32_t)(row_in[mt] ? (p.gather ? p.gather[row] : row) : 0) * K;
    }
    const int steps = (p.K + 63) / 64, per = (steps + kWaves - 1) / kWaves;
    const int last = min(steps, (wave + 1) * per);
    f32x4 acc[F][2][MT] = {};
    for (int s0 = wave * per; s0 < last; s0 += DEPTH) {
        Chunk<ET, WT> w[DEPTH][2][F][2];
        Chunk<ET, ET> x[DEPTH][2][MT];
#pragma unroll
        for (int d = 0; d < DEPTH; ++d)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const uint32_t k = (uint32_t)(s0 + d) * 64 + 32 * h + 8 * (lane / 16);
                const bool in = s0 + d < last && k < K;
#pragma unroll
                for (int f = 0; f < F; ++f)
#pragma unroll
                    for (int c = 0; c < 2; ++c) w[d][h][f][c].load(rw, in && col_in[c] ? wk[f][c] + k : kOutside);
#pragma unroll
                for (int mt = 0; mt < MT; ++mt) x[d][h][mt].load(ra, in && row_in[mt] ? ak[mt] + k : kOutside);
            }
        __builtin_amdgcn_sched_barrier(0);   // the loads stay together in front
#pragma unroll
        for (int d = 0; d < DEPTH; ++d)
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int f = 0; f < F; ++f)
#pragma unroll
                    for (int c = 0; c < 2; ++c)
#pragma unroll
                        for (int mt = 0; mt < MT; ++mt) acc[f][c][mt] = Few<ET>::mul(w[d][h][f][c].frag(), x[d][h][mt].frag(), acc[f][c][mt]);
    }
#pragma unroll
    for (int f = 0; f < F; ++f)
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) sums[wave][f][c][mt][lane] = acc[f][c][mt];
    __syncthreads();
    // four consecutive columns of one row a thread
    for (int item = wave; item < 2 * MT; item += kWaves) {
        const int c = item % 2, mt = item / 2;
        const int row = row0 + 16 * mt + lane % 16, n = n0 + 16 * c + 4 * (lane / 16);
        if (row >= end || n >= p.N) continue;
        f32x4 v[F];
#pragma unroll
        for (int f = 0; f < F; ++f) {
            v[f] = sums[0][f][c][mt][lane];
#pragma unroll
            for (int k = 1; k < kWaves; ++k)
#pragma unroll
                for (int r = 0; r < 4; ++r) v[f][r] += sums[k][f][c][mt][lane][r];
        }
        if constexpr (SWIGLU) {
            const float s = p.route_w ? (float)((const ET*)p.route_w)[p.s_scatter[row]] : 1.f;
            quad g, u, a;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                g[r] = (ET)v[0][r], u[r] = (ET)v[1][r];
                a[r] = (ET)(v[0][r] * __builtin_amdgcn_rcpf(1.0f + __expf(-v[0][r])) * v[1][r] * s);
            }
            if (p.C) {
                ET* pre = (ET*)p.C + (int64_t)row * 2 * p.N + n;
                *reinterpret_cast<quad*>(pre) = g;
                *reinterpret_cast<quad*>(pre + p.N) = u;
            }
            *reinterpret_cast<quad*>((ET*)p.C2 + (int64_t)row * p.N + n) = a;
        } else {
            quad y;
#pragma unroll
            for (int r = 0; r < 4; ++r) y[r] = (ET)v[0][r];
            *reinterpret_cast<quad*>((ET*)p.C + (int64_t)row * p.N + n) = y;
        }
    }
}

// rows of a block's tile, in sixteens: what an expert has on average
int row_tiles(int64_t TK, int E) { return TK <= 16LL * E ? 1 : (TK <= 32LL * E ? 2 : 4); }

template <typename ET, typename WT, bool SWIGLU>
int launch_few(FewRows p, int64_t TK, hipStream_t st) {
    const int mt = row_tiles(TK, p.E);
    const int64_t tiles = TK / (16 * mt) + p.E, most = tiles < TK ? tiles : TK;
    p.n_tiles = (p.N + kCols - 1) / kCols;
    p.m_tiles = (int)most;
    const dim3 grid((unsigned)((p.n_tiles + 7) / 8 * 8 * most));
    if (mt == 4) few_rows_kernel<ET, WT, SWIGLU, 4><<<grid, kThreads, 0, st>>>(p);
    else if (mt == 2) few_rows_kernel<ET, WT, SWIGLU, 2><<<grid, kThreads, 0, st>>>(p);
    else few_rows_kernel<ET, WT, SWIGLU, 1><<<grid, kThreads, 0, st>>>(p);
    MTS_CHECK_LAUNCH();
    return MTS_OK;
}

template <typename ET, typename WT>
int launch_pair(const FewRows& up, const FewRows& down, int64_t TK, hipStream_t st) {
    const int rc = launch_few<ET, WT, true>(up, TK, st);
    return rc ? rc : launch_few<ET, WT, false>(down, TK, st);
}

}  // namespace

extern "C" int mts_moe_fwd_few_rows_supported(int act_dtype, int weight_dtype, int64_t T, int64_t TK, int E, int H, int I) {
    if (act_dtype != MTS_BF16 && act_dtype != MTS_F16) return 0;
    if (weight_dtype != act_dtype && weight_dtype != MTS_F32) return 0;
    if (T <= 0 || TK <= 0 || E < 1 || E > MTS_MAX_MOE_EXPERTS || H < 8 || I < 8 || H % 8 || I % 8) return 0;
    const int64_t most = 1LL << 31, wb = weight_dtype == MTS_F32 ? 4 : 2;   // 32-bit byte offsets
    if (T * H * 2 >= most || TK * I * 2 >= most || 2LL * I * H * wb >= most) return 0;
    const int64_t wide = H > I ? H : I;
    return ((wide + kCols - 1) / kCols + 7) / 8 * 8 * (TK / 16 + E) * kThreads < (1LL << 32);
}

// Against the tiles, in us.  What this path does more: for 2^20 weights an expert's first 8 rows read the activations for every 32 columns, 0.2, and so does every further
// 16 of them.  What it does less: the tiles' down projection is one chain over I where four waves share it here, 1 for 256 of I; and their rounds behind
// the first, of 256 CUs with 128 columns of gate and up or 256 of the down projection each, cost 6 for 256 of k.  With fp32 weights the tiles want rounded copies as well: a
// launch in front, 7, and the time that more than 21 M weights take at the rate of memory, 1 a M.  Beside the head they are made while it runs, which hides 9 more of them.
// Placed on 1800 calls, each with three sets of weights in turn and with as many as the caches do not hold (512 to 2048 by 256 to 2048, 4 to 128 experts, 3 to 210 M
// weights, 1.4 to 64 rows an expert, routes evenly spread and not, the operator and the layer): behind the better path by 0.6 % on average (copies in front 0.5 %), furthest
// by 15 to 19 %.  On 500 calls that had no part in it 0.4 to 1.2 %, up to 30 %.  Here / there: layer, fp32, 8 experts of 768/1024 with one
// route a token, 65 tokens 43.9 / 44.7, 80 47.5 / 44.4, 128 48.2 / 45.0; 16 of 1024/768 10 rows 60.5 / 71.9; 128 of 512/1024 9 rows 193 / 371; 64 of 768/512
// 39 rows 121 / 124; operator, fp32, 8 of 768/768 36 rows 29 / 38; 16 of 1024/1536 50 rows 105 / 134; 16 of 512/512 57 rows 38 / 35; 16 bits, 16 of 1024/768 11 rows
// 54 / 45 (layer), 64 of 768/1000 2 rows 73 / 84, 16 of 2048/1024 5 rows 57 / 49 (operator), 4 of 1024/1024 23 rows 35 / 37 (layer).
enum { MASTERS_NONE, MASTERS_COPIED_IN_FRONT, MASTERS_COPIED_BESIDE_HEAD };
static int few_rows_ahead(int masters, int64_t TK, int E, int H, int I) {
    auto beyond = [](double value, double border) { return value > border ? value - border : 0.0; };
    const double weights = 3.0 * E * H * I / (1 << 20), rows = (double)TK / E, chain = I / 256.0;
    double there = 0.0;
    if (masters == MASTERS_NONE) there = 2.0 + chain + 6.0 * (beyond(E * (I / 128.0) / 256, 1.0) * H / 256 + beyond(E * (H / 256.0) / 256, 1.0) * chain);
    if (masters == MASTERS_COPIED_IN_FRONT) there = 7.0 + chain + beyond(weights, 21.0);
    if (masters == MASTERS_COPIED_BESIDE_HEAD) there = 0.75 + 0.75 * chain + beyond(weights, 30.0);
    return rows <= 64.0 && weights * 0.2 * ((rows < 8.0 ? rows : 8.0) / 8 + beyond(rows, 8.0) / 16) <= there;   // more rows: not measured
}
extern "C" int mts_moe_fwd_few_rows_preferred(int act_dtype, int weight_dtype, int64_t T, int64_t TK, int E, int H, int I) {
    return mts_moe_fwd_few_rows_supported(act_dtype, weight_dtype, T, TK, E, H, I) &&
           few_rows_ahead(weight_dtype == MTS_F32 ? MASTERS_COPIED_IN_FRONT : MASTERS_NONE, TK, E, H, I);
}
extern "C" int mts_moe_fwd_few_rows_preferred_to_ride(int act_dtype, int64_t T, int64_t TK, int E, int H, int I) {
    return mts_moe_fwd_few_rows_supported(act_dtype, MTS_F32, T, TK, E, H, I) && few_rows_ahead(MASTERS_COPIED_BESIDE_HEAD, TK, E, H, I);
}

extern "C" int mts_moe_fwd_few_rows(const void* x, const void* w1, const void* w2, int weight_dtype, const int32_t* x_gather, const int32_t* expert_start,
                                    const void* weights, const int32_t* s_scatter, int64_t T, int K, int E, int H, int I, int act_dtype, void* pre_act,
                                    void* post_act, void* y, void* stream) {
    if (!x || !w1 || !w2 || !x_gather || !expert_start || !post_act || !y) return MTS_ERR_NULL;
    if ((weights != nullptr) != (s_scatter != nullptr)) return MTS_ERR_NULL;
    if (K < 1 || !mts_moe_fwd_few_rows_supported(act_dtype, weight_dtype, T, T * K, E, H, I)) return MTS_ERR_SHAPE;
    if (!mts_aligned16(x) || !mts_aligned16(w1) || !mts_aligned16(w2) || !mts_aligned16(pre_act) || !mts_aligned16(post_act) || !mts_aligned16(y))
        return MTS_ERR_ALIGN;
    FewRows up = {}, down = {};
    up.A = x, up.W = w1, up.gather = x_gather, up.a_rows = T, up.N = I, up.K = H, up.C = pre_act, up.C2 = post_act;
    up.route_w = weights, up.s_scatter = s_scatter;
    down.A = post_act, down.W = w2, down.a_rows = T * K, down.N = H, down.K = I, down.C = y;
    up.expert_start = down.expert_start = expert_start, up.E = down.E = E;
    hipStream_t st = (hipStream_t)stream;
    if (act_dtype == MTS_BF16)
        return weight_dtype == MTS_F32 ? launch_pair<bf16_t, float>(up, down, T * K, st) : launch_pair<bf16_t, bf16_t>(up, down, T * K, st);
    return weight_dtype == MTS_F32 ? launch_pair<mts_f16_t, float>(up, down, T * K, st) : launch_pair<mts_f16_t, mts_f16_t>(up, down, T * K, st);
}
