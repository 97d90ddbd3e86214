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

// Against the tiles, in us.  What this path does more, for 2^20 weights: every 16 rows of an expert behind the first 16 (half of them, on average) read the
// activations again for every 32 columns, 0.2; and more blocks start, 0.025.  What it does less: the tiles' down projection is one chain over I where four
// waves share it here, 1 for 256 of I; and a routing of up to 64 tokens is one launch, behind which this path has the shorter start, 1.  With fp32 weights the
// tiles want rounded copies as well: a launch in front, 6, and the time that more than 27 M weights take at the rate of memory, 1 a M.  Beside the head they
// are made while it runs: its launches cover 6 of that with up to 16 experts, 20 with more.
// Placed on 140 shapes and tried on 60 others (512 to 2048 by 256 to 2048, 3 to 128 experts, 3 to 200 M weights, 2 to 80 rows an expert, the operator and the
// layer, weights not in the caches): on those the call is behind the better path by 0.2 % (fp32), 0.4 % (16 bits, layer) and 1.0 % (operator) on average; furthest
// with 80 experts and 2 rows, of whom many have none (776/640, 16 bits 72 / 95).  Here / there:
// operator, fp32, 768/1024, 8 experts, 16 rows 40 / 45, 32 rows 45 / 45, 64 rows 59 / 46; 128 experts of 768/256, 8 rows 86 / 135, 32 rows 130 / 138, 64 rows
// 176 / 148; layer, fp32, 64 experts of 1024/512 32 rows 153 / 168, 64 rows 192 / 170; 8 of 768/1024, 16 rows 49 / 57 (64 tokens), 32 rows 59 / 51; 32 of 768/256
// 8 rows 54 / 53, 16 rows 62 / 54; 16 bits, 8 of 768/1024 16 rows 39 / 42, 32 rows 48 / 44; 512/2048 32 rows 51 / 51, 64 rows 67 / 52.
enum { MASTERS_NONE, MASTERS_COPIED_IN_FRONT, MASTERS_COPIED_BESIDE_HEAD };
static int few_rows_ahead(int masters, int64_t T, int64_t TK, int E, int H, int I) {
    const double weights = 3.0 * E * H * I / (1 << 20), rows = (double)TK / E, again = rows > 8 ? rows / 16 - 0.5 : 0.0;
    double there = I / 256.0 + (T <= 64 ? 1.0 : 0.0);
    if (masters != MASTERS_NONE) there += weights > 33.0 ? weights - 27.0 : 6.0;
    if (masters == MASTERS_COPIED_BESIDE_HEAD) there -= E <= 16 ? 6.0 : 20.0;
    return rows <= 64.0 && weights * (0.2 * again + 0.025) <= there;   // more rows: not measured
}
extern "C" int mts_moe_fwd_few_rows_preferred(int act_dtype, int weight_dtype, int64_t T, int64_t TK, int E, int H, int I) {
    return mts_moe_fwd_few_rows_supported(act_dtype, weight_dtype, T, TK, E, H, I) &&
           few_rows_ahead(weight_dtype == MTS_F32 ? MASTERS_COPIED_IN_FRONT : MASTERS_NONE, T, TK, E, H, I);
}
extern "C" int mts_moe_fwd_few_rows_preferred_to_ride(int act_dtype, int64_t T, int64_t TK, int E, int H, int I) {
    return mts_moe_fwd_few_rows_supported(act_dtype, MTS_F32, T, TK, E, H, I) && few_rows_ahead(MASTERS_COPIED_BESIDE_HEAD, T, TK, E, H, I);
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
