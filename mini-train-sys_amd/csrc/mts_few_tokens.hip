// Forward pass of the whole layer for few tokens (decoding): two launches, the second summing a token's routes.
//
// Such a call is a chain of latencies.  As head, gate/up, down and combine (mts_router_linear.hip, mts_few_rows.hip, mts_combine.hip) it was four launches of
// 9.3, 10.4, 5.4 and 3.0 us (16 tokens, 8 experts of 768/1024), each of two or three trips to memory, the weights waiting for the routing; and the host
// spends as long on four launches.  Here
//  * a block of the first launch belongs to an expert and 32 columns of its gate and up, whatever the routing: its weights are on their way while it works
//    the routing out for itself (48 fp32 matrix instructions a wave for a tile of 16 tokens at 768 columns, whose operands lie in the L2s), and they are
//    multiplied with all tokens, 16 a tile, as a tile of fewer costs the same.  The routing says which of the products are stored, and where.  One
//    block leaves the router's results and the routing metadata, and clears the counters of the second launch;
//  * a block of the second launch takes 32 columns of the down projection of ONE expert and writes its rows of y to memory.  It then counts itself at its range of
//    columns; the block that arrives there last, of those of the experts with rows, reads the rows again and adds the tokens' routes, each rounded as a row
//    of the down projection is.  Rows and counter pass between the XCDs, which few_tokens_down_kernel says how they may.
// The products are the same sums in the same order as those of mts_few_rows.hip; the logits are the fp32 instruction's in four parts.  16 tokens, 8 experts of
// 768/1024: 28.1 us of kernels in four launches, 13.9 + 7.7 in two (1.8 TB/s of weights in both); 31.6 -> 23.9 us a call.
#include "mts_few_block.h"
#include "mts_router_row.h"

namespace {

using namespace mts_few;
using namespace mts_router;

constexpr int kMostExperts = 16;   // rows of the projection's tile
constexpr int kTokens = 16;        // a tile of tokens

struct FewTokens {
    const void* x;
    const float* w_r;
    const void *w1, *w2;
    int64_t T;
    int H, E, I, K, normalize, act_dtype, n_tiles;
    int extra;   // the first block has no columns
    int eager;   // the weights are asked for before the routing is known
    float inv_t, inv_routes;
    float *logits, *weights;
    int32_t* indices;
    void* weights_act;
    float *prob_mean, *z_loss, *entropy;
    int32_t* counts;
    float *load_balance, *load_stats;
    int32_t *expert_start, *s_scatter, *s_reverse, *x_gather;
    void *pre_act, *post_act, *y, *out;
    int32_t* arrived;   // a counter for every range of columns of the down projection
};

// The router's results and the routing metadata, by one block: lane t of its first wave holds the post-process of token t.
template <int EP>
__device__ __forceinline__ void leave_routing(const FewTokens& p, const RowState<EP, 1>& rs, const int (&sel_e)[MTS_MAX_TOP_K], const float (&sel_w)[MTS_MAX_TOP_K],
                                              bool live, int wave, int lane) {
    __shared__ StatsOf<kMostExperts> sh;
    for (int i = threadIdx.x; i * kCols < p.H; i += kThreads) p.arrived[i] = 0;
    if (wave == 0) {
        int64_t t = lane;
        float zsum = 0.f, hsum = 0.f, mine = 0.f;
        int routes = 0, start = 0;
#pragma unroll
        for (int e = 0; e < EP; ++e) {
            const float lp = fmaxf(rs.l[e] - rs.L, kLogFloor);
            hsum -= (live && rs.p[e] > 0.f) ? rs.p[e] * lp : 0.f;
            if (live && e < p.E) p.logits[t * p.E + e] = rs.l[e];
        }
        if (live) zsum = rs.L * rs.L;
        if (live) {
#pragma unroll
            for (int k = 0; k < MTS_MAX_TOP_K; ++k)
                if (k < p.K) {
                    p.weights[t * p.K + k] = sel_w[k];
                    p.indices[t * p.K + k] = sel_e[k];
                    if (p.act_dtype == MTS_BF16) reinterpret_cast<bf16_t*>(p.weights_act)[t * p.K + k] = (bf16_t)sel_w[k];
                    else reinterpret_cast<mts_f16_t*>(p.weights_act)[t * p.K + k] = (mts_f16_t)sel_w[k];
                }
        }
        // a token has at most one route to an expert: rows in token order are rows in entry order
#pragma unroll
        for (int e = 0; e < EP; ++e) {
            int entry = -1;
#pragma unroll
            for (int k = 0; k < MTS_MAX_TOP_K; ++k)
                if (k < p.K && sel_e[k] == e) entry = (int)t * p.K + k;
            const uint64_t here = __ballot(live && entry >= 0);
            if (live && entry >= 0) {
                const int row = start + __popcll(here & lanemask_lt());
                p.s_reverse[entry] = row;
                p.s_scatter[row] = entry;
                p.x_gather[row] = (int)t;
            }
            if (lane == 0 && e < p.E) p.expert_start[e] = start;
            const float mass = wave_sum(live ? rs.p[e] : 0.f);
            if (lane == e) mine = mass, routes = (int)__popcll(here);
            start += (int)__popcll(here);
        }
        if (lane == 0) p.expert_start[p.E] = start;
        zsum = wave_sum(zsum);
        hsum = wave_sum(hsum);
        if (lane == p.E) mine = zsum;
        if (lane == p.E + 1) mine = hsum;
        if (lane < p.E + 2) stats_column(sh, lane, mine * p.inv_t, routes, p.E, p.inv_routes, p.prob_mean, p.z_loss, p.entropy, p.counts);
    }
    __syncthreads();
    stats_finalize(sh, wave, 1, 2, p.E, p.load_balance, p.load_stats);
}

// MT tiles of 16 tokens.  EP: 8 or 16, the experts rounded up.
template <typename ET, typename WT, int MT, int EP>
__global__ __launch_bounds__(kThreads, 2) void few_tokens_up_kernel(FewTokens p) {
    typedef typename Few<ET>::quad quad;
    constexpr int STEP_REGS = 8 * (4 * (int)(sizeof(WT) / sizeof(ET)) + MT);
    constexpr int DEPTH = STEP_REGS > 64 || MT > 1 || EP > 8 ? 2 : 3;   // steps of 64 k in flight
    constexpr bool WIDE = sizeof(WT) > sizeof(ET);
    constexpr int HEAD = MT > 1 || (WIDE && EP > 8) ? 1 : EP > 8 || WIDE ? 2 : 3;           // those of the projection
    __shared__ f32x4 sums[kWaves][2][2][MT][MTS_WAVE];
    __shared__ f32x4 parts[kWaves][MT][MTS_WAVE];
    const int lane = threadIdx.x % MTS_WAVE, wave = threadIdx.x / MTS_WAVE;
    const bool router = blockIdx.x == 0, alone = router && p.extra;
    const int tile = (int)blockIdx.x - p.extra, e = alone ? 0 : tile / p.n_tiles, n0 = alone ? p.I : tile % p.n_tiles * kCols;
    const uint32_t H = (uint32_t)p.H;
    const int T = (int)p.T;
    const __amdgpu_buffer_rsrc_t rx = operand(p.x, p.T * p.H * 2), rr = operand(p.w_r, (int64_t)p.E * p.H * 4);
    const __amdgpu_buffer_rsrc_t rw = operand((const WT*)p.w1 + (int64_t)e * 2 * p.I * p.H, (int64_t)2 * p.I * p.H * sizeof(WT));
    const int steps = (p.H + 63) / 64, per = (steps + kWaves - 1) / kWaves;
    const int first = wave * per, last = min(steps, first + per);
    bool col_in[2], tok_in[MT];
    uint32_t wk[2][2], xk[MT];
#pragma unroll
    for (int c = 0; c < 2; ++c) {
        const int n = n0 + 16 * c + lane % 16;
        col_in[c] = n < p.I;
#pragma unroll
        for (int f = 0; f < 2; ++f) wk[f][c] = (uint32_t)(f * p.I + n) * H;
    }
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
        const int t = kTokens * mt + lane % 16;
        tok_in[mt] = t < T;
        xk[mt] = (uint32_t)(tok_in[mt] ? t : 0) * H;
    }
    const bool expert_in = lane % 16 < p.E;
    const uint32_t rk = (uint32_t)(lane % 16) * H;

    Chunk<ET, WT> w[DEPTH][2][2][2];
    Chunk<ET, ET> x[DEPTH][2][MT];
    auto ask = [&](int s0, bool wanted) {
#pragma unroll
        for (int d = 0; d < DEPTH; ++d)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const uint32_t k = (uint32_t)(s0 + d) * 64 + 32 * h + 8 * (lane / 16);
                const bool in = wanted && s0 + d < last && k < H;
#pragma unroll
                for (int f = 0; f < 2; ++f)
#pragma unroll
                    for (int c = 0; c < 2; ++c) w[d][h][f][c].load(rw, in && col_in[c] ? wk[f][c] + k : kOutside);
#pragma unroll
                for (int mt = 0; mt < MT; ++mt) x[d][h][mt].load(rx, in && tok_in[mt] ? xk[mt] + k : kOutside);
            }
    };

    // The projection: rows are experts, columns tokens, and a lane's eight consecutive k those of eight instructions.  The loads of its last steps are in
    // front of the weights' (loads return in order).
    f32x4 head[MT] = {};
    {
        Chunk<ET, float> hw[HEAD][2];
        Chunk<ET, ET> hx[HEAD][2][MT];
        auto ask_head = [&](int s0) {
#pragma unroll
            for (int d = 0; d < HEAD; ++d)
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const uint32_t k = (uint32_t)(s0 + d) * 64 + 32 * h + 8 * (lane / 16);
                    const bool in = s0 + d < last && k < H;
                    hw[d][h].load(rr, in && expert_in ? rk + k : kOutside);
#pragma unroll
                    for (int mt = 0; mt < MT; ++mt) hx[d][h][mt].load(rx, in && tok_in[mt] ? xk[mt] + k : kOutside);
                }
        };
        auto add_head = [&]() {
#pragma unroll
            for (int d = 0; d < HEAD; ++d)
#pragma unroll
                for (int h = 0; h < 2; ++h)
#pragma unroll
                    for (int j = 0; j < 8; ++j)
#pragma unroll
                        for (int mt = 0; mt < MT; ++mt)
                            head[mt] = __builtin_amdgcn_mfma_f32_16x16x4f32(j < 4 ? hw[d][h].a[j % 4] : hw[d][h].b[j % 4], (float)hx[d][h][mt].frag()[j], head[mt], 0, 0, 0);
        };
        int s0 = first;
        for (; s0 + HEAD < last; s0 += HEAD) {
            ask_head(s0);
            __builtin_amdgcn_sched_barrier(0);   // the loads stay together in front
            add_head();
        }
        ask_head(s0);
        __builtin_amdgcn_sched_barrier(0);
        ask(first, p.eager);
        __builtin_amdgcn_sched_barrier(0);
        add_head();
    }
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) parts[wave][mt][lane] = head[mt];
    // a barrier for LDS alone: __syncthreads would wait for the weights
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");

    // every wave works the routing out, a token a lane
    const bool live = lane < T;
    RowState<EP, 1> rs;
    {
        const int mt = lane / kTokens < MT ? lane / kTokens : 0;
#pragma unroll
        for (int g = 0; g < EP / 4; ++g) {
            f32x4 v = parts[0][mt][g * 16 + lane % 16];
#pragma unroll
            for (int q = 1; q < kWaves; ++q) v += parts[q][mt][g * 16 + lane % 16];
#pragma unroll
            for (int i = 0; i < 4; ++i) rs.l[4 * g + i] = !live ? (4 * g + i == 0 ? 0.f : -INFINITY) : 4 * g + i < p.E ? v[i] : -INFINITY;
        }
    }
    softmax_row<EP, 1>(rs);
    float sel_w[MTS_MAX_TOP_K], mass;
    int sel_e[MTS_MAX_TOP_K];
    select_top_k<EP, 1>(rs, p.E, p.K, 0, sel_w, sel_e, mass);
    const float inv = p.normalize ? 1.0f / fmaxf(mass, 1.1920928955078125e-07f) : 1.0f;
    bool mine = false;
    int row = 0;       // rows of the experts in front, and of the tokens in front: where this lane's token stands
    float weight = 0.f;
#pragma unroll
    for (int k = 0; k < MTS_MAX_TOP_K; ++k)
        if (k < p.K) {
            sel_w[k] *= inv;
            row += (int)__popcll(__ballot(live && sel_e[k] < e));
            if (live && sel_e[k] == e) mine = true, weight = (float)(ET)sel_w[k];
        }
    if (router) leave_routing<EP>(p, rs, sel_e, sel_w, live, wave, lane);
    if (alone) return;
    const uint64_t here = __ballot(mine);
    if (!here) return;
    row = mine ? row + (int)__popcll(here & lanemask_lt()) : -1;

    if (!p.eager) ask(first, true);
    f32x4 acc[2][2][MT] = {};
    for (int s0 = first;;) {
#pragma unroll
        for (int d = 0; d < DEPTH; ++d)
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int f = 0; f < 2; ++f)
#pragma unroll
                    for (int c = 0; c < 2; ++c)
#pragma unroll
                        for (int mt = 0; mt < MT; ++mt) acc[f][c][mt] = Few<ET>::mul(w[d][h][f][c].frag(), x[d][h][mt].frag(), acc[f][c][mt]);
        s0 += DEPTH;
        if (s0 >= last) break;
        ask(s0, true);
        __builtin_amdgcn_sched_barrier(0);   // the loads stay together in front
    }
#pragma unroll
    for (int f = 0; f < 2; ++f)
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) sums[wave][f][c][mt][lane] = acc[f][c][mt];
    __syncthreads();
    // four consecutive columns of one token a thread
    if (wave >= 2 * MT) return;
    const int c = wave % 2, mt = wave / 2, n = n0 + 16 * c + 4 * (lane / 16);
    const int to = __shfl(row, kTokens * mt + lane % 16);
    const float s = __shfl(weight, kTokens * mt + lane % 16);
    if (to < 0 || n >= p.I) return;
    f32x4 v[2];
#pragma unroll
    for (int f = 0; f < 2; ++f) {
        v[f] = sums[0][f][c][mt][lane];
#pragma unroll
        for (int q = 1; q < kWaves; ++q) v[f] += sums[q][f][c][mt][lane];
    }
    quad g, u, a;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        g[r] = (ET)v[0][r], u[r] = (ET)v[1][r];
        a[r] = (ET)(v[0][r] * __builtin_amdgcn_rcpf(1.0f + __expf(-v[0][r])) * v[1][r] * s);
    }
    if (p.pre_act) {
        ET* pre = (ET*)p.pre_act + (int64_t)to * 2 * p.I + n;
        *reinterpret_cast<quad*>(pre) = g;
        *reinterpret_cast<quad*>(pre + p.I) = u;
    }
    *reinterpret_cast<quad*>((ET*)p.post_act + (int64_t)to * p.I + n) = a;
}

typedef uint32_t Pair;
template <typename ET>
struct Two {   // as one access
    ET v[2];
};

// 32 columns of one expert's down projection; the block that arrives last at a range of columns, counted over the experts with rows, adds the tokens'
// routes.  Rows and counter pass between the XCDs' L2s: both are written and read by agent-scope accesses, and every wave waits for its rows to be
// acknowledged before the barrier in front of the counter (which by itself waits for LDS alone).
template <typename ET, typename WT, int MT>
__global__ __launch_bounds__(kThreads) void few_tokens_down_kernel(FewTokens p) {
    constexpr int STEP_REGS = 8 * (2 * (int)(sizeof(WT) / sizeof(ET)) + MT);
    constexpr int DEPTH = STEP_REGS > 32 ? 3 : 4;   // steps of 64 k in flight
    __shared__ f32x4 sums[kWaves][2][MT][MTS_WAVE];
    __shared__ int arrived;
    const int lane = threadIdx.x % MTS_WAVE, wave = threadIdx.x / MTS_WAVE;
    // the experts of a range of columns: one XCD, one after the other
    const int j = (int)blockIdx.x / 8, nt = j / p.E * 8 + (int)blockIdx.x % 8, e = j % p.E, n0 = nt * kCols;
    if (n0 >= p.H) return;
    const int begin = lane < p.E ? p.expert_start[lane] : 0, end = lane < p.E ? p.expert_start[lane + 1] : 0;
    const uint64_t filled = __ballot(end > begin);
    if (!(filled >> e & 1)) return;
    const int row0 = __builtin_amdgcn_readlane(begin, e), rows = __builtin_amdgcn_readlane(end, e) - row0;
    const uint32_t I = (uint32_t)p.I;
    const int steps = (p.I + 63) / 64, per = (steps + kWaves - 1) / kWaves;
    const int first = wave * per, last = min(steps, first + per);
    const __amdgpu_buffer_rsrc_t rw = operand((const WT*)p.w2 + (int64_t)e * p.H * p.I, (int64_t)p.H * p.I * sizeof(WT));
    const __amdgpu_buffer_rsrc_t ra = operand((const ET*)p.post_act + (int64_t)row0 * p.I, (int64_t)rows * p.I * 2);
    f32x4 acc[2][MT] = {};
    for (int s0 = first; s0 < last; s0 += DEPTH) {
        Chunk<ET, WT> w[DEPTH][2][2];
        Chunk<ET, ET> a[DEPTH][2][MT];
#pragma unroll
        for (int d = 0; d < DEPTH; ++d)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const uint32_t k = (uint32_t)(s0 + d) * 64 + 32 * h + 8 * (lane / 16);
                const bool in = s0 + d < last && k < I;
#pragma unroll
                for (int c = 0; c < 2; ++c) {
                    const int n = n0 + 16 * c + lane % 16;
                    w[d][h][c].load(rw, in && n < p.H ? (uint32_t)n * I + k : kOutside);
                }
#pragma unroll
                for (int mt = 0; mt < MT; ++mt) {
                    const int r = kTokens * mt + lane % 16;
                    a[d][h][mt].load(ra, in && r < rows ? (uint32_t)r * I + k : kOutside);
                }
            }
        __builtin_amdgcn_sched_barrier(0);   // the loads stay together in front
#pragma unroll
        for (int d = 0; d < DEPTH; ++d)
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int c = 0; c < 2; ++c)
#pragma unroll
                    for (int mt = 0; mt < MT; ++mt) acc[c][mt] = Few<ET>::mul(w[d][h][c].frag(), a[d][h][mt].frag(), acc[c][mt]);
    }
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) sums[wave][c][mt][lane] = acc[c][mt];
    __syncthreads();
    // four consecutive columns of one row a thread
    if (wave < 2 * MT) {
        const int c = wave % 2, mt = wave / 2, r = kTokens * mt + lane % 16, n = n0 + 16 * c + 4 * (lane / 16);
        if (r < rows && n < p.H) {
            f32x4 v = sums[0][c][mt][lane];
#pragma unroll
            for (int q = 1; q < kWaves; ++q) v += sums[q][c][mt][lane];
            Pair* y = (Pair*)p.y + ((int64_t)(row0 + r) * p.H + n) / 2;
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                const Two<ET> two = {{(ET)v[2 * q], (ET)v[2 * q + 1]}};
                __hip_atomic_store(y + q, __builtin_bit_cast(Pair, two), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
        }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // the rows' stores stay in front of it, the counter behind
    __syncthreads();
    if (threadIdx.x == 0) arrived = __hip_atomic_fetch_add(p.arrived + nt, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
    if (arrived != (int)__popcll(filled) - 1) return;
    for (int i = threadIdx.x; i < (int)p.T * (kCols / 2); i += kThreads) {
        const int t = i / (kCols / 2), n = n0 + i % (kCols / 2) * 2;
        if (n >= p.H) continue;
        Pair v[MTS_MAX_TOP_K];
#pragma unroll
        for (int k = 0; k < MTS_MAX_TOP_K; ++k)
            if (k < p.K)
                v[k] = __hip_atomic_load((const Pair*)p.y + ((int64_t)p.s_reverse[t * p.K + k] * p.H + n) / 2, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        float o[2] = {0.f, 0.f};
#pragma unroll
        for (int k = 0; k < MTS_MAX_TOP_K; ++k)
            if (k < p.K) {
                const Two<ET> two = __builtin_bit_cast(Two<ET>, v[k]);
                o[0] += (float)two.v[0], o[1] += (float)two.v[1];
            }
        const Two<ET> two = {{(ET)o[0], (ET)o[1]}};
        *((Pair*)p.out + ((int64_t)t * p.H + n) / 2) = __builtin_bit_cast(Pair, two);
    }
}

int down_ranges(int H) { return (H + kCols - 1) / kCols; }

template <typename ET, typename WT, int MT, int EP>
int launch(FewTokens p, hipStream_t s) {
    // The router's results by a block of their own (15.4 -> 14.1 us, 16 tokens, 8 experts of 768/1024), where it is not one behind whole rounds of the chip
    // (two blocks a CU; 8 experts of 1024/2048: 24.5 -> 32.7).
    constexpr int kRound = 2 * 256;
    p.extra = p.n_tiles * p.E % kRound != 0;
    few_tokens_up_kernel<ET, WT, MT, EP><<<(unsigned)(p.n_tiles * p.E + p.extra), kThreads, 0, s>>>(p);
    MTS_CHECK_LAUNCH();
    few_tokens_down_kernel<ET, WT, MT><<<(unsigned)((down_ranges(p.H) + 7) / 8 * 8 * p.E), kThreads, 0, s>>>(p);
    MTS_CHECK_LAUNCH();
    return MTS_OK;
}
template <typename ET, typename WT>
int launch_any(const FewTokens& p, hipStream_t s) {
    if constexpr (sizeof(WT) == sizeof(ET))
        if (p.E > 8) return p.T <= kTokens ? launch<ET, WT, 1, 16>(p, s) : launch<ET, WT, 2, 16>(p, s);
    return p.T <= kTokens ? launch<ET, WT, 1, 8>(p, s) : launch<ET, WT, 2, 8>(p, s);
}

}  // namespace

extern "C" int mts_moe_few_tokens_supported(int act_dtype, int weight_dtype, int64_t T, int K, int E, int H, int I) {
    return T > 0 && T <= 2 * kTokens && E <= (weight_dtype == MTS_F32 ? 8 : kMostExperts) && K >= 1 && K <= E && K <= MTS_MAX_TOP_K &&
           mts_moe_fwd_few_rows_supported(act_dtype, weight_dtype, T, T * K, E, H, I);
}

// Every block reads x and W_r, and one that does not wait for the routing its weights whether they are wanted or not: with large weights that costs
// more than two launches.  us a call, 1 / 4 / 16 / 32 tokens, as four launches (as three behind a cast) and here: 768/1024, 8 experts, bf16 (36 MiB)
// 31.6 / 31.8 / 31.8 / 32.1 and 25.4 / 24.9 / 24.9 / 26.3, fp32 (72) 32.1 / 34.2 / 41.8 / 42.8 and 25.8 / 27.7 / 30.1 / 35.4; 1024/1024, 16 experts (96)
// 32.4 / 34.7 / 50.6 / 59.2 and 28.0 / 31.0 / 47.5 / 55.9; 1024/2048, 8 experts, fp32 (192) 38.9 / 53.3 / 66.1 / 69.8 and 36.5 / 47.5 / 54.5 / 67.5;
// 2048/2048, 12 experts (288) 42.4 / 65.8 / 90.0 / 102 and 44.9 / 74.1 / 102 / 123; 4096/14336, 8 experts (2688) 159 / 476 / 563 / 597 and 340 / 551 / 680 / 825.
extern "C" int mts_moe_few_tokens_preferred(int act_dtype, int weight_dtype, int64_t T, int K, int E, int H, int I) {
    constexpr int64_t kMostBytes = 192LL << 20;
    return mts_moe_few_tokens_supported(act_dtype, weight_dtype, T, K, E, H, I) && 3LL * E * H * I * (weight_dtype == MTS_F32 ? 4 : 2) <= kMostBytes;
}

extern "C" int mts_moe_few_tokens_fwd(const void* x, const float* w_r, const void* w1, const void* w2, int weight_dtype, int64_t T, int H, int E, int I, int K,
                                      int normalize, int act_dtype, float* logits, float* weights, int32_t* indices, void* weights_act, float* prob_mean,
                                      float* z_loss, float* entropy, int32_t* counts, float* load_balance, float* load_stats, int32_t* expert_start,
                                      int32_t* s_scatter, int32_t* s_reverse, int32_t* x_gather, void* pre_act, void* post_act, void* y, int32_t* arrived, void* out,
                                      void* stream) {
    if (!x || !w_r || !w1 || !w2 || !logits || !weights || !indices || !weights_act || !prob_mean || !z_loss || !entropy || !counts || !expert_start || !s_scatter ||
        !s_reverse || !x_gather || !post_act || !y || !arrived || !out)
        return MTS_ERR_NULL;
    if (!mts_moe_few_tokens_supported(act_dtype, weight_dtype, T, K, E, H, I)) return MTS_ERR_SHAPE;
    if (!mts_aligned16(x) || !mts_aligned16(w_r) || !mts_aligned16(w1) || !mts_aligned16(w2) || !mts_aligned16(pre_act) || !mts_aligned16(post_act) ||
        !mts_aligned16(y) || !mts_aligned16(out))
        return MTS_ERR_ALIGN;
    FewTokens p = {x, w_r, w1, w2, T, H, E, I, K, normalize, act_dtype, (I + kCols - 1) / kCols, 0, T * K >= E, 1.0f / (float)T, 1.0f / ((float)T * (float)K),
                   logits, weights, indices, weights_act, prob_mean, z_loss, entropy, counts, load_balance, load_stats, expert_start, s_scatter, s_reverse, x_gather,
                   pre_act, post_act, y, out, arrived};
    hipStream_t s = (hipStream_t)stream;
    if (act_dtype == MTS_BF16) return weight_dtype == MTS_F32 ? launch_any<bf16_t, float>(p, s) : launch_any<bf16_t, bf16_t>(p, s);
    return weight_dtype == MTS_F32 ? launch_any<mts_f16_t, float>(p, s) : launch_any<mts_f16_t, mts_f16_t>(p, s);
}
