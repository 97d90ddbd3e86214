// Per-row arithmetic of the router post-process (softmax of a row of fp32 logits held by G
// adjacent lanes, top-k on the logits with the lower expert index winning ties, the gradient
// of a row) and the one-block reduction of the routing statistics.  Shared by the stand-alone
// post-process kernels and the kernels that chain the router projection to them.
#pragma once

#include "mts_common.h"

#include <math.h>

namespace mts_router {

// A token's routing weights under a capacity limit: routes without a row (kept_reverse < 0) weigh nothing and the others are
// divided by their sum.  What a gradient of the result is for the weights it was formed from; `g_of(k)`: that gradient.
struct KeptWeights {
    const int32_t* kept;
    float scale = 1.f, dot = 0.f;   // 1 / sum, and sum_j g_j w'_j
    template <class G>
    __device__ __forceinline__ KeptWeights(const float* w, const int32_t* kept_reverse, int K, int normalize, G g_of) : kept(kept_reverse) {
        if (!normalize) return;
        float total = 0.f;
        for (int k = 0; k < K; ++k) total += kept[k] >= 0 ? w[k] : 0.f;
        if (!(total > 0.f)) return;
        constexpr float smallest = 1.1920929e-07f;   // below it the forward pass divides by this constant
        scale = 1.f / (total > smallest ? total : smallest);
        if (total > smallest)
            for (int k = 0; k < K; ++k) dot += kept[k] >= 0 ? g_of(k) * w[k] * scale : 0.f;
    }
    __device__ __forceinline__ float gradient(int k, float g) const { return kept[k] >= 0 ? (g - dot) * scale : 0.f; }
};


constexpr float kLogFloor = -20.72326583694641f;  // log(1e-9): the entropy clamps p at 1e-9

template <int G>
__device__ __forceinline__ float group_sum(float v) { return lane_reduce<G / 2, 1>(v, LaneSum()); }
template <int G>
__device__ __forceinline__ float group_max(float v) {
    return lane_reduce<G / 2, 1>(v, [](float a, float b) { return fmaxf(a, b); });
}

template <int EP, int G>
struct RowState {
    float l[EP];
    float p[EP];
    float m, s, L;
};

// softmax of the row whose logits are in r.l (slots past E hold -inf): p, the row maximum, the
// sum of exponentials and the log-partition
template <int EP, int G>
__device__ __forceinline__ void softmax_row(RowState<EP, G>& r) {
    float m = r.l[0];
#pragma unroll
    for (int j = 1; j < EP; ++j) m = fmaxf(m, r.l[j]);
    m = group_max<G>(m);
    float s = 0.f;
#pragma unroll
    for (int j = 0; j < EP; ++j) {
        r.p[j] = expf(r.l[j] - m);
        s += r.p[j];
    }
    s = group_sum<G>(s);
    float inv = 1.0f / s;
#pragma unroll
    for (int j = 0; j < EP; ++j) r.p[j] *= inv;
    r.m = m;
    r.s = s;
    r.L = m + logf(s);
}

template <int EP, int G>
__device__ __forceinline__ void load_row(const float* __restrict__ logits, int64_t row, int E, int g,
                                         RowState<EP, G>& r) {
    const float* src = logits + row * (int64_t)E;
    if (G == 1 && EP == 8 && E == 8) {
        const f32x4* v = reinterpret_cast<const f32x4*>(src);
        f32x4 a = v[0], b = v[1];
        r.l[0] = a[0]; r.l[1] = a[1]; r.l[2] = a[2]; r.l[3] = a[3];
        r.l[4 % EP] = b[0]; r.l[5 % EP] = b[1]; r.l[6 % EP] = b[2]; r.l[7 % EP] = b[3];
    } else {
#pragma unroll
        for (int j = 0; j < EP; ++j) {
            int e = j * G + g;
            r.l[j] = (e < E) ? src[e] : -INFINITY;
        }
    }
    softmax_row<EP, G>(r);
}


// the larger value of the lanes that share a row, and its expert; the lower expert where two are equal
template <int O>
__device__ __forceinline__ void best_of_lanes(float& bv, int& be) {
    if constexpr (O > 0) {
        const float ov = lane_other<O>(bv);
        const int oe = lane_other<O>(be);
        if (ov > bv || (ov == bv && oe < be)) bv = ov, be = oe;
        best_of_lanes<O / 2>(bv, be);
    }
}

// K rounds of arg-max over the logits of a row (ties to the lower expert index).  `taken` has a
// bit per slot j of this lane (expert j*G + g); sel_e / sel_p get the expert and its softmax
// probability per rank, mass the sum of the selected probabilities.  A NaN counts as -infinity: such
// a row's weights are NaN, but its routes are K different experts as any row's are, which the counters,
// the scan and the scatter of the routing metadata rely on.
template <int EP, int G>
__device__ __forceinline__ void select_top_k(const RowState<EP, G>& r, int E, int K, int g,
                                             float (&sel_p)[MTS_MAX_TOP_K], int (&sel_e)[MTS_MAX_TOP_K], float& mass) {
    uint32_t taken = 0;
#pragma unroll
    for (int j = 0; j < EP; ++j)
        if (j * G + g >= E) taken |= 1u << j;
    mass = 0.f;
#pragma unroll
    for (int k = 0; k < MTS_MAX_TOP_K; ++k) {
        sel_p[k] = 0.f;
        sel_e[k] = -1;
        if (k < K) {
            float bv = -INFINITY;
            int be = 0x7fffffff;
#pragma unroll
            for (int j = 0; j < EP; ++j) {
                int e = j * G + g;
                bool free_slot = !((taken >> j) & 1u);
                if (free_slot && (r.l[j] > bv || be == 0x7fffffff)) {   // the lane's experts ascend: an equal one stays behind
                    bv = fmaxf(r.l[j], bv);
                    be = e;
                }
            }
            best_of_lanes<G / 2>(bv, be);
            if (be % G == g) taken |= 1u << (be / G);
            float pk = expf(bv - r.m) / r.s;
            sel_p[k] = pk;
            sel_e[k] = be;
            mass += pk;
        }
    }
}

// What a lane has summed over its rows, G lanes a row: probability mass and routes of its experts (slot j is expert j*G + g), squared
// log-partitions, entropies.
template <int EP, int G>
struct RowTotals {
    float psum[EP] = {};
    int csum[EP] = {};
    float zsum = 0.f, hsum = 0.f;

    // top-k of a row: its weights and indices go out, its statistics to the sums (rows that are not `live`: neither)
    __device__ __forceinline__ void take(const RowState<EP, G>& r, bool live, int64_t row, int E, int K, int normalize, int g, float* __restrict__ weights,
                                         int32_t* __restrict__ indices, void* __restrict__ weights_act, int act_dtype) {
        float sel_p[MTS_MAX_TOP_K];
        int sel_e[MTS_MAX_TOP_K];
        float mass;
        select_top_k<EP, G>(r, E, K, g, sel_p, sel_e, mass);
#pragma unroll
        for (int k = 0; k < MTS_MAX_TOP_K; ++k)
#pragma unroll
            for (int j = 0; j < EP; ++j) csum[j] += (live && k < K && j * G + g == sel_e[k]) ? 1 : 0;
        if (live && g == 0) {
            float inv = normalize ? 1.0f / fmaxf(mass, 1.1920928955078125e-07f) : 1.0f;
#pragma unroll
            for (int k = 0; k < MTS_MAX_TOP_K; ++k) {
                if (k < K) {
                    const float wk = sel_p[k] * inv;
                    weights[row * K + k] = wk;
                    indices[row * K + k] = sel_e[k];
                    // the copy the MoE block hands to fused_moe: rounded once, as tensor.to() rounds
                    if (weights_act) {
                        if (act_dtype == MTS_BF16) reinterpret_cast<bf16_t*>(weights_act)[row * K + k] = (bf16_t)wk;
                        else reinterpret_cast<mts_f16_t*>(weights_act)[row * K + k] = (mts_f16_t)wk;
                    }
                }
            }
        }
        if (live) {
#pragma unroll
            for (int j = 0; j < EP; ++j) {
                psum[j] += r.p[j];
                // p * log(max(p, 1e-9)); p == 0 (padding or underflow) contributes 0
                float lp = fmaxf(r.l[j] - r.L, kLogFloor);
                hsum -= (r.p[j] > 0.f) ? r.p[j] * lp : 0.f;
            }
            if (g == 0) zsum += r.L * r.L;
        }
    }

    // the sums of a wave's lanes to the wave's row of LDS
    __device__ __forceinline__ void to_lds(float* red, int32_t* cred) {
        const int lane = threadIdx.x % MTS_WAVE;
#pragma unroll
        for (int j = 0; j < EP; ++j) psum[j] = lane_reduce<32, G>(psum[j], LaneSum());   // lanes that hold the same experts
        zsum = wave_sum(zsum);
        hsum = wave_sum(hsum);
#pragma unroll
        for (int j = 0; j < EP; ++j) csum[j] = lane_reduce<32, G>(csum[j], LaneSum());
        if (lane < G) {
#pragma unroll
            for (int j = 0; j < EP; ++j) {
                red[j * G + lane] = psum[j];
                cred[j * G + lane] = csum[j];
            }
        }
        if (lane == 0) {
            red[EP * G] = zsum;
            red[EP * G + 1] = hsum;
        }
    }
};

// column i < E + 2 of a block's statistics, and for i < E its routes, from its waves' rows
template <int EP, int G, int WAVES>
__device__ __forceinline__ float block_column(const float (&red)[WAVES][EP * G + 2], int i, int E) {
    const int src = i < E ? i : EP * G + (i - E);
    float v = 0.f;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) v += red[w][src];
    return v;
}

// Gradient of a row's logits.  dp: gradient that reaches the row's probabilities through the mean
// probability (and the load-balancing term), per slot of this lane; gz: gradient of the z-loss
// times 2/T; weights / indices / grad_w(k): the row's selected weights, experts and weight gradients.
template <int EP, int G, class GradW>
__device__ __forceinline__ void row_logit_gradient(const RowState<EP, G>& r, const float (&gp)[EP], float gz, int K,
                                                   int normalize, int g, const float* __restrict__ weights,
                                                   const int32_t* __restrict__ indices, GradW grad_w, float (&o)[EP]) {
    float dp[EP], extra[EP];
#pragma unroll
    for (int j = 0; j < EP; ++j) {
        dp[j] = gp[j];
        extra[j] = 0.f;
    }
    float wdot = 0.f;
    if (normalize) {
        for (int k = 0; k < K; ++k) wdot += weights[k] * grad_w(k);
    }
    for (int k = 0; k < K; ++k) {
        int e = indices[k];
        float gw = grad_w(k);
        float w = weights[k];
#pragma unroll
        for (int j = 0; j < EP; ++j) {
            if (j * G + g == e) {
                if (normalize) extra[j] += w * (gw - wdot);
                else dp[j] += gw;
            }
        }
    }
    float dot = 0.f;
#pragma unroll
    for (int j = 0; j < EP; ++j) dot += r.p[j] * dp[j];
    dot = group_sum<G>(dot);
#pragma unroll
    for (int j = 0; j < EP; ++j) o[j] = r.p[j] * (dp[j] - dot) + gz * r.L * r.p[j] + extra[j];
}

// ---- reduction of the routing statistics (one block) ----------------------------------------
// Column i < E of the per-block partials is the probability mass of expert i, column E the sum
// of squared log-partitions, column E+1 the entropy sum.  Sums run in a fixed order (bit-stable).
template <int EXPERTS>
struct StatsOf {
    float prod[EXPERTS];    // fraction of routes x mean probability, per expert
    float share[EXPERTS];   // fraction of routes, per expert
    int routes_of[EXPERTS];
    float entropy_s;
};
typedef StatsOf<MTS_MAX_EXPERTS> StatsShared;

// what one thread does with the mean `v` of column i and, for i < E, the routes `c` of expert i
template <class Stats>
__device__ __forceinline__ void stats_column(Stats& sh, int i, float v, int c, int E, float inv_routes,
                                             float* __restrict__ prob_mean, float* __restrict__ z_loss,
                                             float* __restrict__ entropy, int32_t* __restrict__ counts) {
    if (i < E) {
        prob_mean[i] = v;
        sh.prod[i] = (float)c * inv_routes * v;
        sh.share[i] = (float)c * inv_routes;
        sh.routes_of[i] = c;
        if (counts) counts[i] = c;
    } else if (i == E) {
        z_loss[0] = v;
    } else {
        entropy[0] = v;
        sh.entropy_s = v;
    }
}

// After a block barrier behind the stats_column calls: wave `lb_wave` writes the load-balancing term
// E * sum_e (routes_e / routes) * mean_prob_e, wave `ls_wave` the load statistics of the router module
// (minitrain/model/moe_router.py:113-135) from the route fractions: [0,E) the fractions, then the
// largest and smallest route count, the coefficient of variation (population standard deviation x E),
// largest fraction x E, the number of experts without a route, a zero (the dropped-route fraction of
// dropless routing) and the entropy over log E.  Either output may be NULL.
template <class Stats>
__device__ __forceinline__ void stats_finalize(const Stats& sh, int wave, int lb_wave, int ls_wave, int E,
                                               float* __restrict__ load_balance, float* __restrict__ load_stats) {
    const int lane = threadIdx.x % MTS_WAVE;
    if (wave == lb_wave && load_balance) {
        float v = 0.f;
        for (int e = lane; e < E; e += MTS_WAVE) v += sh.prod[e];
        v = wave_sum(v);
        if (lane == 0) load_balance[0] = (float)E * v;
    }
    if (wave == ls_wave && load_stats) {
        float sum = 0.f, hi = 0.f, dead = 0.f;
        int most = 0, fewest = 0x7fffffff;
        for (int e = lane; e < E; e += MTS_WAVE) {
            const float f = sh.share[e];
            load_stats[e] = f;
            sum += f;
            hi = fmaxf(hi, f);
            most = max(most, sh.routes_of[e]);
            fewest = min(fewest, sh.routes_of[e]);
            dead += sh.routes_of[e] == 0 ? 1.f : 0.f;
        }
        sum = wave_sum(sum);
        dead = wave_sum(dead);
        hi = lane_reduce<32, 1>(hi, [](float a, float b) { return fmaxf(a, b); });
        most = lane_reduce<32, 1>(most, [](int a, int b) { return max(a, b); });
        fewest = lane_reduce<32, 1>(fewest, [](int a, int b) { return min(a, b); });
        const float mean = sum / (float)E;
        float var = 0.f;
        for (int e = lane; e < E; e += MTS_WAVE) {
            const float d = sh.share[e] - mean;
            var += d * d;
        }
        var = wave_sum(var) / (float)E;
        if (lane == 0) {
            load_stats[E] = (float)most;
            load_stats[E + 1] = (float)fewest;
            load_stats[E + 2] = sqrtf(var) * (float)E;
            load_stats[E + 3] = hi * (float)E;
            load_stats[E + 4] = dead;
            load_stats[E + 5] = 0.f;
            load_stats[E + 6] = sh.entropy_s / (E > 1 ? logf((float)E) : 1.0f);
        }
    }
}

// The whole reduction by one block: neighbouring threads take neighbouring columns of the partials, sets of them every
// (sets)th row, and the sets' sums are added in order.  (A column per wave, a row per lane, asks for a line per value: 17 us for
// 256 rows of 66 columns, this 9.)
template <int THREADS>
__device__ __forceinline__ void stats_block(
    const float* __restrict__ partial, const int32_t* __restrict__ partial_counts, int nblocks, int E,
    float inv_t, float inv_routes, float* __restrict__ prob_mean, float* __restrict__ z_loss,
    float* __restrict__ entropy, int32_t* __restrict__ counts, float* __restrict__ load_balance,
    float* __restrict__ load_stats, int wave) {
    __shared__ StatsShared sh;
    __shared__ float set_sum[THREADS];
    __shared__ int32_t set_count[THREADS];
    int width = 16;
    while (width < E + 2 && width < THREADS) width <<= 1;
    const int sets = THREADS / width, set = threadIdx.x / width;
    for (int i0 = 0; i0 < E + 2; i0 += width) {
        const int i = i0 + threadIdx.x % width;
        float v = 0.f;
        int32_t c = 0;
        // sixteen rows in flight, whatever the lane: a load that some lanes skip waits for the ones before it
        const float* p = partial + (i < E + 2 ? i : E + 1);
        const int32_t* pc = partial_counts + (i < E ? i : E - 1);
        constexpr int kBatch = 16;
        for (int b0 = set; b0 < nblocks; b0 += kBatch * sets) {
            float vb[kBatch];
            int32_t cb[kBatch];
#pragma unroll
            for (int k = 0; k < kBatch; ++k) {
                const int64_t b = b0 + k * sets < nblocks ? b0 + k * sets : nblocks - 1;
                vb[k] = p[b * (E + 2)];
                cb[k] = pc[b * E];
            }
#pragma unroll
            for (int k = 0; k < kBatch; ++k) {
                const bool there = b0 + k * sets < nblocks;
                v = there ? v + vb[k] : v;
                c += there ? cb[k] : 0;
            }
        }
        if (i >= E) c = 0;
        set_sum[threadIdx.x] = v;
        set_count[threadIdx.x] = c;
        __syncthreads();
        if (set == 0 && i < E + 2) {
#pragma unroll 8
            for (int k = 1; k < sets; ++k) {
                v += set_sum[k * width + threadIdx.x];
                c += set_count[k * width + threadIdx.x];
            }
            stats_column(sh, i, v * inv_t, c, E, inv_routes, prob_mean, z_loss, entropy, counts);
        }
        __syncthreads();
    }
    if (!load_balance && !load_stats) return;   // block-uniform
    stats_finalize(sh, wave, 0, 1, E, load_balance, load_stats);
}

}  // namespace mts_router
