// Capacity-limited routing: of the routes that chose expert e, the `capacity` routes with
// the largest router weights are kept; among equal weights the lower flat entry t*K+k is
// kept first.  Integer and comparison work only: the result is exact.
//
// The stable expert-major permutation of the routing metadata puts the entries of an
// expert into one segment, in ascending entry order.  One block per expert then finds the
// capacity-th largest weight of its segment with a radix select over order-preserving
// 32-bit keys (four passes of 8 bits, histogram in LDS), and a last pass in segment order
// ranks the entries that tie with that weight.
#include "mts_common.h"
#include "mts_router_row.h"

namespace {

constexpr int kSelThreads = 1024;
constexpr int kSelWaves = kSelThreads / MTS_WAVE;
constexpr int kUnroll = 4;
constexpr int kParts = 4;      // blocks per expert
constexpr int kRegKeys = 32;   // segments of up to 32768 routes keep their keys in registers

// float -> unsigned key with the same order; -0 and +0 get the same key
__device__ __forceinline__ uint32_t order_key(float w) {
    uint32_t b = __float_as_uint(w);
    if (w == 0.0f) b = 0u;
    return (b & 0x80000000u) ? ~b : (b | 0x80000000u);
}

// One pass of the select over the keys of a thread: counts the digit at `shift` of the keys
// whose higher digits equal `prefix`.  Router weights share their leading bits, so most lanes
// of a wave hit the same bin in the first pass (`crowded`), where the two most common digits of a wave are
// added once per wave; the digits behind it are mantissa bits, spread over the bins (all passes that way: 38 us for 49 152 routes to 8 experts, this 33).
__device__ __forceinline__ void count_digit(uint32_t* hist, bool count, uint32_t d, int lane, bool crowded) {
#pragma unroll
    for (int r = 0; crowded && r < 2; ++r) {
        const uint64_t todo = __ballot(count);
        if (!todo) break;
        const int leader = __ffsll((unsigned long long)todo) - 1;
        const uint32_t dl = (uint32_t)__builtin_amdgcn_readlane((int)d, leader);
        const uint64_t same = __ballot(count && d == dl);
        if (lane == leader) atomicAdd(&hist[dl], (uint32_t)__popcll(same));
        count = count && d != dl;
    }
    if (count) atomicAdd(&hist[d], 1u);
}

// Where the answer for position i of an expert's segment (entry `entry`) goes.  MaskOut: 1/0 and the expert index or -1 per
// entry.  CompactOut: the compacted permutation, in which the kept entries of an expert keep their order; `rank` counts the
// kept entries in front of this one.
struct MaskOut {
    static constexpr bool kRanked = false;
    uint8_t* keep;
    int32_t* kept_index;   // may be NULL
    int e;
    __device__ __forceinline__ void put(int32_t entry, bool kept, uint32_t) const {
        keep[entry] = kept ? 1 : 0;
        if (kept_index) kept_index[entry] = kept ? e : -1;
    }
};
struct CompactOut {
    static constexpr bool kRanked = true;
    int32_t* s_scatter;
    int32_t* s_reverse;
    int32_t* x_gather;
    int first;             // first row of the expert's kept entries
    uint32_t K, inverse;   // routes per token, floor((2^32 - 1) / K)
    __device__ __forceinline__ void put(int32_t entry, bool kept, uint32_t rank) const {
        const int row = first + (int)rank;
        s_reverse[entry] = kept ? row : -1;
        if (kept) {
            s_scatter[row] = entry;
            const uint32_t q = __umulhi((uint32_t)entry, inverse);   // the quotient or one less
            x_gather[row] = (int32_t)((uint32_t)entry - q * K >= K ? q + 1 : q);
        }
    }
};

// exclusive scan, in place, of one word per (slice, wave) in segment order; called by one wave
__device__ __forceinline__ void scan_table(uint32_t* table, int lane) {
    constexpr int PER_LANE = kRegKeys * kSelWaves / MTS_WAVE;
    uint32_t v[PER_LANE], sum = 0;
#pragma unroll
    for (int j = 0; j < PER_LANE; ++j) {
        v[j] = table[lane * PER_LANE + j];
        sum += v[j];
    }
    uint32_t run = (uint32_t)wave_scan((int)sum) - sum;
#pragma unroll
    for (int j = 0; j < PER_LANE; ++j) {
        table[lane * PER_LANE + j] = run;
        run += v[j];
    }
}

// REGS: the segment has at most kRegKeys keys per thread and they stay in registers; otherwise
// they are written to `kseg` in the first pass and read back in the later ones (the same thread
// touches kseg[i] in every pass).  Position i of the segment belongs to thread i % kSelThreads.
template <bool REGS, class Out>
__device__ __forceinline__ void select_segment(const float* __restrict__ w, const int32_t* __restrict__ seg,
                                               uint32_t* __restrict__ kseg, int n, uint32_t capacity, const Out& out,
                                               uint32_t* hist, uint32_t* chosen, uint32_t* wave_ties,
                                               uint32_t* tie_table, uint32_t* kept_table, int part) {
    const int tid = threadIdx.x, lane = tid % MTS_WAVE, wave = tid / MTS_WAVE;
    uint32_t kr[REGS ? kRegKeys : 1];
    if (REGS) {
        int32_t entry[kRegKeys];
        // (slices behind the segment's end are skipped by the whole block, here and below)
#pragma unroll
        for (int u = 0; u < kRegKeys; ++u) {
            const int i = tid + u * kSelThreads;
            if (u * kSelThreads < n) entry[u] = i < n ? seg[i] : 0;
        }
#pragma unroll
        for (int u = 0; u < kRegKeys; ++u) {
            const int i = tid + u * kSelThreads;
            kr[u] = 0u;
            if (u * kSelThreads < n) kr[u] = i < n ? order_key(w[entry[u]]) : 0u;
        }
    } else {
        for (int i0 = tid; i0 < n; i0 += kUnroll * kSelThreads) {
            int32_t entry[kUnroll];
#pragma unroll
            for (int u = 0; u < kUnroll; ++u) {
                const int i = i0 + u * kSelThreads;
                entry[u] = i < n ? seg[i] : 0;
            }
#pragma unroll
            for (int u = 0; u < kUnroll; ++u) {
                const int i = i0 + u * kSelThreads;
                if (i < n) kseg[i] = order_key(w[entry[u]]);
            }
        }
    }

    uint32_t prefix = 0;          // the digits chosen so far, right-aligned
    uint32_t need = capacity;     // keys still to take among those that match prefix
    for (int pass = 0; pass < 4; ++pass) {
        const int shift = 24 - 8 * pass;
        if (tid < 256) hist[tid] = 0;
        __syncthreads();
        if (REGS) {
#pragma unroll
            for (int u = 0; u < kRegKeys; ++u) {
                const int i = tid + u * kSelThreads;
                const bool count = i < n && (pass == 0 || (kr[u] >> (shift + 8)) == prefix);
                if (u * kSelThreads < n) count_digit(hist, count, (kr[u] >> shift) & 255u, lane, pass == 0);
            }
        } else {
            for (int i0 = tid; i0 < n; i0 += kUnroll * kSelThreads) {
                uint32_t k[kUnroll];
#pragma unroll
                for (int u = 0; u < kUnroll; ++u) {
                    const int i = i0 + u * kSelThreads;
                    k[u] = i < n ? kseg[i] : 0u;
                }
#pragma unroll
                for (int u = 0; u < kUnroll; ++u) {
                    const int i = i0 + u * kSelThreads;
                    const bool count = i < n && (pass == 0 || (k[u] >> (shift + 8)) == prefix);
                    count_digit(hist, count, (k[u] >> shift) & 255u, lane, pass == 0);
                }
            }
        }
        __syncthreads();
        if (wave == 0) {
            // lane l owns bins 4l..4l+3; suffix sums over the lanes find the bin in which the
            // need-th largest matching key lies
            const uint32_t h0 = hist[4 * lane], h1 = hist[4 * lane + 1], h2 = hist[4 * lane + 2],
                           h3 = hist[4 * lane + 3];
            const uint32_t mine = h0 + h1 + h2 + h3;
            const int upto = wave_scan((int)mine);
            uint32_t above = (uint32_t)(__builtin_amdgcn_readlane(upto, MTS_WAVE - 1) - upto);   // matching keys in the bins of higher lanes
            const uint32_t suffix = above + mine;
            if (above < need && need <= suffix) {
                int d;
                if (above + h3 >= need) d = 3;
                else {
                    above += h3;
                    if (above + h2 >= need) d = 2;
                    else {
                        above += h2;
                        if (above + h1 >= need) d = 1;
                        else {
                            above += h1;
                            d = 0;
                        }
                    }
                }
                chosen[0] = (prefix << 8) | (uint32_t)(4 * lane + d);
                chosen[1] = need - above;
            }
        }
        __syncthreads();
        prefix = chosen[0];
        need = chosen[1];
    }

    // prefix is now the key of the capacity-th largest weight; `need` of the entries with
    // exactly that key are kept, the earliest in segment order (= ascending entry)
    const uint64_t lt = lanemask_lt();
    if (REGS) {
        // all slices at once: ties per (slice, wave) to LDS, one exclusive scan over that table in
        // segment order, then every thread ranks and writes its entries with the loads of their
        // entry numbers in flight together (a barrier per slice would expose one L2 round trip each);
        // the compacted permutation counts the kept entries the same way
#pragma unroll
        for (int u = 0; u < kRegKeys; ++u) {
            const int i = tid + u * kSelThreads;
            uint64_t b = 0;
            if (u * kSelThreads < n) b = __ballot(i < n && kr[u] == prefix);
            if (lane == 0) tie_table[u * kSelWaves + wave] = (uint32_t)__popcll(b);
        }
        __syncthreads();
        if (wave == 0) scan_table(tie_table, lane);
        __syncthreads();
        uint32_t kept_mask = 0;   // bit u: this thread's position of slice u is kept
#pragma unroll
        for (int u = 0; u < kRegKeys; ++u) {
            bool kept = false;
            if (u * kSelThreads < n) {
                const int i = tid + u * kSelThreads;
                const bool tie = i < n && kr[u] == prefix;
                const uint32_t rank = tie_table[u * kSelWaves + wave] + (uint32_t)__popcll(__ballot(tie) & lt);
                kept = i < n && (kr[u] > prefix || (tie && rank < need));
                kept_mask |= (kept ? 1u : 0u) << u;
            }
            if constexpr (Out::kRanked) {
                const uint64_t b = __ballot(kept);
                if (lane == 0) kept_table[u * kSelWaves + wave] = (uint32_t)__popcll(b);
            }
        }
        if constexpr (Out::kRanked) {
            __syncthreads();
            if (wave == 0) scan_table(kept_table, lane);
            __syncthreads();
        }
        constexpr int BATCH = 4;
#pragma unroll
        for (int u0 = 0; u0 < kRegKeys; u0 += BATCH) {
            if (u0 * kSelThreads >= n) break;   // block-uniform, as the next
            if (u0 / BATCH % kParts != part) continue;
            int32_t entry[BATCH];
#pragma unroll
            for (int j = 0; j < BATCH; ++j) {
                const int i = tid + (u0 + j) * kSelThreads;
                entry[j] = i < n ? seg[i] : 0;
            }
#pragma unroll
            for (int j = 0; j < BATCH; ++j) {
                const int u = u0 + j;
                const bool kept = (kept_mask >> u) & 1u;
                uint32_t rank = 0;
                if constexpr (Out::kRanked) rank = kept_table[u * kSelWaves + wave] + (uint32_t)__popcll(__ballot(kept) & lt);
                if (tid + u * kSelThreads < n) out.put(entry[j], kept, rank);
            }
        }
    } else {
        uint32_t carry = 0, kept_carry = 0;
        for (int base = 0; base < n; base += kSelThreads) {   // one block-wide slice of kSelThreads positions
            const int i = base + tid;
            const bool in = i < n;
            const uint32_t k = in ? kseg[i] : 0u;
            const bool tie = in && k == prefix;
            auto count_before = [&](bool flag, uint32_t& running) {   // flags of the segment in front of this position
                const uint64_t b = __ballot(flag);
                if (lane == 0) wave_ties[wave] = (uint32_t)__popcll(b);
                __syncthreads();
                uint32_t before = running, total = 0;
#pragma unroll
                for (int j = 0; j < kSelWaves; ++j) {
                    const uint32_t c = wave_ties[j];
                    if (j < wave) before += c;
                    total += c;
                }
                running += total;
                __syncthreads();
                return before + (uint32_t)__popcll(b & lt);
            };
            const uint32_t tie_rank = count_before(tie, carry);
            const bool kept = in && (k > prefix || (tie && tie_rank < need));
            uint32_t rank = 0;
            if constexpr (Out::kRanked) rank = count_before(kept, kept_carry);
            if (in) out.put(seg[i], kept, rank);
        }
    }
}

// One expert's segment: everything, nothing, or the selection.  kParts blocks select, all of them the same (on CUs that would
// idle), and each writes a part of the answer: its scattered stores were a third of the time.
template <class Out>
__device__ __forceinline__ void select_expert(const float* __restrict__ w, const int32_t* __restrict__ seg, uint32_t* __restrict__ keys, int n,
                                              int64_t capacity, const Out& out, int part) {
    __shared__ uint32_t hist[256];
    __shared__ uint32_t chosen[2];          // prefix, number still to take inside it
    __shared__ uint32_t wave_ties[kSelWaves];
    __shared__ uint32_t tie_table[kRegKeys * kSelWaves];   // ties per (slice of kSelThreads positions, wave)
    __shared__ uint32_t kept_table[Out::kRanked ? kRegKeys * kSelWaves : 1];
    const bool all = (int64_t)n <= capacity, none = capacity <= 0;
    if (all || none) {   // block-uniform
        for (int i = part * kSelThreads + threadIdx.x; i < n; i += kParts * kSelThreads) out.put(seg[i], !none, (uint32_t)i);
        return;
    }
    if (n <= kRegKeys * kSelThreads)
        select_segment<true>(w, seg, (uint32_t*)nullptr, n, (uint32_t)capacity, out, hist, chosen, wave_ties, tie_table, kept_table, part);
    else if (part == 0)   // its keys are in memory
        select_segment<false>(w, seg, keys, n, (uint32_t)capacity, out, hist, chosen, wave_ties, tie_table, kept_table, part);
}

__device__ __forceinline__ int32_t accepted_of(int n, int64_t capacity) { return capacity <= 0 ? 0 : ((int64_t)n <= capacity ? n : (int32_t)capacity); }

__global__ __launch_bounds__(kSelThreads) void capacity_select_kernel(
    const float* __restrict__ w, const int32_t* __restrict__ s_scatter,
    const int32_t* __restrict__ counts, const int32_t* __restrict__ expert_start, int64_t capacity,
    uint32_t* __restrict__ keys, uint8_t* __restrict__ keep, int32_t* __restrict__ kept_index,
    int32_t* __restrict__ accepted) {
    const int e = blockIdx.x, n = counts[e], first = expert_start[e];
    if (blockIdx.y == 0 && threadIdx.x == 0) accepted[e] = accepted_of(n, capacity);
    select_expert(w, s_scatter + first, keys + first, n, capacity, MaskOut{keep, kept_index, e}, blockIdx.y);
}

// The same selection as a compacted permutation: how many routes every expert accepts is known from the counts alone, so
// every block knows where its expert's kept rows start.  24 576 x 2 routes over 8 experts, the fullest with 11 000: 21 us (26 with one
// block an expert and shuffles through LDS; three passes of 11 bits: 24), four counting passes over an expert's keys
// and its scattered stores, in place of the routing metadata twice (25 us), the mask (34 us) and its application.
__global__ __launch_bounds__(kSelThreads) void capacity_compact_kernel(
    const float* __restrict__ w, const int32_t* __restrict__ s_scatter, const int32_t* __restrict__ counts,
    const int32_t* __restrict__ expert_start, int E, int K, int64_t capacity, uint32_t* __restrict__ keys, int32_t* __restrict__ accepted,
    int32_t* __restrict__ kept_start, int32_t* __restrict__ kept_scatter, int32_t* __restrict__ kept_reverse, int32_t* __restrict__ kept_gather) {
    __shared__ int32_t in_front[kSelWaves];
    const int e = blockIdx.x, tid = threadIdx.x, n = counts[e], first = expert_start[e];
    int32_t v = tid < e ? accepted_of(counts[tid], capacity) : 0;   // at most 1024 experts: one per thread
    v = wave_sum(v);
    if (tid % MTS_WAVE == 0) in_front[tid / MTS_WAVE] = v;
    __syncthreads();
    int32_t kept_first = 0;
#pragma unroll
    for (int j = 0; j < kSelWaves; ++j) kept_first += in_front[j];
    if (blockIdx.y == 0 && tid == 0) {
        const int32_t a = accepted_of(n, capacity);
        accepted[e] = a;
        kept_start[e] = kept_first;
        if (e == E - 1) kept_start[E] = kept_first + a;
    }
    select_expert(w, s_scatter + first, keys + first, n, capacity, CompactOut{kept_scatter, kept_reverse, kept_gather, kept_first, (uint32_t)K, 0xffffffffu / (uint32_t)K}, blockIdx.y);
}

// Weights under a capacity limit: those of dropped routes become zero, a token's others are renormalised (a token may lose
// every route).  One thread per token; block 0 also writes the load statistics of the accepted routes, in the layout of
// mts_router_fwd's.
constexpr float kSmallest = 1.1920929e-07f;   // fp32 epsilon: the least sum that is divided by
constexpr int kWeightThreads = 256;
template <typename ET>
__global__ __launch_bounds__(kWeightThreads) void capacity_weights_kernel(const float* __restrict__ w, const int32_t* __restrict__ kept_reverse,
                                                                          const int32_t* __restrict__ accepted, const float* __restrict__ entropy,
                                                                          int64_t T, int K, int E, int normalize, ET* __restrict__ out,
                                                                          float* __restrict__ load_stats) {
    for (int64_t t = (int64_t)blockIdx.x * kWeightThreads + threadIdx.x; t < T; t += (int64_t)gridDim.x * kWeightThreads) {
        float total = 0.f;
        for (int k = 0; k < K; ++k) total += kept_reverse[t * K + k] >= 0 ? w[t * K + k] : 0.f;
        const float div = normalize && total > 0.f ? (total > kSmallest ? total : kSmallest) : 1.f;
        for (int k = 0; k < K; ++k) out[t * K + k] = (ET)((kept_reverse[t * K + k] >= 0 ? w[t * K + k] : 0.f) / div);
    }
    if (blockIdx.x != 0 || threadIdx.x >= MTS_WAVE) return;
    const int lane = threadIdx.x;
    const float routes = (float)((double)T * K), scale = (float)E;
    float most = -1.f, least = INFINITY, sum = 0.f, dead = 0.f;
    for (int e = lane; e < E; e += MTS_WAVE) {
        const float a = (float)accepted[e];
        load_stats[e] = a / routes;
        most = fmaxf(most, a);
        least = fminf(least, a);
        sum += a;
        dead += a == 0.f ? 1.f : 0.f;
    }
    sum = wave_sum(sum), dead = wave_sum(dead);
    most = lane_reduce<32, 1>(most, [](float a, float b) { return fmaxf(a, b); });
    least = lane_reduce<32, 1>(least, [](float a, float b) { return fminf(a, b); });
    const float mean = sum / routes / scale;
    float dev = 0.f;
    for (int e = lane; e < E; e += MTS_WAVE) {
        const float d = (float)accepted[e] / routes - mean;
        dev += d * d;
    }
    dev = wave_sum(dev);
    if (lane == 0) {
        float* s = load_stats + E;
        s[0] = most;
        s[1] = least;
        s[2] = sqrtf(dev / scale) * scale;
        s[3] = most / routes * scale;
        s[4] = dead;
        s[5] = 1.0f - sum / routes;
        s[6] = *entropy / (E > 1 ? logf(scale) : 1.0f);
    }
}

// the gradient of those weights, which arrives in the activation dtype, taken back to the unlimited weights
template <typename ET>
__global__ __launch_bounds__(kWeightThreads) void capacity_weights_bwd_kernel(const ET* __restrict__ g, const float* __restrict__ w,
                                                                              const int32_t* __restrict__ kept_reverse, int64_t T, int K,
                                                                              int normalize, float* __restrict__ g_w) {
    for (int64_t t = (int64_t)blockIdx.x * kWeightThreads + threadIdx.x; t < T; t += (int64_t)gridDim.x * kWeightThreads) {
        const mts_router::KeptWeights kw(w + t * K, kept_reverse + t * K, K, normalize, [&](int k) { return (float)g[t * K + k]; });
        for (int k = 0; k < K; ++k) g_w[t * K + k] = kw.gradient(k, (float)g[t * K + k]);
    }
}

// entries whose index is negative on input belong to no segment: they read as dropped
__global__ __launch_bounds__(256) void capacity_init_kernel(int64_t TK, uint8_t* __restrict__ keep,
                                                            int32_t* __restrict__ kept_index) {
    for (int64_t n = (int64_t)blockIdx.x * 256 + threadIdx.x; n < TK; n += (int64_t)gridDim.x * 256) {
        keep[n] = 0;
        if (kept_index) kept_index[n] = -1;
    }
}

int64_t align256(int64_t b) { return (b + 255) & ~(int64_t)255; }

}  // namespace

extern "C" int64_t mts_moe_capacity_workspace_bytes(int64_t T, int K, int E) {
    const int64_t TK = T * K;
    // route workspace, counts [E], expert_start [E+1], s_scatter / s_reverse / x_gather [TK], keys [TK]
    return align256(mts_moe_route_workspace_bytes(T, K, E)) + align256((2 * (int64_t)E + 1) * 4) +
           4 * align256(TK * 4);
}

extern "C" int mts_moe_capacity_mask(const int32_t* top_k_index, const float* top_k_weights, int64_t T,
                                     int K, int E, int64_t capacity, uint8_t* keep, int32_t* kept_index,
                                     int32_t* accepted_counts, void* workspace, int64_t workspace_bytes,
                                     void* stream) {
    if (!top_k_index || !top_k_weights || !keep || !accepted_counts || !workspace) return MTS_ERR_NULL;
    if (T <= 0 || K < 1 || E < 1 || E > MTS_MAX_EXPERTS || T * (int64_t)K > 0x7fffffffLL)
        return MTS_ERR_SHAPE;
    if (workspace_bytes < mts_moe_capacity_workspace_bytes(T, K, E)) return MTS_ERR_WORKSPACE;
    const int64_t TK = T * K;
    char* ws = (char*)workspace;
    const int64_t route_bytes = align256(mts_moe_route_workspace_bytes(T, K, E));
    void* route_ws = ws;
    ws += route_bytes;
    int32_t* counts = (int32_t*)ws;
    int32_t* expert_start = counts + E;
    ws += align256((2 * (int64_t)E + 1) * 4);
    int32_t* s_scatter = (int32_t*)ws;
    ws += align256(TK * 4);
    int32_t* s_reverse = (int32_t*)ws;
    ws += align256(TK * 4);
    int32_t* x_gather = (int32_t*)ws;
    ws += align256(TK * 4);
    uint32_t* keys = (uint32_t*)ws;
    int rc = mts_moe_route(top_k_index, T, K, E, 1, counts, expert_start, s_scatter, s_reverse, x_gather,
                           nullptr, nullptr, nullptr, route_ws, route_bytes, stream);
    if (rc != MTS_OK) return rc;
    const int64_t init_blocks = (TK + 255) / 256;
    capacity_init_kernel<<<(int)(init_blocks < 2048 ? init_blocks : 2048), 256, 0, (hipStream_t)stream>>>(
        TK, keep, kept_index);
    MTS_CHECK_LAUNCH();
    capacity_select_kernel<<<dim3((unsigned)E, kParts), kSelThreads, 0, (hipStream_t)stream>>>(
        top_k_weights, s_scatter, counts, expert_start, capacity, keys, keep, kept_index, accepted_counts);
    MTS_CHECK_LAUNCH();
    return MTS_OK;
}

extern "C" int64_t mts_moe_capacity_compact_workspace_bytes(int64_t T, int K) { return align256(T * K * 4); }

extern "C" int mts_moe_capacity_compact(const float* top_k_weights, const int32_t* counts, const int32_t* expert_start, const int32_t* s_scatter,
                                        int64_t T, int K, int E, int64_t capacity, int32_t* accepted_counts, int32_t* kept_start,
                                        int32_t* kept_scatter, int32_t* kept_reverse, int32_t* kept_gather, void* workspace,
                                        int64_t workspace_bytes, void* stream) {
    if (!top_k_weights || !counts || !expert_start || !s_scatter || !accepted_counts || !kept_start || !kept_scatter || !kept_reverse ||
        !kept_gather || !workspace)
        return MTS_ERR_NULL;
    if (T <= 0 || K < 1 || E < 1 || E > MTS_MAX_EXPERTS || T * (int64_t)K > 0x7fffffffLL) return MTS_ERR_SHAPE;
    if (workspace_bytes < mts_moe_capacity_compact_workspace_bytes(T, K)) return MTS_ERR_WORKSPACE;
    capacity_compact_kernel<<<dim3((unsigned)E, kParts), kSelThreads, 0, (hipStream_t)stream>>>(top_k_weights, s_scatter, counts, expert_start, E, K, capacity,
                                                                        (uint32_t*)workspace, accepted_counts, kept_start, kept_scatter,
                                                                        kept_reverse, kept_gather);
    MTS_CHECK_LAUNCH();
    return MTS_OK;
}

extern "C" int mts_moe_capacity_weights_fwd(const float* top_k_weights, const int32_t* kept_reverse, const int32_t* accepted_counts,
                                            const float* entropy, int64_t T, int K, int E, int normalize, int act_dtype, void* weights_out,
                                            float* load_stats, void* stream) {
    if (!top_k_weights || !kept_reverse || !accepted_counts || !entropy || !weights_out || !load_stats) return MTS_ERR_NULL;
    if (T <= 0 || K < 1 || E < 1 || T * (int64_t)K > 0x7fffffffLL) return MTS_ERR_SHAPE;
    const int64_t want = (T + kWeightThreads - 1) / kWeightThreads;
    const dim3 grid((unsigned)(want < 1024 ? want : 1024));
    hipStream_t s = (hipStream_t)stream;
    if (act_dtype == MTS_BF16)
        capacity_weights_kernel<bf16_t><<<grid, kWeightThreads, 0, s>>>(top_k_weights, kept_reverse, accepted_counts, entropy, T, K, E, normalize, (bf16_t*)weights_out, load_stats);
    else if (act_dtype == MTS_F16)
        capacity_weights_kernel<mts_f16_t><<<grid, kWeightThreads, 0, s>>>(top_k_weights, kept_reverse, accepted_counts, entropy, T, K, E, normalize, (mts_f16_t*)weights_out, load_stats);
    else if (act_dtype == MTS_F32)
        capacity_weights_kernel<float><<<grid, kWeightThreads, 0, s>>>(top_k_weights, kept_reverse, accepted_counts, entropy, T, K, E, normalize, (float*)weights_out, load_stats);
    else return MTS_ERR_DTYPE;
    MTS_CHECK_LAUNCH();
    return MTS_OK;
}

extern "C" int mts_moe_capacity_weights_bwd(const void* g_weights, const float* top_k_weights, const int32_t* kept_reverse, int64_t T, int K,
                                            int normalize, int act_dtype, float* g_top_k_weights, void* stream) {
    if (!g_weights || !top_k_weights || !kept_reverse || !g_top_k_weights) return MTS_ERR_NULL;
    if (T <= 0 || K < 1 || T * (int64_t)K > 0x7fffffffLL) return MTS_ERR_SHAPE;
    const int64_t want = (T + kWeightThreads - 1) / kWeightThreads;
    const dim3 grid((unsigned)(want < 1024 ? want : 1024));
    hipStream_t s = (hipStream_t)stream;
    if (act_dtype == MTS_BF16)
        capacity_weights_bwd_kernel<bf16_t><<<grid, kWeightThreads, 0, s>>>((const bf16_t*)g_weights, top_k_weights, kept_reverse, T, K, normalize, g_top_k_weights);
    else if (act_dtype == MTS_F16)
        capacity_weights_bwd_kernel<mts_f16_t><<<grid, kWeightThreads, 0, s>>>((const mts_f16_t*)g_weights, top_k_weights, kept_reverse, T, K, normalize, g_top_k_weights);
    else if (act_dtype == MTS_F32)
        capacity_weights_bwd_kernel<float><<<grid, kWeightThreads, 0, s>>>((const float*)g_weights, top_k_weights, kept_reverse, T, K, normalize, g_top_k_weights);
    else return MTS_ERR_DTYPE;
    MTS_CHECK_LAUNCH();
    return MTS_OK;
}
