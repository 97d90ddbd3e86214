// The stable scatter of one chunk of routes by one wave: shared by the routing kernels (mts_route.hip) and the router head of few
// tokens (mts_router_linear.hip), whose only block finishes the routing metadata itself.
#pragma once

#include "mts_common.h"

namespace mts_route {

constexpr int kHeadExperts = 16;   // experts of the chained head, at most
constexpr int kChunk = 256;   // entries per wave
constexpr int kSteps = kChunk / MTS_WAVE;
constexpr int kFewExperts = 8;   // windows up to this many experts are ranked with one ballot per expert

// Expert ids >= E are a caller error; they are clamped so that no address derived from
// them can leave the output arrays.  Negative ids (dropped routes) stay negative.
__device__ __forceinline__ int clamp_expert(int e, int E) { return e >= E ? E - 1 : e; }

// The stable scatter of one chunk (entries [cbeg, cend)) by one wave; next[e] is the next free row
// of window expert e for this chunk (LDS, private to the wave).
// E: all experts; [e0, e0 + EW): the window of this pass.
// scatter_load fetches the window-relative expert ids of kSteps x 64 entries starting at `base`
// (-1: dropped route, whose -1 goes to s_reverse in the first pass; -2: not this pass);
// scatter_place ranks and writes them.
__device__ __forceinline__ void scatter_load(int (&ev)[kSteps], const int32_t* __restrict__ idx, int E, int e0, int EW,
                                             int64_t base, int64_t cend) {
    const int lane = threadIdx.x % MTS_WAVE;
#pragma unroll
    for (int s = 0; s < kSteps; ++s) {  // these loads are in flight together
        const int64_t n = base + s * MTS_WAVE + lane;
        const int e = n < cend ? clamp_expert(idx[n], E) : -1;
        ev[s] = e < 0 ? (e0 == 0 && n < cend ? -1 : -2) : (e >= e0 && e < e0 + EW ? e - e0 : -2);
    }
}

// Division of an entry (below 2^31) by the routes per token: a multiplication and a correction for each, one division for all
struct TokenOf {
    uint32_t K, inverse;
    __device__ __forceinline__ explicit TokenOf(int k) : K((uint32_t)k), inverse(0xffffffffu / (uint32_t)k) {}
    __device__ __forceinline__ uint32_t operator()(uint32_t n) const {
        const uint32_t q = __umulhi(n, inverse);   // the quotient or one less
        return n - q * K >= K ? q + 1 : q;
    }
};

// LDS the compiler knows as LDS: through a generic pointer every access would wait for the global ones in flight
typedef volatile __attribute__((address_space(3))) int32_t* LdsRows;

__device__ __forceinline__ void scatter_place(const int (&ev)[kSteps], int K, int EW, int64_t base, int64_t cend,
                                              LdsRows next, int32_t* __restrict__ s_scatter,
                                              int32_t* __restrict__ s_reverse, int32_t* __restrict__ x_gather) {
    const int lane = threadIdx.x % MTS_WAVE;
    const uint64_t lt = lanemask_lt();
    const TokenOf by_K(K);
    if (EW <= kFewExperts) {   // wave-uniform
        // A window of few experts: one ballot per expert ranks the 64 entries of a step, and the next free rows
        // stay in registers from step to step (the same positions as below: entries of one expert in lane order).
        int32_t nx[kFewExperts];
#pragma unroll
        for (int x = 0; x < kFewExperts; ++x) nx[x] = x < EW ? next[x] : 0;
#pragma unroll
        for (int s = 0; s < kSteps; ++s) {
            const int64_t n = base + s * MTS_WAVE + lane;
            if (base + s * MTS_WAVE >= cend) break;   // wave-uniform
            const int e = ev[s];
            int pos = -1;
#pragma unroll
            for (int x = 0; x < kFewExperts; ++x) {
                const uint64_t same = __ballot(e == x);
                if (e == x) pos = nx[x] + __popcll(same & lt);
                nx[x] += __popcll(same);
            }
            if (e >= -1 && n < cend) s_reverse[n] = pos;
            if (e >= 0) {
                s_scatter[pos] = (int32_t)n;
                x_gather[pos] = (int32_t)by_K((uint32_t)n);
            }
        }
#pragma unroll
        for (int x = 0; x < kFewExperts; ++x)
            if (lane == x && x < EW) next[x] = nx[x];
        return;
    }
#pragma unroll
    for (int s = 0; s < kSteps; ++s) {
        const int64_t n = base + s * MTS_WAVE + lane;
        if (base + s * MTS_WAVE >= cend) break;   // wave-uniform
        const int e = ev[s];
        const bool valid = e >= 0;
        int pos = -1;
        // the lanes with the same expert: one ballot per bit of the id
        uint64_t same = __ballot(valid);
#pragma unroll 1
        for (int bit = 0; (1 << bit) < EW; ++bit) {
            const uint64_t set = __ballot((e >> bit) & 1);
            same &= ((e >> bit) & 1) ? set : ~set;
        }
        if (valid) {
            const int first = next[e];   // every lane reads before the first of its group updates
            pos = first + __popcll(same & lt);
            if ((same & lt) == 0) next[e] = first + __popcll(same);
        }
        if (e >= -1 && n < cend) s_reverse[n] = pos;
        if (valid) {
            s_scatter[pos] = (int32_t)n;
            x_gather[pos] = (int32_t)by_K((uint32_t)n);
        }
    }
}

// `first` holds the ids of the chunk's first kSteps x 64 entries already (scatter_load at cbeg)
__device__ __forceinline__ void scatter_chunk(int (&first)[kSteps], const int32_t* __restrict__ idx, int K, int E, int e0,
                                              int EW, int64_t cbeg, int64_t cend, LdsRows next,
                                              int32_t* __restrict__ s_scatter, int32_t* __restrict__ s_reverse,
                                              int32_t* __restrict__ x_gather) {
    scatter_place(first, K, EW, cbeg, cend, next, s_scatter, s_reverse, x_gather);
    for (int64_t base = cbeg + kChunk; base < cend; base += kChunk) {
        int ev[kSteps];
        scatter_load(ev, idx, E, e0, EW, base, cend);
        scatter_place(ev, K, EW, base, cend, next, s_scatter, s_reverse, x_gather);
    }
}

}  // namespace mts_route
