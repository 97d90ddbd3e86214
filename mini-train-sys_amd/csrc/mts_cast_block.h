// fp32 -> 16-bit copies of weights as blocks of another launch: the router's launches in front of the experts are chains of latencies that
// leave the memory idle, and the copies need nothing of them.
//
// Bound by HBM (6 bytes a value).  18.9 M values (8 experts of 768/1024): 19 to 21 us in a launch of their own; two thirds of them beside the head of 8192 tokens
// make 14 us of it 18, the rest beside the scatter launch makes 6.6 us of it 11.  A lane takes two pieces of eight values (head and scatter, 8192
// tokens: 18.0 + 11.4 us; four pieces 18.6 + 11.7, eight 19.7 + 10.7).  The layer's step of 5003 tokens 290 -> 276 us, of 600 tokens and 64 experts of
// 1024/512 411 -> 362, a pass of 300 tokens without gradients 56 -> 45, the validation pass of 8 x 1024 tokens through twelve layers 3.98 -> 3.79 ms.
#pragma once
#include "mts_combine_block.h"
#include "mts_common.h"

// the first blocks of a launch are its own, those from `own_blocks` on belong to the copy
struct MtsCastJob {
    MtsCast cast;
    unsigned own_blocks;
};

namespace mts_cast {

constexpr int kItems = 2;

inline int64_t blocks(const MtsCast* c, int threads) { return c ? (c->n / 8 + threads * kItems - 1) / (threads * kItems) : 0; }
inline MtsCastJob job(const MtsCast* c, unsigned own_blocks) { return {c ? *c : MtsCast{}, own_blocks}; }

template <typename ET, int THREADS>
__device__ __forceinline__ void cast_block(const MtsCast& c, unsigned block) {
    typedef typename mts_cb::Vec8<ET>::type vec8;
    const int64_t items = c.n / 8, first = (int64_t)block * (THREADS * kItems) + threadIdx.x;
    f32x4 lo[kItems], hi[kItems];
#pragma unroll
    for (int q = 0; q < kItems; ++q) {
        const int64_t i = first + q * THREADS < items ? first + q * THREADS : items - 1;
        lo[q] = *reinterpret_cast<const f32x4*>(c.src + i * 8), hi[q] = *reinterpret_cast<const f32x4*>(c.src + i * 8 + 4);
    }
#pragma unroll
    for (int q = 0; q < kItems; ++q) {
        vec8 v;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            v[j] = (ET)lo[q][j];
            v[4 + j] = (ET)hi[q][j];
        }
        if (first + q * THREADS < items) *reinterpret_cast<vec8*>(static_cast<ET*>(c.dst) + (first + q * THREADS) * 8) = v;
    }
}

}  // namespace mts_cast
