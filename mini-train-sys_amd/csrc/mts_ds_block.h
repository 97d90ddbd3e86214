// The gradient of the routing weights: a route's partial sums, added as the work of one block.  Shared by the stand-alone kernel (mts_combine.hip) and
// the fp32 launch of the other gradients (mts_gemm_f32.hip).
#pragma once

#include "mts_common.h"

namespace mts_ds {

// block `block` of `blocks`
template <typename OutT, int THREADS>
__device__ __forceinline__ void sum_block(const float* __restrict__ part, const int32_t* __restrict__ s_rev, int64_t TK, int np, OutT* __restrict__ d_w, int block,
                                          int blocks) {
    for (int64_t n = (int64_t)block * THREADS + threadIdx.x; n < TK; n += (int64_t)blocks * THREADS) {
        const int32_t r = s_rev[n];   // negative: dropped route, no gradient
        float v = 0.f;
        if (r >= 0) {
            // one add after the other (a fixed order), but 16 loads in flight at a time
            const float* p = part + (int64_t)r * np;
            for (int j0 = 0; j0 < np; j0 += 16) {
                float t[16];
#pragma unroll
                for (int j = 0; j < 16; ++j) t[j] = j0 + j < np ? p[j0 + j] : 0.f;
#pragma unroll
                for (int j = 0; j < 16; ++j)
                    if (j0 + j < np) v += t[j];
            }
        }
        d_w[n] = (OutT)v;
    }
}

}  // namespace mts_ds
