// Shared device helpers for the gfx950 MoE kernels (wave size 64).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "mts_moe.h"

typedef __bf16 bf16_t;
typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) __bf16 bf16x4;
typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;
typedef _Float16 mts_f16_t;
typedef __attribute__((ext_vector_type(8))) _Float16 mts_f16x8;
typedef __attribute__((ext_vector_type(4))) _Float16 mts_f16x4;
typedef __attribute__((ext_vector_type(16))) float f32x16;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(4))) uint32_t u32x4;

#define MTS_WAVE 64

#define MTS_CHECK_LAUNCH()                       \
    do {                                         \
        hipError_t _e = hipGetLastError();       \
        if (_e != hipSuccess) return (int)_e;    \
    } while (0)

__device__ __forceinline__ float bf16_bits_to_f32(uint32_t bits16) {
    return __uint_as_float(bits16 << 16);
}

// The value of lane ^ O, on the vector unit (a shuffle goes through LDS: a hundred cycles of latency); O < 16.
template <int O>
__device__ __forceinline__ uint32_t lane_xor_bits(uint32_t v) {
    static_assert(O == 8 || O == 4 || O == 2 || O == 1, "within a row of 16 lanes");
    if constexpr (O == 8) return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x128, 0xf, 0xf, true);   // rotate the row by 8
    else if constexpr (O == 4) {   // lanes 0..3 and 8..11 of a row from four lanes up, the others from four lanes down
        const int up = __builtin_amdgcn_update_dpp((int)v, (int)v, 0x104, 0xf, 0x5, false);
        return (uint32_t)__builtin_amdgcn_update_dpp(up, (int)v, 0x114, 0xf, 0xa, false);
    } else if constexpr (O == 2) return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x4e, 0xf, 0xf, true);
    else return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0xb1, 0xf, 0xf, true);
}

// op(value of this lane, value of lane ^ O) for a commutative op
template <int O, typename V, class Op>
__device__ __forceinline__ V lane_pair(V v, Op op) {
    static_assert(sizeof(V) == 4, "one register");
    const uint32_t bits = __builtin_bit_cast(uint32_t, v);
    if constexpr (O == 32) {
        const auto r = __builtin_amdgcn_permlane32_swap(bits, bits, false, false);
        return op(__builtin_bit_cast(V, (uint32_t)r[0]), __builtin_bit_cast(V, (uint32_t)r[1]));
    } else if constexpr (O == 16) {
        const auto r = __builtin_amdgcn_permlane16_swap(bits, bits, false, false);
        return op(__builtin_bit_cast(V, (uint32_t)r[0]), __builtin_bit_cast(V, (uint32_t)r[1]));
    } else return op(v, __builtin_bit_cast(V, lane_xor_bits<O>(bits)));
}

// the value of lane ^ O
template <int O, typename V>
__device__ __forceinline__ V lane_other(V v) {
    static_assert(sizeof(V) == 4, "one register");
    const uint32_t bits = __builtin_bit_cast(uint32_t, v);
    if constexpr (O >= 16) {   // the swap leaves the lower lanes' values in the first register and the upper ones' in the second
        const bool upper = threadIdx.x & O;
        if constexpr (O == 32) {
            const auto r = __builtin_amdgcn_permlane32_swap(bits, bits, false, false);
            return __builtin_bit_cast(V, (uint32_t)(upper ? r[0] : r[1]));
        } else {
            const auto r = __builtin_amdgcn_permlane16_swap(bits, bits, false, false);
            return __builtin_bit_cast(V, (uint32_t)(upper ? r[0] : r[1]));
        }
    } else return __builtin_bit_cast(V, lane_xor_bits<O>(bits));
}

// op over lanes that agree but for the bits from `LOW` up to FROM, widest distance first
template <int FROM, int LOW, typename V, class Op>
__device__ __forceinline__ V lane_reduce(V v, Op op) {
    if constexpr (FROM >= LOW && FROM > 0) return lane_reduce<FROM / 2, LOW>(lane_pair<FROM>(v, op), op);
    else return v;
}
struct LaneSum {
    template <typename V>
    __device__ __forceinline__ V operator()(V a, V b) const { return a + b; }
};
__device__ __forceinline__ float wave_sum(float v) { return lane_reduce<32, 1>(v, LaneSum()); }
__device__ __forceinline__ int32_t wave_sum(int32_t v) { return lane_reduce<32, 1>(v, LaneSum()); }

// inclusive sum over the wave's lanes
__device__ __forceinline__ int wave_scan(int v) {
    v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, false);   // one lane up within a row of 16, then 2, 4, 8
    v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);   // the last lane of rows 0 and 2 to rows 1 and 3
    v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);   // lane 31 to rows 2 and 3
    return v;
}

__device__ __forceinline__ uint64_t lanemask_lt() {
    return (1ull << (threadIdx.x & 63)) - 1ull;
}

// round(a * b) + round(c * d), rounded, as separate elementwise operators leave them (contraction would drop the two conversions in between)
template <typename ET>
__device__ __forceinline__ ET sum_of_rounded_products(float a, float b, float c, float d) {
#pragma clang fp contract(off)
    const ET p = (ET)(a * b), q = (ET)(c * d);
    return (ET)((float)p + (float)q);
}

template <typename ET>
__device__ __forceinline__ ET difference_of_rounded_products(float a, float b, float c, float d) {
#pragma clang fp contract(off)
    const ET p = (ET)(a * b), q = (ET)(c * d);
    return (ET)((float)p - (float)q);
}

static inline bool mts_aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

// fp16 instantiation of the grouped GEMMs (mts_gemm_f16.hip); the public entry points forward to it
extern "C" {
int mts_moe_fwd_gateup_swiglu_f16(const void* x, const void* w1, const int32_t* x_gather, const int32_t* expert_start,
                                  const void* weights, const int32_t* s_scatter, int64_t T, int K, int E, int H, int I, int act_dtype, void* pre_act, void* post_act,
                                  void* stream);
int mts_moe_fwd_down_f16(const void* post_act, const void* w2, const int32_t* expert_start, int64_t TK, int E, int H,
                         int I, int act_dtype, void* y, void* stream);
int mts_moe_fwd_gateup_down_f16(const void* x, const void* w1, const void* w2, const int32_t* x_gather,
                                const int32_t* expert_start, const void* weights, const int32_t* s_scatter, int64_t T, int K,
                                int E, int H, int I, int act_dtype, void* pre_act, void* post_act, void* y,
                                int32_t* workspace, int64_t workspace_bytes, void* stream);
int mts_moe_bwd_dy1_f16(const void* d_out, const void* w2, int w2_as_stored, const void* pre_act, const void* weights,
                        const int32_t* x_gather, const int32_t* s_scatter, const int32_t* expert_start, int64_t T,
                        int K, int E, int H, int I, int act_dtype, void* d_pre_act, void* weighted_act,
                        float* ds_partial, int32_t* schedule, void* stream);
int mts_moe_bwd_dx_f16(const void* d_pre_act, const void* w1, int w1_as_stored, const int32_t* expert_start,
                       int64_t TK, int E, int H, int I, int act_dtype, void* dx_expanded, void* stream);
int mts_moe_bwd_dw2_f16(const void* d_out, const void* weighted_act, const int32_t* x_gather,
                        const int32_t* expert_start, int64_t T, int K, int E, int H, int I, int act_dtype,
                        int grad_dtype, void* d_w2, void* workspace, int64_t workspace_bytes, void* stream);
int mts_linear_fwd_f16(const void* x, const void* w, int64_t T, int N, int K, int act_dtype, void* y, void* stream);
int mts_linear_dx_f16(const void* g, const void* w, int64_t T, int N, int K, int act_dtype, void* dx, void* stream);
int mts_linear_dw_tiles_f16(const void* g, const void* x, int64_t T, int N, int K, float* part, void* stream);
int mts_linear_dw_rounds_f16(const void* g, int64_t ldg, const void* x, int64_t T, int N, int K, float* dw, float* part, void* stream);
int mts_linear_dx_rounds_f16(const void* g, int64_t ldg, const void* w, int64_t T, int N, int K, void* dx, float* part, void* stream);
int mts_moe_bwd_dw1_f16(const void* d_pre_act, const void* x, const int32_t* x_gather, const int32_t* expert_start,
                        int64_t T, int K, int E, int H, int I, int act_dtype, int grad_dtype, void* d_w1,
                        void* workspace, int64_t workspace_bytes, void* stream);
int mts_moe_bwd_joint_f16(const void* d_out, const void* weighted_act, const void* d_pre_act, const void* x,
                          const void* w1, const int32_t* x_gather, const int32_t* expert_start,
                          const int32_t* s_reverse, const float* ds_partial, int64_t T, int K, int E, int H, int I,
                          int act_dtype, int grad_dtype, void* dx_expanded, void* d_w1, void* d_w2, void* d_weights,
                          void* workspace1, int64_t workspace1_bytes, void* workspace2, int64_t workspace2_bytes,
                          const int32_t* schedule, void* stream);
int mts_moe_bwd_joint_router_f16(const void* d_out, const void* weighted_act, const void* d_pre_act, const void* x,
                                 const void* w1, const int32_t* x_gather, const int32_t* expert_start,
                                 const int32_t* s_reverse, const float* ds_partial, int64_t T, int K, int E, int H,
                                 int I, int act_dtype, int grad_dtype, void* dx_expanded, void* d_w1, void* d_w2,
                                 void* d_weights, void* workspace1, int64_t workspace1_bytes, void* workspace2,
                                 int64_t workspace2_bytes, const float* w_r, const float* logits,
                                 const float* weights, const int32_t* indices, const int32_t* counts,
                                 const float* g_prob_mean, const float* g_z_loss, const float* g_load_balance,
                                 int normalize, void* dx_router, void* dx, float* d_w_r, void* router_workspace,
                                 int64_t router_workspace_bytes, const int32_t* schedule, void* stream);
}

// fp32 GEMM launchers (mts_gemm_f32.hip); epi: 0 plain, 1 SwiGLU, 2 dO*W2 with SwiGLU backward
int mts_f32_rows(int epi, const float* A, int lda, const int32_t* a_gather, const float* B, int b_rows, int b_kmajor,
                 int N, int Kdim, const int32_t* expert_start, int E, int64_t TK, float* C, float* C2,
                 const float* pre_act, const float* route_w, const int32_t* s_scatter, float* ds_part,
                 int np, hipStream_t s);
int mts_f32_dw(const float* P, const int32_t* p_gather, const float* Q, const int32_t* q_gather, int M,
               int N, const int32_t* expert_start, int E, int grad_dtype, void* C, hipStream_t s);

// chained router forward (mts_router_linear.hip), launched by mts_moe_head_fwd (mts_route.hip)
#define MTS_HEAD_MAX_CHUNKS 512
// Launch shape of the chained router backward (mts_router_linear.hip): row blocks x column ranges, the threads
// a block needs (groups sets of col_threads) and its dynamic LDS; contract checks of that path; the reduction
// of its per-block dW_r partials.
struct MtsRouterBwdShape {
    int row_blocks, rows_per_block, groups, col_threads, cols_per_block, ranges;
};
int mts_router_bwd_check(const void* x, const float* w_r, int64_t T, int H, int E, int act_dtype);
void mts_router_bwd_shape(int64_t T, int H, int E, MtsRouterBwdShape* shape);
int mts_launch_router_dw_reduce(const float* part, int row_blocks, int64_t EH, float* d_w_r, hipStream_t s);
int mts_router_head_group(int H, int E, int act_dtype);   // rows a wave of the chained forward kernel finishes together
void mts_router_head_geometry(int64_t T, int group, int* blocks, int* rows_per_wave);
// Routing statistics that are still to be reduced from the partial sums of a router launch's blocks: arguments of mts_router::stats_block
struct MtsRouterStats {
    const float* partial;
    const int32_t* partial_counts;
    int blocks, E;
    float inv_t, inv_routes;
    float *prob_mean, *z_loss, *entropy;
    int32_t* counts;
    float *load_balance, *load_stats;
};
// mts_router_fwd without that reduction
int mts_launch_router_fwd(const float* logits, int64_t T, int E, int K, int normalize, float* weights, int32_t* indices, float* prob_mean, float* z_loss,
                          float* entropy, int32_t* counts, float* load_balance, float* load_stats, void* weights_act, int act_dtype, void* workspace,
                          int64_t workspace_bytes, MtsRouterStats* stats, hipStream_t s);
// rows of a block of the chained head of 17 to 64 experts (mts_router_wide.hip), which are a chunk of its routing metadata, and the most of them
#define MTS_WIDE_HEAD_ROWS 32
#define MTS_WIDE_HEAD_CHUNKS 1024
int mts_launch_wide_head(const void* x, const float* w_r, int64_t T, int H, int E, int K, int normalize, int act_dtype, float* logits, float* weights, int32_t* indices,
                         void* weights_act, float* partial, int32_t* partial_counts, int32_t* cnt, const MtsCast* cast, hipStream_t s);
// What the launch behind the head writes from partial and cnt.  Where the head is one block (up to 64 tokens) the block writes it itself:
// *finished is 1 then, and partial and cnt are left as they are.
struct MtsHeadFinish {
    float inv_t, inv_routes;
    float *prob_mean, *z_loss, *entropy;
    int32_t* counts;
    float *load_balance, *load_stats;
    int32_t *expert_start, *s_scatter, *s_reverse, *x_gather;
};
bool mts_router_head_carries(int64_t T, int H, int E, int act_dtype);   // whether copies of weights gain as further blocks of it
int mts_launch_router_head(const void* x, const float* w_r, int64_t T, int H, int E, int K, int normalize, int act_dtype,
                           float* logits, float* weights, int32_t* indices, void* weights_act, float* partial,
                           int32_t* cnt, MtsHeadFinish finish, int* finished, const MtsCast* cast, hipStream_t s);   // cast: more blocks of the launch, or NULL
