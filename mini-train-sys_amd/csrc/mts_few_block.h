// Weights read once, straight into matrix-instruction operands: what the expert GEMMs for few rows an expert (mts_few_rows.hip) and the layer for few
// tokens (mts_few_tokens.hip) share.
#pragma once

#include "mts_common.h"

namespace mts_few {

template <typename ET>
struct Few;
template <>
struct Few<bf16_t> {
    typedef bf16x8 frag;
    typedef bf16x4 quad;
    static __device__ __forceinline__ f32x4 mul(frag a, frag b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0); }
};
template <>
struct Few<mts_f16_t> {
    typedef mts_f16x8 frag;
    typedef mts_f16x4 quad;
    static __device__ __forceinline__ f32x4 mul(frag a, frag b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0); }
};

constexpr int kWaves = 4, kThreads = kWaves * MTS_WAVE;   // the waves split k
constexpr int kCols = 32;
constexpr uint32_t kOutside = 0x60000000u;   // an element whose bytes, of two or of four modulo 2^32, lie behind the end of every operand (smaller than 2 GiB): reads as zero

__device__ __forceinline__ __amdgpu_buffer_rsrc_t operand(const void* p, int64_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, (int)(uint32_t)bytes, 0x00020000);
}

// eight consecutive k of a row as they lie in memory, and as a fragment
template <typename ET, typename WT>
struct Chunk;
template <typename ET>
struct Chunk<ET, ET> {
    u32x4 v;
    __device__ __forceinline__ void load(__amdgpu_buffer_rsrc_t r, uint32_t element) {
        v = __builtin_amdgcn_raw_buffer_load_b128(r, (int)(element * 2), 0, 0);
    }
    __device__ __forceinline__ typename Few<ET>::frag frag() const { return __builtin_bit_cast(typename Few<ET>::frag, v); }
};
template <typename ET>
struct Chunk<ET, float> {
    f32x4 a, b;
    __device__ __forceinline__ void load(__amdgpu_buffer_rsrc_t r, uint32_t element) {
        const uint32_t at = element * 4;
        a = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(r, (int)at, 0, 0));
        b = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(r, (int)at, 16, 0));
    }
    __device__ __forceinline__ typename Few<ET>::frag frag() const {
        typename Few<ET>::frag f;
#pragma unroll
        for (int j = 0; j < 4; ++j) f[j] = (ET)a[j], f[4 + j] = (ET)b[j];
        return f;
    }
};

}  // namespace mts_few
