// The decoder's operators around its matrix products: RMSNorm (with the residual sum in front of it), rotary
// position encoding of the packed query/key/value projection, and the cross-entropy of the logits.  All of them are
// bound by HBM: every kernel reads each operand once and writes each result once, in the activation dtype, with fp32
// arithmetic in registers.
#include "mts_common.h"

#include <type_traits>

namespace {

template <typename ET>
struct DenseVec;   // 4 elements
template <>
struct DenseVec<bf16_t> {
    typedef bf16x4 v4;
    typedef bf16x8 v8;
};
template <>
struct DenseVec<mts_f16_t> {
    typedef mts_f16x4 v4;
    typedef mts_f16x8 v8;
};
template <>
struct DenseVec<float> {
    typedef f32x4 v4;
    typedef __attribute__((ext_vector_type(8))) float v8;
};

// Where a sum is taken of values as they read back after a store in ET, contraction is off: the compiler otherwise drops
// the two conversions in between and fuses the operations.
template <typename ET>
__device__ __forceinline__ ET rounded_sum(ET a, ET b) {
#pragma clang fp contract(off)
    return (ET)((float)a + (float)b);
}
constexpr int kNormWaves = 4;
constexpr int kNormThreads = kNormWaves * MTS_WAVE;

// ---------------------------------------------------------------------------
// RMSNorm.  A wave holds one row in registers (NV groups of four elements per lane), so the row is read once and the
// sum of squares never leaves the wave; groups of four (8 bytes of a 16-bit type) because 768, the usual width, is three
// whole groups a lane.  24 576 x 768 bf16: 27 us forward with the residual sum (151 MB, 5.7 TB/s), 31 us backward (4.9 TB/s);
// the chain of stock kernels these replace took 160 and 390 us.
// ---------------------------------------------------------------------------

// y = (s * rsqrt(mean(s^2) + eps)) * w with s = x + residual (rounded to the activation dtype, as it is stored)
template <typename ET, int NV>
__global__ __launch_bounds__(kNormThreads) void rmsnorm_fwd_kernel(const ET* __restrict__ x, const ET* __restrict__ residual,
                                                                   const float* __restrict__ w, int64_t N, int H, float eps,
                                                                   ET* __restrict__ s_out, ET* __restrict__ y, float* __restrict__ rstd) {
    typedef typename DenseVec<ET>::v4 v4;
    const int lane = threadIdx.x % MTS_WAVE;
    const int64_t row = (int64_t)blockIdx.x * kNormWaves + threadIdx.x / MTS_WAVE;
    if (row >= N) return;
    const int groups = H / 4;
    const v4* xr = reinterpret_cast<const v4*>(x + row * H);
    const v4* rr = reinterpret_cast<const v4*>(residual + (residual ? row * H : 0));
    v4 v[NV], r[NV];
#pragma unroll
    for (int i = 0; i < NV; ++i) {
        const int c = i * MTS_WAVE + lane;
        v[i] = c < groups ? xr[c] : v4{};
        r[i] = (residual && c < groups) ? rr[c] : v4{};
    }
    float sum = 0.f;
#pragma unroll
    for (int i = 0; i < NV; ++i) {
        if (residual) {
#pragma unroll
            for (int j = 0; j < 4; ++j) v[i][j] = rounded_sum<ET>(v[i][j], r[i][j]);
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) sum += (float)v[i][j] * (float)v[i][j];
    }
    const float scale = rsqrtf(wave_sum(sum) / (float)H + eps);
    if (lane == 0) rstd[row] = scale;
    v4* yr = reinterpret_cast<v4*>(y + row * H);
    v4* sr = reinterpret_cast<v4*>(s_out + (s_out ? row * H : 0));
#pragma unroll
    for (int i = 0; i < NV; ++i) {
        const int c = i * MTS_WAVE + lane;
        if (c >= groups) continue;
        const f32x4 wv = reinterpret_cast<const f32x4*>(w)[c];
        v4 o;
#pragma unroll
        for (int j = 0; j < 4; ++j) o[j] = (ET)((float)v[i][j] * scale * wv[j]);
        yr[c] = o;
        if (s_out) sr[c] = v[i];
    }
}

// d_s = gs + rstd * (gy * w - n * mean(gy * w * n)) with n = s * rstd; partial sums of gy * n per block for dw.
template <typename ET, int NV>
__global__ __launch_bounds__(kNormThreads) void rmsnorm_bwd_kernel(const ET* __restrict__ gy, const ET* __restrict__ gs,
                                                                   const ET* __restrict__ s, const float* __restrict__ w,
                                                                   const float* __restrict__ rstd, int64_t N, int H,
                                                                   ET* __restrict__ d_s, float* __restrict__ dw_part) {
    typedef typename DenseVec<ET>::v4 v4;
    const int lane = threadIdx.x % MTS_WAVE, wave = threadIdx.x / MTS_WAVE;
    const int groups = H / 4;
    float dw[NV][4] = {};
    for (int64_t row = (int64_t)blockIdx.x * kNormWaves + wave; row < N; row += (int64_t)gridDim.x * kNormWaves) {
        const v4* gr = reinterpret_cast<const v4*>(gy + row * H);
        const v4* sr = reinterpret_cast<const v4*>(s + row * H);
        const v4* ar = reinterpret_cast<const v4*>(gs + (gs ? row * H : 0));
        v4 g[NV], v[NV], a[NV];
#pragma unroll
        for (int i = 0; i < NV; ++i) {
            const int c = i * MTS_WAVE + lane;
            const bool in = c < groups;
            g[i] = in ? gr[c] : v4{};
            v[i] = in ? sr[c] : v4{};
            a[i] = (gs && in) ? ar[c] : v4{};
        }
        const float scale = rstd[row];
        float dot = 0.f;
#pragma unroll
        for (int i = 0; i < NV; ++i) {
            const int c = i * MTS_WAVE + lane;
            const f32x4 wv = c < groups ? reinterpret_cast<const f32x4*>(w)[c] : f32x4{};
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const float n = (float)v[i][j] * scale;
                dw[i][j] += (float)g[i][j] * n;
                dot += (float)g[i][j] * wv[j] * n;
            }
        }
        dot = wave_sum(dot) / (float)H;
        v4* dr = reinterpret_cast<v4*>(d_s + row * H);
#pragma unroll
        for (int i = 0; i < NV; ++i) {
            const int c = i * MTS_WAVE + lane;
            if (c >= groups) continue;
            const f32x4 wv = reinterpret_cast<const f32x4*>(w)[c];
            v4 o;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const float n = (float)v[i][j] * scale;
                o[j] = (ET)(scale * ((float)g[i][j] * wv[j] - n * dot) + (float)a[i][j]);
            }
            dr[c] = o;
        }
    }
    // the four waves' sums, in wave order
    extern __shared__ float lds[];   // [H]
#pragma unroll 1
    for (int k = 0; k < kNormWaves; ++k) {
        if (wave == k) {
#pragma unroll
            for (int i = 0; i < NV; ++i) {
                const int c = i * MTS_WAVE + lane;
                if (c >= groups) continue;
                f32x4* slot = reinterpret_cast<f32x4*>(lds) + c;
                f32x4 t = k ? *slot : f32x4{};
#pragma unroll
                for (int j = 0; j < 4; ++j) t[j] += dw[i][j];
                *slot = t;
            }
        }
        __syncthreads();
    }
    f32x4* part = reinterpret_cast<f32x4*>(dw_part + (int64_t)blockIdx.x * H);
    for (int c = threadIdx.x; c < groups; c += kNormThreads) part[c] = reinterpret_cast<const f32x4*>(lds)[c];
}

// dw[c] = sum over the blocks' partials, in a fixed two-level order: 16 row groups of 64 columns per block
constexpr int kNormRedGroups = 16;
__global__ __launch_bounds__(64 * kNormRedGroups) void rmsnorm_dw_kernel(const float* __restrict__ part, int blocks, int H, float* __restrict__ dw) {
    __shared__ float sums[kNormRedGroups][64];
    const int col = blockIdx.x * 64 + threadIdx.x % 64, group = threadIdx.x / 64;
    float t = 0.f;
    if (col < H) {
#pragma unroll 4
        for (int b = group; b < blocks; b += kNormRedGroups) t += part[(int64_t)b * H + col];
    }
    sums[group][threadIdx.x % 64] = t;
    __syncthreads();
    if (group == 0 && col < H) {
#pragma unroll
        for (int g = 1; g < kNormRedGroups; ++g) t += sums[g][threadIdx.x];
        dw[col] = t;
    }
}

// groups of four elements a lane holds, rounded up to the next instantiated size; 0: row too wide
int norm_groups(int H) {
    const int need = (H / 4 + MTS_WAVE - 1) / MTS_WAVE;
    for (int v : {1, 2, 3, 4, 6, 8, 12, 16})
        if (need <= v) return v;
    return 0;
}

// 256 CUs x 4 blocks of 4 waves fill the chip; more blocks only add partials to sum
int norm_bwd_blocks(int64_t N) {
    const int64_t need = (N + kNormWaves - 1) / kNormWaves;
    return (int)(need < 1024 ? need : 1024);
}

template <typename ET, int NV>
void launch_norm_fwd(const void* x, const void* r, const float* w, int64_t N, int H, float eps, void* s, void* y, float* rstd, hipStream_t st) {
    rmsnorm_fwd_kernel<ET, NV><<<dim3((unsigned)((N + kNormWaves - 1) / kNormWaves)), dim3(kNormThreads), 0, st>>>(
        (const ET*)x, (const ET*)r, w, N, H, eps, (ET*)s, (ET*)y, rstd);
}
template <typename ET, int NV>
void launch_norm_bwd(const void* gy, const void* gs, const void* s, const float* w, const float* rstd, int64_t N, int H, void* d_s,
                     float* part, int blocks, hipStream_t st) {
    rmsnorm_bwd_kernel<ET, NV><<<dim3(blocks), dim3(kNormThreads), (size_t)H * 4, st>>>((const ET*)gy, (const ET*)gs, (const ET*)s, w, rstd, N, H,
                                                                                        (ET*)d_s, part);
}

#define MTS_NORM_DISPATCH(FN, ET, nv, ...)            \
    switch (nv) {                                     \
        case 1: FN<ET, 1>(__VA_ARGS__); break;        \
        case 2: FN<ET, 2>(__VA_ARGS__); break;        \
        case 3: FN<ET, 3>(__VA_ARGS__); break;        \
        case 4: FN<ET, 4>(__VA_ARGS__); break;        \
        case 6: FN<ET, 6>(__VA_ARGS__); break;        \
        case 8: FN<ET, 8>(__VA_ARGS__); break;        \
        case 12: FN<ET, 12>(__VA_ARGS__); break;      \
        default: FN<ET, 16>(__VA_ARGS__); break;      \
    }

// ---------------------------------------------------------------------------
// Rotary encoding.  One thread turns VEC pairs (d, d + D/2) of one head of one token: two 16-byte loads and stores
// where the half head is a multiple of eight 16-bit elements.  Up to three tensors per launch, each with its own
// strides (elements): queries and keys are read where the packed projection left them, and the backward launch writes
// the gradient of that projection in place of three scattered pieces.  24 x 1024 tokens, 12 heads of 64, bf16: 37 us either
// way (151 / 226 MB); the stock products, negations and concatenations took 270 us forward and 400 us backward.
// ---------------------------------------------------------------------------
enum RopeMode { ROPE_TURN = 0, ROPE_TURN_BACK = 1, ROPE_COPY = 2 };

template <typename ET>
struct RopeTensor {
    const ET* in;
    ET* out;
    int64_t in_b, in_s, in_h, out_b, out_s, out_h;
    int mode;
};
template <typename ET>
struct RopeArgs {
    RopeTensor<ET> t[3];
    const ET* cos;
    const ET* sin;
    int64_t B, S;
    int heads, D;
};

// The products are rounded to the activation dtype before they are added, as separate elementwise operators leave them.
template <typename ET, int VEC>
__global__ __launch_bounds__(256) void rope_kernel(RopeArgs<ET> a) {
    typedef __attribute__((ext_vector_type(VEC))) ET vec;
    const RopeTensor<ET>& t = a.t[blockIdx.y];
    const int half = a.D / 2, chunks = half / VEC;
    const int64_t total = a.B * a.S * a.heads * chunks;
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= total) return;
    const int c = (int)(i % chunks) * VEC;
    const int64_t rest = i / chunks;
    const int h = (int)(rest % a.heads);
    const int64_t tok = rest / a.heads;
    const int64_t s = tok % a.S;
    const int64_t b = tok / a.S;
    const ET* in = t.in + b * t.in_b + s * t.in_s + h * t.in_h + c;
    ET* out = t.out + b * t.out_b + s * t.out_s + h * t.out_h + c;
    const vec v1 = *reinterpret_cast<const vec*>(in), v2 = *reinterpret_cast<const vec*>(in + half);
    if (t.mode == ROPE_COPY) {
        *reinterpret_cast<vec*>(out) = v1;
        *reinterpret_cast<vec*>(out + half) = v2;
        return;
    }
    const ET* cs = a.cos + s * a.D + c;
    const ET* sn = a.sin + s * a.D + c;
    const vec c1 = *reinterpret_cast<const vec*>(cs), c2 = *reinterpret_cast<const vec*>(cs + half);
    const vec s1 = *reinterpret_cast<const vec*>(sn), s2 = *reinterpret_cast<const vec*>(sn + half);
    vec o1, o2;
#pragma unroll
    for (int j = 0; j < VEC; ++j) {
        const float x1 = (float)v1[j], x2 = (float)v2[j];
        if (t.mode == ROPE_TURN) {
            o1[j] = sum_of_rounded_products<ET>(x1, (float)c1[j], -x2, (float)s1[j]);
            o2[j] = sum_of_rounded_products<ET>(x2, (float)c2[j], x1, (float)s2[j]);
        } else {
            o1[j] = sum_of_rounded_products<ET>(x1, (float)c1[j], x2, (float)s2[j]);
            o2[j] = sum_of_rounded_products<ET>(x2, (float)c2[j], -x1, (float)s1[j]);
        }
    }
    *reinterpret_cast<vec*>(out) = o1;
    *reinterpret_cast<vec*>(out + half) = o2;
}

template <typename ET>
int launch_rope(const MtsRopeTensor* tensors, int count, const void* cos, const void* sin, int64_t B, int64_t S, int heads, int D, hipStream_t st) {
    RopeArgs<ET> a = {};
    int vec = 16 / (int)sizeof(ET);
    while (vec > 1 && (D / 2) % vec) vec /= 2;
    auto fits = [&](const void* p, int64_t x, int64_t y, int64_t z) {
        while (vec > 1 && (((uintptr_t)p % (vec * sizeof(ET))) || x % vec || y % vec || z % vec)) vec /= 2;
    };
    for (int i = 0; i < count; ++i) {
        const MtsRopeTensor& m = tensors[i];
        a.t[i] = RopeTensor<ET>{(const ET*)m.in, (ET*)m.out, m.in_b, m.in_s, m.in_h, m.out_b, m.out_s, m.out_h, m.mode};
        fits(m.in, m.in_b, m.in_s, m.in_h);
        fits(m.out, m.out_b, m.out_s, m.out_h);
    }
    fits(cos, 0, 0, 0);
    fits(sin, 0, 0, 0);
    a.cos = (const ET*)cos, a.sin = (const ET*)sin;
    a.B = B, a.S = S, a.heads = heads, a.D = D;
    const int64_t total = B * S * heads * (D / 2 / vec);
    const dim3 grid((unsigned)((total + 255) / 256), count);
    if (vec == 8) {
        if constexpr (sizeof(ET) == 2) rope_kernel<ET, 8><<<grid, 256, 0, st>>>(a);
    } else if (vec == 4) rope_kernel<ET, 4><<<grid, 256, 0, st>>>(a);
    else if (vec == 2) rope_kernel<ET, 2><<<grid, 256, 0, st>>>(a);
    else rope_kernel<ET, 1><<<grid, 256, 0, st>>>(a);
    MTS_CHECK_LAUNCH();
    return MTS_OK;
}

// ---------------------------------------------------------------------------
// Cross-entropy over rows of logits.  A row need not start on a 16-byte boundary (vocabularies are odd): a block peels
// the elements in front of the first boundary and those behind the last one, and streams the rest in 16-byte loads, four
// in flight per thread.  24 576 x 50 257 bf16: 405 us forward (2.5 GB read, 6.1 TB/s), 950 us backward (4.9 GB, 5.2 TB/s);
// by way of an fp32 copy of the logits it was 4.2 and 6.5 ms.
// ---------------------------------------------------------------------------
constexpr int kCeThreads = 512;
constexpr float kLog2e = 1.4426950408889634f;

template <typename ET>
struct CeRow {
    static constexpr int W = 16 / (int)sizeof(ET);
    int head, vecs, tail;   // elements in front, 16-byte groups, elements behind
    __device__ __forceinline__ CeRow(const ET* p, int V) {
        const int mis = (int)(((uintptr_t)p % 16) / sizeof(ET));
        head = mis ? W - mis : 0;
        if (head > V) head = V;
        vecs = (V - head) / W;
        tail = V - head - vecs * W;
    }
};

// v_exp_f32: results below the smallest normal number become zero, which no sum here notices
__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }

// running maximum and sum of 2^((v - max) * log2 e)
struct MaxSum {
    float m, s;
    __device__ __forceinline__ void merge(float m2, float s2) {
        const float hi = fmaxf(m, m2);
        if (hi == -INFINITY) return;   // nothing but -inf so far
        s = s * fast_exp2((m - hi) * kLog2e) + s2 * fast_exp2((m2 - hi) * kLog2e);
        m = hi;
    }
};

template <int O, class Acc>
__device__ __forceinline__ void merge_lanes(Acc& acc) {
    if constexpr (O > 0) {
        acc.merge(lane_other<O>(acc.m), lane_other<O>(acc.s));
        merge_lanes<O / 2>(acc);
    }
}

template <typename ET>
__global__ __launch_bounds__(kCeThreads) void cross_entropy_fwd_kernel(const ET* __restrict__ logits, const int64_t* __restrict__ targets, int V,
                                                                       int64_t ignore, float* __restrict__ row_max, float* __restrict__ row_log_sum,
                                                                       float* __restrict__ row_loss) {
    constexpr int W = CeRow<ET>::W, UN = 4;
    typedef __attribute__((ext_vector_type(W))) ET vec;
    const int64_t row = blockIdx.x;
    const ET* p = logits + row * V;
    const CeRow<ET> r(p, V);
    const vec* body = reinterpret_cast<const vec*>(p + r.head);
    MaxSum acc = {-INFINITY, 0.f};
    bool nan = false;
    auto take = [&](const float (&x)[W]) {
        float hi = x[0];
#pragma unroll
        for (int j = 1; j < W; ++j) hi = fmaxf(hi, x[j]);
        if (hi > acc.m) {
            acc.s *= fast_exp2((acc.m - hi) * kLog2e);
            acc.m = hi;
        }
        const float base = acc.m == -INFINITY ? 0.f : acc.m;
        float t = 0.f;
#pragma unroll
        for (int j = 0; j < W; ++j) t += fast_exp2((x[j] - base) * kLog2e);
        acc.s += t;
    };
    auto one = [&](float v) {
        nan |= v != v;
        acc.merge(v, 1.f);
    };
    if ((int)threadIdx.x < r.head) one((float)p[threadIdx.x]);
    if ((int)threadIdx.x < r.tail) one((float)p[r.head + r.vecs * W + threadIdx.x]);
    int i = threadIdx.x;
    for (; i + (UN - 1) * kCeThreads < r.vecs; i += UN * kCeThreads) {
        vec v[UN];
#pragma unroll
        for (int u = 0; u < UN; ++u) v[u] = body[i + u * kCeThreads];
#pragma unroll
        for (int u = 0; u < UN; ++u) {
            float x[W];
#pragma unroll
            for (int j = 0; j < W; ++j) x[j] = (float)v[u][j];
            take(x);
        }
    }
    for (; i < r.vecs; i += kCeThreads) {
        const vec v = body[i];
        float x[W];
#pragma unroll
        for (int j = 0; j < W; ++j) x[j] = (float)v[j];
        take(x);
    }
    nan |= acc.s != acc.s;
    merge_lanes<32>(acc);
    __shared__ float ms[kCeThreads / MTS_WAVE], ss[kCeThreads / MTS_WAVE];
    const int any_nan = __syncthreads_or(nan);
    if (threadIdx.x % MTS_WAVE == 0) {
        ms[threadIdx.x / MTS_WAVE] = acc.m;
        ss[threadIdx.x / MTS_WAVE] = acc.s;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        acc = {ms[0], ss[0]};
#pragma unroll
        for (int k = 1; k < kCeThreads / MTS_WAVE; ++k) acc.merge(ms[k], ss[k]);
        const float l = any_nan ? NAN : logf(acc.s);
        row_max[row] = acc.m;
        row_log_sum[row] = l;
        const int64_t t = targets[row];
        // a target outside the vocabulary gives NaN rather than a read outside the row
        row_loss[row] = t == ignore ? 0.f : ((t < 0 || t >= V) ? NAN : l - ((float)p[t] - acc.m));
    }
}

// mean over the rows whose target is not `ignore` (0/0 = NaN when there is none), sums in a fixed order
constexpr int kCeMeanThreads = 1024;
__global__ __launch_bounds__(kCeMeanThreads) void cross_entropy_mean_kernel(const float* __restrict__ row_loss, const int64_t* __restrict__ targets,
                                                                            int64_t N, int64_t ignore, float* __restrict__ loss,
                                                                            float* __restrict__ inv_count) {
    float s = 0.f, c = 0.f;
#pragma unroll 4
    for (int64_t i = threadIdx.x; i < N; i += kCeMeanThreads) {
        s += row_loss[i];
        c += targets[i] == ignore ? 0.f : 1.f;   // at most 2^24 rows per thread: exact
    }
    s = wave_sum(s), c = wave_sum(c);
    __shared__ float ls[kCeMeanThreads / MTS_WAVE], lc[kCeMeanThreads / MTS_WAVE];
    if (threadIdx.x % MTS_WAVE == 0) ls[threadIdx.x / MTS_WAVE] = s, lc[threadIdx.x / MTS_WAVE] = c;
    __syncthreads();
    if (threadIdx.x == 0) {
        double ts = 0, tc = 0;
        for (int k = 0; k < kCeMeanThreads / MTS_WAVE; ++k) ts += ls[k], tc += lc[k];
        *loss = (float)(ts / tc);
        *inv_count = (float)(1.0 / tc);
    }
}

// d_logits = (softmax - onehot) * g / count, zero where the target is ignored, NaN as the loss where it is outside the vocabulary.
// PITCHED: rows of d_logits start on 16 bytes, pitch elements apart, whatever V is (the projection's gradients read them so); the 16-byte
// pieces then follow the output and are read from wherever they lie in the logits.  Memory-bound either way: 24 576 rows of 50 257 949 us dense,
// 900 to 960 pitched (5.3 TB/s).
template <typename ET, bool PITCHED>
__global__ __launch_bounds__(kCeThreads) void cross_entropy_bwd_kernel(const ET* __restrict__ logits, const int64_t* __restrict__ targets, int V,
                                                                       int64_t ignore, const float* __restrict__ row_max,
                                                                       const float* __restrict__ row_log_sum, const float* __restrict__ g,
                                                                       const float* __restrict__ inv_count, ET* __restrict__ d_logits, int64_t pitch,
                                                                       bool unless_one) {
    if (unless_one && *g == 1.f) return;   // d_logits is that gradient already
    constexpr int W = CeRow<ET>::W, UN = 4;
    typedef __attribute__((ext_vector_type(W))) ET vec;
    typedef __attribute__((ext_vector_type(W), aligned(PITCHED ? sizeof(ET) : 16))) ET in_vec;
    const int64_t row = blockIdx.x;
    const int64_t target = targets[row];
    const ET* p = logits + row * V;
    ET* d = d_logits + row * (PITCHED ? pitch : V);
    const CeRow<ET> r(PITCHED ? d : p, V);
    const float scale = target == ignore ? 0.f : ((target < 0 || target >= V) ? NAN : *g * *inv_count);
    // maximum and logarithm of the sum apart: their sum would carry the rounding of a large maximum into every probability
    const float hi = row_max[row], base = row_log_sum[row] * kLog2e;
    const int t = (int)target;
    auto grad = [&](float x, int col) {
        const float q = fast_exp2((x - hi) * kLog2e - base);
        return (ET)(target == ignore ? 0.f : (col == t ? q - 1.f : q) * scale);
    };
    if ((int)threadIdx.x < r.head) d[threadIdx.x] = grad((float)p[threadIdx.x], threadIdx.x);
    if ((int)threadIdx.x < r.tail) {
        const int c = r.head + r.vecs * W + threadIdx.x;
        d[c] = grad((float)p[c], c);
    }
    const in_vec* body = reinterpret_cast<const in_vec*>(p + r.head);
    vec* out = reinterpret_cast<vec*>(d + r.head);
    int i = threadIdx.x;
    for (; i < r.vecs; i += UN * kCeThreads) {
        vec v[UN];
#pragma unroll
        for (int u = 0; u < UN; ++u)
            if (i + u * kCeThreads < r.vecs) v[u] = body[i + u * kCeThreads];
#pragma unroll
        for (int u = 0; u < UN; ++u) {
            const int k = i + u * kCeThreads;
            if (k >= r.vecs) break;
            vec o;
#pragma unroll
            for (int j = 0; j < W; ++j) o[j] = grad((float)v[u][j], r.head + k * W + j);
            out[k] = o;
        }
    }
}

// Loss and gradient of a row at once, for a loss that nothing scales: the row stays in registers between the two, so that the logits
// are read once (4.9 GB for 24 576 rows of 50 257 in the place of 7.4) where a forward and a backward launch read them twice.
// Two blocks a CU, one of them streams while the other adds up; rows of d_logits as in the PITCHED backward kernel.  24 576 rows of 50 257:
// 1050 us (4.7 TB/s) for 405 + 960; the training step around it 14.87 -> 14.49 ms.
template <typename ET, int THREADS, int NV>
__global__ __launch_bounds__(THREADS, 8) void cross_entropy_both_kernel(const ET* __restrict__ logits, const int64_t* __restrict__ targets, int V, int64_t ignore,
                                                                        float* __restrict__ row_max, float* __restrict__ row_log_sum,
                                                                        float* __restrict__ row_loss, const float* __restrict__ inv_count,
                                                                        ET* __restrict__ d_logits, int64_t pitch) {
    constexpr int W = 8, WAVES = THREADS / MTS_WAVE;
    static_assert(sizeof(ET) == 2 && WAVES <= 16, "rows of a 16-bit type");
    typedef __attribute__((ext_vector_type(W))) ET vec;
    typedef __attribute__((ext_vector_type(W), aligned(sizeof(ET)))) ET in_vec;
    const int64_t row = blockIdx.x;
    const ET* p = logits + row * V;
    ET* d = d_logits + row * pitch;
    const int tid = threadIdx.x, vecs = V / W, tail = V % W;
    const in_vec* body = reinterpret_cast<const in_vec*>(p);
    vec v[NV];
#pragma unroll
    for (int u = 0; u < NV; ++u)
        if (u * THREADS < vecs) v[u] = body[min(tid + u * THREADS, vecs - 1)];
    const float last = tid < tail ? (float)p[vecs * W + tid] : -INFINITY;
    const int64_t target = targets[row];
    const float at_target = target >= 0 && target < V ? (float)p[target] : 0.f, share = *inv_count;
    MaxSum acc = {last, last == -INFINITY ? 0.f : 1.f};
    bool nan = last != last;
    if (nan) acc.m = -INFINITY;
    float hi = -INFINITY;
#pragma unroll
    for (int u = 0; u < NV; ++u)
        if (tid + u * THREADS < vecs)
#pragma unroll
            for (int j = 0; j < W; ++j) hi = fmaxf(hi, (float)v[u][j]);
    float sum = 0.f;
    const float from = hi == -INFINITY ? 0.f : hi;
#pragma unroll
    for (int u = 0; u < NV; ++u)
        if (tid + u * THREADS < vecs)
#pragma unroll
            for (int j = 0; j < W; ++j) sum += fast_exp2(((float)v[u][j] - from) * kLog2e);
    nan |= sum != sum;
    acc.merge(hi, sum);
    merge_lanes<32>(acc);
    __shared__ float ms[16], ss[16];
    const int any_nan = __syncthreads_or(nan);
    if (tid % MTS_WAVE == 0) ms[tid / MTS_WAVE] = acc.m, ss[tid / MTS_WAVE] = acc.s;
    __syncthreads();
    const int from_wave = tid % 16 < WAVES ? tid % 16 : 0;
    acc = {tid % 16 < WAVES ? ms[from_wave] : -INFINITY, tid % 16 < WAVES ? ss[from_wave] : 0.f};
    merge_lanes<8>(acc);
    // lane 0's: the two sides of a merge may differ in the last bit
    const float top = __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(acc.m)));
    const float total = __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(acc.s)));
    const float log_sum = any_nan ? NAN : logf(total);
    const bool ignored = target == ignore, inside = target >= 0 && target < V;
    if (tid == 0) {
        row_max[row] = top;
        row_log_sum[row] = log_sum;
        row_loss[row] = ignored ? 0.f : (inside ? log_sum - (at_target - top) : NAN);
    }
    vec* out = reinterpret_cast<vec*>(d);
    if (ignored) {
#pragma unroll
        for (int u = 0; u < NV; ++u)
            if (tid + u * THREADS < vecs) out[tid + u * THREADS] = vec{};
        if (tid < tail) d[vecs * W + tid] = (ET)0.f;
        return;
    }
    const float scale = inside ? share : NAN, base = log_sum * kLog2e;
    const int t = inside ? (int)target : -1;
    auto probability = [&](float x) { return fast_exp2((x - top) * kLog2e - base); };
#pragma unroll
    for (int u = 0; u < NV; ++u) {
        const int i = tid + u * THREADS;
        if (i >= vecs) break;
        vec o;
#pragma unroll
        for (int j = 0; j < W; ++j) o[j] = (ET)(probability((float)v[u][j]) * scale);
        if (i == t / W) {
#pragma unroll
            for (int j = 0; j < W; ++j)
                if (t == i * W + j) o[j] = (ET)((probability((float)v[u][j]) - 1.f) * scale);
        }
        out[i] = o;
    }
    if (tid < tail) {
        const int c = vecs * W + tid;
        d[c] = (ET)((c == t ? probability(last) - 1.f : probability(last)) * scale);
    }
}

// 1 / the rows whose target is not `ignore`
__global__ __launch_bounds__(kCeMeanThreads) void cross_entropy_count_kernel(const int64_t* __restrict__ targets, int64_t N, int64_t ignore,
                                                                             float* __restrict__ inv_count) {
    float c = 0.f;
#pragma unroll 8
    for (int64_t i = threadIdx.x; i < N; i += kCeMeanThreads) c += targets[i] == ignore ? 0.f : 1.f;
    c = wave_sum(c);
    __shared__ float lc[kCeMeanThreads / MTS_WAVE];
    if (threadIdx.x % MTS_WAVE == 0) lc[threadIdx.x / MTS_WAVE] = c;
    __syncthreads();
    if (threadIdx.x == 0) {
        double tc = 0;
        for (int k = 0; k < kCeMeanThreads / MTS_WAVE; ++k) tc += lc[k];
        *inv_count = (float)(1.0 / tc);
    }
}

constexpr int kBothMost = 8 * 1024 * 8;   // columns that the registers of a block hold

template <typename ET>
void launch_both(const void* logits, const int64_t* targets, int64_t N, int V, int64_t ignore, float* row_max, float* row_log_sum, float* row_loss,
                 const float* inv_count, void* d_logits, int64_t pitch, hipStream_t st) {
    auto launch = [&](auto threads, auto nv) {
        constexpr int T = decltype(threads)::value;
        cross_entropy_both_kernel<ET, T, decltype(nv)::value><<<dim3((unsigned)N), dim3(T), 0, st>>>((const ET*)logits, targets, V, ignore, row_max, row_log_sum,
                                                                                                     row_loss, inv_count, (ET*)d_logits, pitch);
    };
    // as many threads as leave each a few pieces to have in flight
    const int vecs = V / 8;
    if (vecs <= 256) launch(std::integral_constant<int, 256>(), std::integral_constant<int, 1>());
    else if (vecs <= 1024) launch(std::integral_constant<int, 256>(), std::integral_constant<int, 4>());
    else if (vecs <= 2048) launch(std::integral_constant<int, 512>(), std::integral_constant<int, 4>());
    else if (vecs <= 4096) launch(std::integral_constant<int, 1024>(), std::integral_constant<int, 4>());
    else if (vecs <= 7168) launch(std::integral_constant<int, 1024>(), std::integral_constant<int, 7>());
    else launch(std::integral_constant<int, 1024>(), std::integral_constant<int, 8>());
}

bool dense_dtype_ok(int dtype) { return dtype == MTS_BF16 || dtype == MTS_F32 || dtype == MTS_F16; }

// ---------------------------------------------------------------------------
// Numbers of a model's layers: the means of its routers' losses and monitoring records, and the loss as their sum.  A launch
// each where stock operators take two a quantity (12 layers: 29 launches of 2 to 5 us; a pass of 640 tokens through two layers is
// bound by the host that makes them).
// ---------------------------------------------------------------------------

struct MeanTable {
    const void* src[MTS_MEAN_TENSORS];
    float* out[MTS_MEAN_GROUPS];
    int n[MTS_MEAN_GROUPS];
    uint16_t first[MTS_MEAN_GROUPS + 1];
    uint8_t whole[MTS_MEAN_GROUPS];
};
static_assert(sizeof(MeanTable) <= 4096, "kernel arguments");

constexpr int kMeanThreads = 64;
template <typename T>
__device__ __forceinline__ float mean_at(const void* const* src, int count, int i) {
    float sum = 0.f;
    for (int l = 0; l < count; ++l) sum += (float)static_cast<const T*>(src[l])[i];
    return sum / (float)count;
}
__global__ __launch_bounds__(kMeanThreads) void layer_means_kernel(MeanTable t) {
    const int g = blockIdx.x, first = t.first[g], count = t.first[g + 1] - first;
    for (int i = threadIdx.x; i < t.n[g]; i += kMeanThreads)
        t.out[g][i] = t.whole[g] ? mean_at<int64_t>(t.src + first, count, i) : mean_at<float>(t.src + first, count, i);
}

struct ScalarSums {
    const float* in[4];
    float* out[4];
    float weight[4][4], divisor[4];
    int inputs, terms[4];
};
__global__ void scalar_sums_kernel(ScalarSums p) {
#pragma clang fp contract(off)
    const int j = threadIdx.x;
    float sum = 0.f;
    for (int i = 0; i < p.inputs; ++i)
        if (p.terms[j] >> i & 1) sum += p.weight[j][i] * *p.in[i];
    *p.out[j] = sum / p.divisor[j];
}

}  // namespace

extern "C" int mts_rmsnorm_supported(int H) { return H > 0 && H % 4 == 0 && norm_groups(H) > 0; }

extern "C" int mts_rmsnorm_fwd(const void* x, const void* residual, const float* weight, int64_t N, int H, float eps, int act_dtype, void* sum,
                               void* y, float* rstd, void* stream) {
    if (!x || !weight || !y || !rstd || (residual && !sum)) return MTS_ERR_NULL;
    if (N <= 0 || N >= MTS_MAX_NORM_ROWS || !mts_rmsnorm_supported(H)) return MTS_ERR_SHAPE;
    if (!dense_dtype_ok(act_dtype)) return MTS_ERR_DTYPE;
    if (!mts_aligned16(x) || !mts_aligned16(residual) || !mts_aligned16(weight) || !mts_aligned16(sum) || !mts_aligned16(y)) return MTS_ERR_ALIGN;
    hipStream_t st = (hipStream_t)stream;
    const int nv = norm_groups(H);
    void* s = residual ? sum : nullptr;
    if (act_dtype == MTS_BF16) { MTS_NORM_DISPATCH(launch_norm_fwd, bf16_t, nv, x, residual, weight, N, H, eps, s, y, rstd, st) }
    else if (act_dtype == MTS_F16) { MTS_NORM_DISPATCH(launch_norm_fwd, mts_f16_t, nv, x, residual, weight, N, H, eps, s, y, rstd, st) }
    else { MTS_NORM_DISPATCH(launch_norm_fwd, float, nv, x, residual, weight, N, H, eps, s, y, rstd, st) }
    MTS_CHECK_LAUNCH();
    return MTS_OK;
}

extern "C" int64_t mts_rmsnorm_bwd_workspace_bytes(int64_t N, int H) { return (int64_t)norm_bwd_blocks(N) * H * 4; }

extern "C" int mts_rmsnorm_bwd(const void* g_y, const void* g_sum, const void* sum, const float* weight, const float* rstd, int64_t N, int H,
                               int act_dtype, void* d_sum, float* d_weight, void* workspace, int64_t workspace_bytes, void* stream) {
    if (!g_y || !sum || !weight || !rstd || !d_sum || !d_weight || !workspace) return MTS_ERR_NULL;
    if (N <= 0 || N >= MTS_MAX_NORM_ROWS || !mts_rmsnorm_supported(H)) return MTS_ERR_SHAPE;
    if (!dense_dtype_ok(act_dtype)) return MTS_ERR_DTYPE;
    if (workspace_bytes < mts_rmsnorm_bwd_workspace_bytes(N, H)) return MTS_ERR_WORKSPACE;
    if (!mts_aligned16(g_y) || !mts_aligned16(g_sum) || !mts_aligned16(sum) || !mts_aligned16(weight) || !mts_aligned16(d_sum) ||
        !mts_aligned16(workspace))
        return MTS_ERR_ALIGN;
    hipStream_t st = (hipStream_t)stream;
    const int nv = norm_groups(H), blocks = norm_bwd_blocks(N);
    float* part = (float*)workspace;
    if (act_dtype == MTS_BF16) { MTS_NORM_DISPATCH(launch_norm_bwd, bf16_t, nv, g_y, g_sum, sum, weight, rstd, N, H, d_sum, part, blocks, st) }
    else if (act_dtype == MTS_F16) { MTS_NORM_DISPATCH(launch_norm_bwd, mts_f16_t, nv, g_y, g_sum, sum, weight, rstd, N, H, d_sum, part, blocks, st) }
    else { MTS_NORM_DISPATCH(launch_norm_bwd, float, nv, g_y, g_sum, sum, weight, rstd, N, H, d_sum, part, blocks, st) }
    MTS_CHECK_LAUNCH();
    rmsnorm_dw_kernel<<<dim3((H + 63) / 64), dim3(64 * kNormRedGroups), 0, st>>>(part, blocks, H, d_weight);
    MTS_CHECK_LAUNCH();
    return MTS_OK;
}

extern "C" int mts_rope(const MtsRopeTensor* tensors, int count, const void* cos, const void* sin, int64_t B, int64_t S, int heads, int head_dim,
                        int act_dtype, void* stream) {
    if (!tensors || !cos || !sin) return MTS_ERR_NULL;
    if (count < 1 || count > 3 || B <= 0 || S <= 0 || heads <= 0 || head_dim <= 0 || head_dim % 2) return MTS_ERR_SHAPE;
    if (B * S * heads * (head_dim / 2) >= MTS_MAX_ROPE_PAIRS) return MTS_ERR_SHAPE;
    for (int i = 0; i < count; ++i) {
        if (!tensors[i].in || !tensors[i].out) return MTS_ERR_NULL;
        if (tensors[i].mode < ROPE_TURN || tensors[i].mode > ROPE_COPY) return MTS_ERR_SHAPE;
    }
    hipStream_t st = (hipStream_t)stream;
    switch (act_dtype) {
        case MTS_BF16: return launch_rope<bf16_t>(tensors, count, cos, sin, B, S, heads, head_dim, st);
        case MTS_F16: return launch_rope<mts_f16_t>(tensors, count, cos, sin, B, S, heads, head_dim, st);
        case MTS_F32: return launch_rope<float>(tensors, count, cos, sin, B, S, heads, head_dim, st);
    }
    return MTS_ERR_DTYPE;
}

extern "C" int mts_cross_entropy_fwd(const void* logits, const int64_t* targets, int64_t N, int V, int64_t ignore_index, int dtype, float* row_max,
                                     float* row_log_sum, float* row_loss, float* loss, float* inv_count, void* stream) {
    if (!logits || !targets || !row_max || !row_log_sum || !row_loss || !loss || !inv_count) return MTS_ERR_NULL;
    if (N <= 0 || N >= MTS_MAX_LOSS_ROWS || V <= 0) return MTS_ERR_SHAPE;
    if (!dense_dtype_ok(dtype)) return MTS_ERR_DTYPE;
    if (!mts_aligned16(logits)) return MTS_ERR_ALIGN;
    hipStream_t st = (hipStream_t)stream;
    const dim3 grid((unsigned)N), block(kCeThreads);
    if (dtype == MTS_BF16) cross_entropy_fwd_kernel<bf16_t><<<grid, block, 0, st>>>((const bf16_t*)logits, targets, V, ignore_index, row_max, row_log_sum, row_loss);
    else if (dtype == MTS_F16) cross_entropy_fwd_kernel<mts_f16_t><<<grid, block, 0, st>>>((const mts_f16_t*)logits, targets, V, ignore_index, row_max, row_log_sum, row_loss);
    else cross_entropy_fwd_kernel<float><<<grid, block, 0, st>>>((const float*)logits, targets, V, ignore_index, row_max, row_log_sum, row_loss);
    MTS_CHECK_LAUNCH();
    cross_entropy_mean_kernel<<<1, kCeMeanThreads, 0, st>>>(row_loss, targets, N, ignore_index, loss, inv_count);
    MTS_CHECK_LAUNCH();
    return MTS_OK;
}

template <bool PITCHED>
static int cross_entropy_bwd(const void* logits, const int64_t* targets, int64_t N, int V, int64_t ignore_index, int dtype, const float* row_max,
                             const float* row_log_sum, const float* g_loss, const float* inv_count, void* d_logits, int64_t pitch, void* stream,
                             bool unless_one = false) {
    if (!logits || !targets || !row_max || !row_log_sum || !g_loss || !inv_count || !d_logits) return MTS_ERR_NULL;
    if (N <= 0 || N >= MTS_MAX_LOSS_ROWS || V <= 0 || (PITCHED && (pitch < V || pitch % 8))) return MTS_ERR_SHAPE;
    if (!dense_dtype_ok(dtype)) return MTS_ERR_DTYPE;
    if (!mts_aligned16(logits) || !mts_aligned16(d_logits)) return MTS_ERR_ALIGN;
    hipStream_t st = (hipStream_t)stream;
    const dim3 grid((unsigned)N), block(kCeThreads);
    if (dtype == MTS_BF16)
        cross_entropy_bwd_kernel<bf16_t, PITCHED><<<grid, block, 0, st>>>((const bf16_t*)logits, targets, V, ignore_index, row_max, row_log_sum, g_loss, inv_count,
                                                                          (bf16_t*)d_logits, pitch, unless_one);
    else if (dtype == MTS_F16)
        cross_entropy_bwd_kernel<mts_f16_t, PITCHED><<<grid, block, 0, st>>>((const mts_f16_t*)logits, targets, V, ignore_index, row_max, row_log_sum, g_loss, inv_count,
                                                                             (mts_f16_t*)d_logits, pitch, unless_one);
    else
        cross_entropy_bwd_kernel<float, PITCHED><<<grid, block, 0, st>>>((const float*)logits, targets, V, ignore_index, row_max, row_log_sum, g_loss, inv_count,
                                                                         (float*)d_logits, pitch, unless_one);
    MTS_CHECK_LAUNCH();
    return MTS_OK;
}
extern "C" int mts_cross_entropy_bwd(const void* logits, const int64_t* targets, int64_t N, int V, int64_t ignore_index, int dtype, const float* row_max,
                                     const float* row_log_sum, const float* g_loss, const float* inv_count, void* d_logits, void* stream) {
    return cross_entropy_bwd<false>(logits, targets, N, V, ignore_index, dtype, row_max, row_log_sum, g_loss, inv_count, d_logits, V, stream);
}
extern "C" int mts_cross_entropy_bwd_pitched(const void* logits, const int64_t* targets, int64_t N, int V, int64_t ignore_index, int dtype, const float* row_max,
                                             const float* row_log_sum, const float* g_loss, const float* inv_count, void* d_logits, int64_t pitch, void* stream) {
    return cross_entropy_bwd<true>(logits, targets, N, V, ignore_index, dtype, row_max, row_log_sum, g_loss, inv_count, d_logits, pitch, stream);
}

extern "C" int mts_cross_entropy_both_supported(int V, int dtype) { return V >= 8 && V <= kBothMost && (dtype == MTS_BF16 || dtype == MTS_F16) ? 1 : 0; }

extern "C" int mts_cross_entropy_both(const void* logits, const int64_t* targets, int64_t N, int V, int64_t ignore_index, int dtype, float* row_max,
                                      float* row_log_sum, float* row_loss, float* loss, float* inv_count, void* d_logits, int64_t pitch, void* stream) {
    if (!logits || !targets || !row_max || !row_log_sum || !row_loss || !loss || !inv_count || !d_logits) return MTS_ERR_NULL;
    if (N <= 0 || N >= MTS_MAX_LOSS_ROWS || V <= 0 || pitch < V || pitch % 8) return MTS_ERR_SHAPE;
    if (!dense_dtype_ok(dtype)) return MTS_ERR_DTYPE;
    if (!mts_cross_entropy_both_supported(V, dtype)) return MTS_ERR_SHAPE;
    if (!mts_aligned16(logits) || !mts_aligned16(d_logits)) return MTS_ERR_ALIGN;
    hipStream_t st = (hipStream_t)stream;
    cross_entropy_count_kernel<<<1, kCeMeanThreads, 0, st>>>(targets, N, ignore_index, inv_count);
    MTS_CHECK_LAUNCH();
    if (dtype == MTS_BF16) launch_both<bf16_t>(logits, targets, N, V, ignore_index, row_max, row_log_sum, row_loss, inv_count, d_logits, pitch, st);
    else launch_both<mts_f16_t>(logits, targets, N, V, ignore_index, row_max, row_log_sum, row_loss, inv_count, d_logits, pitch, st);
    MTS_CHECK_LAUNCH();
    cross_entropy_mean_kernel<<<1, kCeMeanThreads, 0, st>>>(row_loss, targets, N, ignore_index, loss, inv_count);
    MTS_CHECK_LAUNCH();
    return MTS_OK;
}

extern "C" int mts_cross_entropy_bwd_unless_one(const void* logits, const int64_t* targets, int64_t N, int V, int64_t ignore_index, int dtype, const float* row_max,
                                                const float* row_log_sum, const float* g_loss, const float* inv_count, void* d_logits, int64_t pitch, void* stream) {
    return cross_entropy_bwd<true>(logits, targets, N, V, ignore_index, dtype, row_max, row_log_sum, g_loss, inv_count, d_logits, pitch, stream, true);
}

extern "C" int mts_layer_means(const void* const* src, const int* first, const int* n, const int* whole, int groups, float* const* out, void* stream) {
    if (!src || !first || !n || !whole || !out) return MTS_ERR_NULL;
    if (groups < 1 || groups > MTS_MEAN_GROUPS || first[0] != 0 || first[groups] > MTS_MEAN_TENSORS) return MTS_ERR_SHAPE;
    MeanTable t = {};
    for (int g = 0; g < groups; ++g) {
        if (first[g + 1] <= first[g] || n[g] < 1) return MTS_ERR_SHAPE;
        if (!out[g]) return MTS_ERR_NULL;
        t.out[g] = out[g], t.n[g] = n[g], t.whole[g] = whole[g] != 0, t.first[g + 1] = (uint16_t)first[g + 1];
    }
    for (int i = 0; i < first[groups]; ++i) {
        if (!src[i]) return MTS_ERR_NULL;
        t.src[i] = src[i];
    }
    layer_means_kernel<<<dim3((unsigned)groups), kMeanThreads, 0, (hipStream_t)stream>>>(t);
    MTS_CHECK_LAUNCH();
    return MTS_OK;
}

extern "C" int mts_scalar_sums(const float* const* in, int inputs, const float* weight, const int* terms, const float* divisor, float* const* out, int outputs,
                               void* stream) {
    if (!in || !weight || !terms || !divisor || !out) return MTS_ERR_NULL;
    if (inputs < 1 || inputs > 4 || outputs < 1 || outputs > 4) return MTS_ERR_SHAPE;
    ScalarSums p = {};
    p.inputs = inputs;
    for (int i = 0; i < inputs; ++i)
        if (!(p.in[i] = in[i])) return MTS_ERR_NULL;
    for (int j = 0; j < outputs; ++j) {
        if (!(p.out[j] = out[j])) return MTS_ERR_NULL;
        p.divisor[j] = divisor[j], p.terms[j] = terms[j];
        for (int i = 0; i < 4; ++i) p.weight[j][i] = weight[4 * j + i];
    }
    scalar_sums_kernel<<<1, outputs, 0, (hipStream_t)stream>>>(p);
    MTS_CHECK_LAUNCH();
    return MTS_OK;
}
