// The optimizer update of a training step: global norm of the gradients with the clipping coefficient, and AdamW (Loshchilov and
// Hutter, "Decoupled Weight Decay Regularization", 2019) on all parameters.
//
// Bound by HBM: the norm reads every gradient once, the update reads parameter, gradient and both moments once and writes three of
// them.  The coefficient is applied where the update reads the gradient, so no pass of its own scales the gradients, and the
// parameters of a model share one launch: a block finds its tensor from the launch's table (a step of a small model is otherwise a
// few hundred microseconds of launches).  162 M parameters of fp32 (a four-layer decoder with 50 257 words): norm 151 us (4.3 TB/s), update
// 824 us (5.5 TB/s; 946 where every gradient is written back), where stock clipping and fused AdamW took 200 + 277 and 1129 us, and some 60 us in small kernels; with them the
// step of 24 576 tokens 15.53 -> 14.62 ms with all gradients written back and another 0.12 less without, the rest of it from enqueuing the update ahead of the host's look at the flag.
#include "mts_common.h"

namespace {

constexpr int kThreads = 256;
constexpr int kNormChunk = 16384, kAdamChunk = 4096;   // elements a block takes
constexpr int kNormSpans = 128, kAdamTensors = 56;     // per launch: the tables travel as kernel arguments, of which there are 4 KiB

__device__ __forceinline__ bool on16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

struct NormTable {
    const float* grad[kNormSpans];
    int64_t n[kNormSpans];
    int first_block[kNormSpans];
    int count;
};

// The entry that block `b` belongs to: the last whose first block is not behind it.
template <int MOST>
__device__ __forceinline__ int entry_of(const int (&first_block)[MOST], int count, int b) {
    const int lane = threadIdx.x % MTS_WAVE;
    int before = 0;
#pragma unroll
    for (int i = 0; i < MOST; i += MTS_WAVE) before += __popcll(__ballot(i + lane < count && first_block[i + lane < MOST ? i + lane : 0] <= b));
    return __builtin_amdgcn_readfirstlane(before) - 1;
}

__device__ __forceinline__ double block_sum(double v) {
    __shared__ double part[kThreads / MTS_WAVE];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
    if (threadIdx.x % MTS_WAVE == 0) part[threadIdx.x / MTS_WAVE] = v;
    __syncthreads();
    double s = 0;
#pragma unroll
    for (int i = 0; i < kThreads / MTS_WAVE; ++i) s += part[i];
    return s;
}

// partial[b] = sum of the squares of a chunk: fp32 within a thread (64 values), fp64 from there on
__global__ __launch_bounds__(kThreads) void grad_norm_kernel(NormTable t, double* __restrict__ partial) {
    const int e = entry_of(t.first_block, t.count, blockIdx.x);
    const float* g = t.grad[e] + (int64_t)(blockIdx.x - t.first_block[e]) * kNormChunk;
    const int64_t left = t.n[e] - (int64_t)(blockIdx.x - t.first_block[e]) * kNormChunk;
    const int n = left < kNormChunk ? (int)left : kNormChunk;
    f32x4 s = {};
    if (on16(g) && n == kNormChunk) {
        constexpr int kLoads = 8;
        for (int i = threadIdx.x * 4; i < kNormChunk; i += kLoads * kThreads * 4) {
            f32x4 v[kLoads];
#pragma unroll
            for (int q = 0; q < kLoads; ++q) v[q] = *reinterpret_cast<const f32x4*>(g + i + q * kThreads * 4);
#pragma unroll
            for (int q = 0; q < kLoads; ++q) s += v[q] * v[q];
        }
    } else {
        for (int i = threadIdx.x; i < n; i += kThreads) s[0] += g[i] * g[i];
    }
    const double sum = block_sum((double)s[0] + (double)s[1] + (double)s[2] + (double)s[3]);
    if (threadIdx.x == 0) partial[blockIdx.x] = sum;
}

// result: norm, min(1, max_norm / (norm + 1e-6)), and 1 where the norm or the loss is not finite
__global__ __launch_bounds__(kThreads) void grad_norm_finish_kernel(const double* __restrict__ partial, int count, float max_norm,
                                                                    const float* __restrict__ loss, float* __restrict__ result) {
    double v = 0;
    for (int i = threadIdx.x; i < count; i += kThreads) v += partial[i];
    const float sum = (float)block_sum(v);   // a sum that leaves the range of fp32 is an infinite norm
    if (threadIdx.x != 0) return;
    const float norm = sqrtf(sum), coefficient = max_norm / (norm + 1e-6f);
    result[0] = norm;
    result[1] = count && !(coefficient > 1.f) ? coefficient : 1.f;   // NaN stays
    result[2] = __builtin_isfinite(norm) && (!loss || __builtin_isfinite(*loss)) ? 0.f : 1.f;
}

struct AdamTable {
    float* param[kAdamTensors];
    float* grad[kAdamTensors];
    float* exp_avg[kAdamTensors];
    float* exp_avg_sq[kAdamTensors];
    float* step[kAdamTensors];
    int64_t n[kAdamTensors];
    int first_block[kAdamTensors];
    int group[kAdamTensors];   // and kKeep: the clipped gradient is written back
    int count;
};
constexpr int kKeep = 1 << 16;
static_assert(sizeof(AdamTable) + sizeof(MtsAdamGroup) * MTS_ADAM_GROUPS + 64 <= 4096, "kernel arguments");
struct AdamGroups {
    MtsAdamGroup of[MTS_ADAM_GROUPS];
};

// one thread a tensor: its step, and from it lr / (1 - beta1^step) and sqrt(1 - beta2^step)
__global__ __launch_bounds__(MTS_WAVE) void adamw_advance_kernel(AdamTable t, AdamGroups groups, const float* __restrict__ skip,
                                                                  float2* __restrict__ factors) {
    const int i = threadIdx.x;
    if (i >= t.count || (skip && *skip != 0.f)) return;
    const MtsAdamGroup g = groups.of[t.group[i] & (kKeep - 1)];
    const float step = *t.step[i] + 1.f;
    *t.step[i] = step;
    factors[i] = {(float)(g.lr / (1.0 - pow(g.beta1, (double)step))), (float)sqrt(1.0 - pow(g.beta2, (double)step))};
}

// The moments and the decay are formed in fp64 and rounded once, as the stock fused operator does; the quotient is fp32.
struct AdamStep {
    double beta1, beta2, eps, kept;   // kept: 1 - lr * weight_decay
    float size, root, clip;
    __device__ __forceinline__ void operator()(float& p, float& g, float& m, float& v) const {
        g *= clip;
        m = (float)(beta1 * m + (1.0 - beta1) * g);
        v = (float)(beta2 * v + (1.0 - beta2) * g * g);
        const float denominator = (float)((double)(sqrtf(v) / root) + eps);
        p = (float)(kept * p) - size * m / denominator;
    }
};

__global__ __launch_bounds__(kThreads) void adamw_kernel(AdamTable t, AdamGroups groups, const float* __restrict__ clip, const float* __restrict__ skip,
                                                         const float2* __restrict__ factors) {
    if (skip && *skip != 0.f) return;
    const int e = entry_of(t.first_block, t.count, blockIdx.x);
    const int64_t first = (int64_t)(blockIdx.x - t.first_block[e]) * kAdamChunk, left = t.n[e] - first;
    const int n = left < kAdamChunk ? (int)left : kAdamChunk;
    const MtsAdamGroup h = groups.of[t.group[e] & (kKeep - 1)];
    const bool keep = t.group[e] & kKeep;
    const AdamStep update = {h.beta1, h.beta2, h.eps, 1.0 - h.lr * h.weight_decay, factors[e].x, factors[e].y, clip ? *clip : 1.f};
    float *p = t.param[e] + first, *g = t.grad[e] + first, *m = t.exp_avg[e] + first, *v = t.exp_avg_sq[e] + first;
    const bool whole = on16(p) && on16(g) && on16(m) && on16(v) && n % 4 == 0;
    if (!whole) {
        for (int i = threadIdx.x; i < n; i += kThreads) {
            float pv = p[i], gv = g[i], mv = m[i], vv = v[i];
            update(pv, gv, mv, vv);
            p[i] = pv, m[i] = mv, v[i] = vv;
            if (keep) g[i] = gv;
        }
        return;
    }
    constexpr int kAtOnce = 2;   // 8 loads of 16 bytes in flight a lane
    for (int i = threadIdx.x * 4; i < n; i += kAtOnce * kThreads * 4) {
        f32x4 pv[kAtOnce], gv[kAtOnce], mv[kAtOnce], vv[kAtOnce];
#pragma unroll
        for (int q = 0; q < kAtOnce; ++q) {
            const int at = i + q * kThreads * 4 < n ? i + q * kThreads * 4 : i;
            pv[q] = *reinterpret_cast<const f32x4*>(p + at), gv[q] = *reinterpret_cast<const f32x4*>(g + at);
            mv[q] = *reinterpret_cast<const f32x4*>(m + at), vv[q] = *reinterpret_cast<const f32x4*>(v + at);
        }
#pragma unroll
        for (int q = 0; q < kAtOnce; ++q) {
            const int at = i + q * kThreads * 4;
            if (at >= n) break;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                float a = pv[q][j], b = gv[q][j], c = mv[q][j], d = vv[q][j];
                update(a, b, c, d);
                pv[q][j] = a, gv[q][j] = b, mv[q][j] = c, vv[q][j] = d;
            }
            *reinterpret_cast<f32x4*>(p + at) = pv[q];
            *reinterpret_cast<f32x4*>(m + at) = mv[q];
            *reinterpret_cast<f32x4*>(v + at) = vv[q];
            if (keep) *reinterpret_cast<f32x4*>(g + at) = gv[q];
        }
    }
}

int64_t chunks(int64_t n, int chunk) { return (n + chunk - 1) / chunk; }
constexpr int64_t kMostBlocks = 1LL << 24;   // of 256 threads: a launch holds fewer than 2^32

}  // namespace

int64_t mts_grad_norm_workspace_bytes(const MtsGradSpan* grads, int count) {
    int64_t blocks = 0;
    for (int i = 0; i < count; ++i) blocks += chunks(grads[i].n, kNormChunk);
    return blocks * (int64_t)sizeof(double);
}

int mts_grad_norm(const MtsGradSpan* grads, int count, float max_norm, const float* loss, float* result, void* workspace, int64_t workspace_bytes,
                  void* stream) {
    if (!result || count < 0 || (count > 0 && (!grads || !workspace))) return MTS_ERR_NULL;
    if (workspace_bytes < mts_grad_norm_workspace_bytes(grads, count)) return MTS_ERR_WORKSPACE;
    double* partial = static_cast<double*>(workspace);
    const hipStream_t s = static_cast<hipStream_t>(stream);
    int64_t all = 0;
    for (int i = 0; i < count; ++i) {
        if (grads[i].n < 0 || (grads[i].n > 0 && !grads[i].data)) return MTS_ERR_NULL;
        all += chunks(grads[i].n, kNormChunk);
    }
    if (all >= kMostBlocks) return MTS_ERR_SHAPE;
    int64_t done = 0;
    for (int i = 0; i < count;) {
        NormTable t;
        t.count = 0;
        int64_t blocks = 0;
        for (; i < count && t.count < kNormSpans; ++i) {
            if (grads[i].n == 0) continue;
            t.grad[t.count] = grads[i].data, t.n[t.count] = grads[i].n, t.first_block[t.count] = (int)blocks;
            ++t.count;
            blocks += chunks(grads[i].n, kNormChunk);
        }
        if (blocks == 0) continue;
        grad_norm_kernel<<<dim3((unsigned)blocks), kThreads, 0, s>>>(t, partial + done);
        MTS_CHECK_LAUNCH();
        done += blocks;
    }
    grad_norm_finish_kernel<<<1, kThreads, 0, s>>>(partial, (int)done, max_norm, loss, result);
    MTS_CHECK_LAUNCH();
    return MTS_OK;
}

int64_t mts_adamw_workspace_bytes(int count) { return (int64_t)count * sizeof(float2); }

int mts_adamw(const MtsAdamTensor* tensors, int count, const MtsAdamGroup* groups, int n_groups, const float* clip, const float* skip, void* workspace,
              int64_t workspace_bytes, void* stream) {
    if (count < 0 || (count > 0 && (!tensors || !groups || !workspace))) return MTS_ERR_NULL;
    if (n_groups < 0 || n_groups > MTS_ADAM_GROUPS) return MTS_ERR_SHAPE;
    if (workspace_bytes < mts_adamw_workspace_bytes(count)) return MTS_ERR_WORKSPACE;
    for (int i = 0; i < count; ++i) {
        const MtsAdamTensor& a = tensors[i];
        if (!a.step || (a.n > 0 && (!a.param || !a.grad || !a.exp_avg || !a.exp_avg_sq))) return MTS_ERR_NULL;
        if (a.n < 0 || a.group < 0 || a.group >= n_groups || chunks(a.n, kAdamChunk) >= kMostBlocks / kAdamTensors) return MTS_ERR_SHAPE;
    }
    AdamGroups g = {};
    for (int i = 0; i < n_groups; ++i) g.of[i] = groups[i];
    const hipStream_t s = static_cast<hipStream_t>(stream);
    for (int i = 0; i < count; i += kAdamTensors) {
        AdamTable t;
        t.count = 0;
        int64_t blocks = 0;
        for (int j = i; j < count && j < i + kAdamTensors; ++j, ++t.count) {
            const MtsAdamTensor& a = tensors[j];
            t.param[t.count] = a.param, t.grad[t.count] = a.grad, t.exp_avg[t.count] = a.exp_avg, t.exp_avg_sq[t.count] = a.exp_avg_sq;
            t.step[t.count] = a.step, t.n[t.count] = a.n, t.first_block[t.count] = (int)blocks, t.group[t.count] = a.group | (a.keep_grad ? kKeep : 0);
            blocks += chunks(a.n, kAdamChunk);
        }
        float2* factors = static_cast<float2*>(workspace) + i;
        adamw_advance_kernel<<<1, MTS_WAVE, 0, s>>>(t, g, skip, factors);
        MTS_CHECK_LAUNCH();
        if (blocks == 0) continue;
        adamw_kernel<<<dim3((unsigned)blocks), kThreads, 0, s>>>(t, g, clip, skip, factors);
        MTS_CHECK_LAUNCH();
    }
    return MTS_OK;
}
