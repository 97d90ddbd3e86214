// The router projection of more than 16 experts: logits[t,e] = sum_h x[t,h] * w_r[e,h] with fp32 weights and fp32 sums, and
// its backward, on the fp32 matrix instruction; 16-bit activations are widened on their way into LDS, so there is no fp32
// copy of x and no cast of dx.  (Up to 16 experts the weights sit in LDS and the projection is a stream over x: see
// mts_router_linear.hip.)
//
// What bounds it: 2*T*H*E FLOP each way at the instruction's 157 TFLOP/s (7 us for 8192 x 1024 x 64, where x is 17 MB, 4 us),
// so what matters is that every SIMD has a share: forward, 32 rows x 64 experts per block with k dealt to its four waves;
// dW_r, whose outputs fill 16 blocks only, the rows cut into chunks and the partial sums added in chunk order.
// 8192 x 1024, 64 experts, bf16: 23 us forward, 20 + 20 + 6 us backward (the library's fp32 products with a widened copy of x
// and a narrowed dx took 24 and 110 us).
#include "mts_f32_tiles.h"

#include <type_traits>

namespace {

using namespace mts_f32;

constexpr int kThreads = kTileThreads;

// 32 rows x 64 experts; wave w multiplies k-steps 2w and 2w+1 of every 64-wide k-tile, the four sums meet in LDS
template <typename XT>
__global__ __launch_bounds__(kThreads) void wide_logits_kernel(const XT* __restrict__ x, const float* __restrict__ w, int64_t T, int H, int E,
                                                               float* __restrict__ logits) {
    constexpr int BM = 32, BN = 64, TKS = 64, STEPS = TKS / 8 / 4;
    typedef RowTile<XT, BM, TKS, true> AT;
    typedef RowTile<float, BN, TKS, true> BT;
    __shared__ __attribute__((aligned(16))) float As[2][AT::SIZE];
    __shared__ __attribute__((aligned(16))) float Bs[2][BT::SIZE];
    const int64_t row0 = (int64_t)blockIdx.x * BM;
    const int e0 = blockIdx.y * BN;
    AT a;
    BT b;
#pragma unroll
    for (int q = 0; q < AT::LOADS; ++q) {
        const int64_t r = row0 + AT::row(q);
        a.ptr[q] = r < T ? x + r * H : nullptr;
    }
#pragma unroll
    for (int q = 0; q < BT::LOADS; ++q) {
        const int e = e0 + BT::row(q);
        b.ptr[q] = e < E ? w + (int64_t)e * H : nullptr;
    }
    const int wave = threadIdx.x / MTS_WAVE, lane = threadIdx.x % MTS_WAVE;
    f32x16 acc[1][2] = {};
    auto fetch = [&](int set, int t) {
        a.fetch(set, t * TKS, H);
        b.fetch(set, t * TKS, H);
    };
    run_k_tiles<AT, BT, STEPS, 1, 2>((H + TKS - 1) / TKS, a, b, As, Bs, acc, [](int) { return 0; }, [](int nf) { return nf * 32; }, fetch, wave * STEPS);
    // the waves' sums, in wave order
    float* sums = &Bs[0][0];   // [32][64]
    static_assert(2 * BT::SIZE >= BM * BN, "the sums fit the weight buffers");
#pragma unroll 1
    for (int k = 0; k < 4; ++k) {
        if (wave == k) {
#pragma unroll
            for (int nf = 0; nf < 2; ++nf)
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    float* s = sums + (8 * (i / 4) + 4 * (lane / 32) + i % 4) * BN + nf * 32 + lane % 32;
                    *s = k ? *s + acc[0][nf][i] : acc[0][nf][i];
                }
        }
        __syncthreads();
    }
    for (int i = threadIdx.x; i < BM * BN; i += kThreads) {
        const int64_t r = row0 + i / BN;
        const int e = e0 + i % BN;
        if (r < T && e < E) logits[r * E + e] = sums[i];
    }
}

// dx[t,h] = sum_e dlogits[t,e] * w_r[e,h], 64 x 64 per block
template <typename XT, bool VEC>
__global__ __launch_bounds__(kThreads) void wide_dx_kernel(const float* __restrict__ dl, const float* __restrict__ w, int64_t T, int H, int E,
                                                           XT* __restrict__ dx) {
    constexpr int BM = 64, BN = 64, TKS = 16;
    typedef RowTile<float, BM, TKS, VEC> AT;
    typedef KTile<float, BN, TKS, true> BT;
    __shared__ __attribute__((aligned(16))) float As[2][AT::SIZE];
    __shared__ __attribute__((aligned(16))) float Bs[2][BT::SIZE];
    const int n_tiles = (H + BN - 1) / BN;
    const int64_t row0 = (int64_t)(blockIdx.x / n_tiles) * BM;
    const int n0 = blockIdx.x % n_tiles * BN;
    AT a;
    BT b;
#pragma unroll
    for (int q = 0; q < AT::LOADS; ++q) {
        const int64_t r = row0 + AT::row(q);
        a.ptr[q] = r < T ? dl + r * E : nullptr;
    }
    b.base = w + n0 + BT::col(), b.ld = H, b.cols = H - n0 - BT::col();
    const int wave = threadIdx.x / MTS_WAVE, lane = threadIdx.x % MTS_WAVE, wm = wave / 2, wn = wave % 2;
    f32x16 acc[1][1] = {};
    auto fetch = [&](int set, int t) {
        a.fetch(set, t * TKS, E);
        int64_t rows[BT::LOADS];
#pragma unroll
        for (int q = 0; q < BT::LOADS; ++q) rows[q] = t * TKS + BT::k(q) < E ? t * TKS + BT::k(q) : -1;
        b.fetch(set, rows);
    };
    run_k_tiles<AT, BT, TKS / 8, 1, 1>((E + TKS - 1) / TKS, a, b, As, Bs, acc, [&](int) { return wm * 32; }, [&](int) { return wn * 32; }, fetch);
    const int n = n0 + wn * 32 + lane % 32;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const int64_t r = row0 + wm * 32 + 8 * (i / 4) + 4 * (lane / 32) + i % 4;
        if (r < T && n < H) dx[r * H + n] = (XT)acc[0][0][i];
    }
}

// partial dW_r[e,h] over one chunk of rows, 64 x 64 per block
template <typename XT, bool VEC>
__global__ __launch_bounds__(kThreads) void wide_dw_kernel(const float* __restrict__ dl, const XT* __restrict__ x, int64_t T, int H, int E,
                                                           int64_t rows_per_chunk, float* __restrict__ part) {
    constexpr int BM = 64, BN = 64, TKS = 16;
    typedef KTile<float, BM, TKS, VEC> PT;
    typedef KTile<XT, BN, TKS, true> QT;
    __shared__ __attribute__((aligned(16))) float Ps[2][PT::SIZE];
    __shared__ __attribute__((aligned(16))) float Qs[2][QT::SIZE];
    const int m0 = blockIdx.y * BM, n0 = blockIdx.x * BN;
    const int64_t r0 = (int64_t)blockIdx.z * rows_per_chunk, r1 = r0 + rows_per_chunk < T ? r0 + rows_per_chunk : T;
    PT a;
    QT b;
    a.base = dl + m0 + PT::col(), a.ld = E, a.cols = E - m0 - PT::col();
    b.base = x + n0 + QT::col(), b.ld = H, b.cols = H - n0 - QT::col();
    const int wave = threadIdx.x / MTS_WAVE, lane = threadIdx.x % MTS_WAVE, wm = wave / 2, wn = wave % 2;
    f32x16 acc[1][1] = {};
    auto fetch = [&](int set, int t) {
        int64_t pr[PT::LOADS], qr[QT::LOADS];
#pragma unroll
        for (int q = 0; q < PT::LOADS; ++q) pr[q] = r0 + t * TKS + PT::k(q) < r1 ? r0 + t * TKS + PT::k(q) : -1;
#pragma unroll
        for (int q = 0; q < QT::LOADS; ++q) qr[q] = r0 + t * TKS + QT::k(q) < r1 ? r0 + t * TKS + QT::k(q) : -1;
        a.fetch(set, pr);
        b.fetch(set, qr);
    };
    run_k_tiles<PT, QT, TKS / 8, 1, 1>((int)((r1 - r0 + TKS - 1) / TKS), a, b, Ps, Qs, acc, [&](int) { return wm * 32; }, [&](int) { return wn * 32; }, fetch);
    float* out = part + (int64_t)blockIdx.z * E * H;
    const int n = n0 + wn * 32 + lane % 32;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const int m = m0 + wm * 32 + 8 * (i / 4) + 4 * (lane / 32) + i % 4;
        if (m < E && n < H) out[(int64_t)m * H + n] = acc[0][0][i];
    }
}

// Rows are cut into as many chunks as make about two blocks per CU, of at least 64 rows.
struct WideChunks {
    int64_t rows;
    int count;
};
WideChunks wide_chunks(int64_t T, int H, int E) {
    const int64_t tiles = (int64_t)((E + 63) / 64) * ((H + 63) / 64);
    int64_t count = (512 + tiles - 1) / tiles;
    const int64_t most = (T + 63) / 64;
    if (count > most) count = most;
    const int64_t rows = ((T + count - 1) / count + 15) / 16 * 16;
    return {rows, (int)((T + rows - 1) / rows)};
}

int wide_check(const void* x, const float* w_r, int64_t T, int H, int E, int act_dtype) {
    if (!x || !w_r) return MTS_ERR_NULL;
    if (!mts_router_wide_supported(H, E) || T <= 0 || (T + 63) / 64 * ((H + 63) / 64) >= (1LL << 31)) return MTS_ERR_SHAPE;
    if (act_dtype != MTS_BF16 && act_dtype != MTS_F16 && act_dtype != MTS_F32) return MTS_ERR_DTYPE;
    if (!mts_aligned16(x) || !mts_aligned16(w_r)) return MTS_ERR_ALIGN;
    return MTS_OK;
}

}  // namespace

extern "C" int mts_router_wide_supported(int H, int E) { return H >= 4 && H % 4 == 0 && E >= 1 && E <= MTS_MAX_EXPERTS ? 1 : 0; }

extern "C" int mts_router_wide_fwd(const void* x, const float* w_r, int64_t T, int H, int E, int act_dtype, float* logits, void* stream) {
    const int rc = wide_check(x, w_r, T, H, E, act_dtype);
    if (rc) return rc;
    if (!logits) return MTS_ERR_NULL;
    const dim3 grid((unsigned)((T + 31) / 32), (unsigned)((E + 63) / 64));
    hipStream_t s = (hipStream_t)stream;
    if (act_dtype == MTS_BF16) wide_logits_kernel<bf16_t><<<grid, kThreads, 0, s>>>((const bf16_t*)x, w_r, T, H, E, logits);
    else if (act_dtype == MTS_F16) wide_logits_kernel<mts_f16_t><<<grid, kThreads, 0, s>>>((const mts_f16_t*)x, w_r, T, H, E, logits);
    else wide_logits_kernel<float><<<grid, kThreads, 0, s>>>((const float*)x, w_r, T, H, E, logits);
    MTS_CHECK_LAUNCH();
    return MTS_OK;
}

extern "C" int64_t mts_router_wide_bwd_workspace_bytes(int64_t T, int H, int E) {
    if (T <= 0 || H <= 0 || E <= 0) return 0;
    return (int64_t)wide_chunks(T, H, E).count * E * H * (int64_t)sizeof(float);
}

extern "C" int mts_router_wide_bwd(const float* dlogits, const void* x, const float* w_r, int64_t T, int H, int E, int act_dtype, void* dx,
                                   float* d_w_r, void* workspace, int64_t workspace_bytes, void* stream) {
    const int rc = wide_check(x, w_r, T, H, E, act_dtype);
    if (rc) return rc;
    if (!dlogits || !dx || !d_w_r || !workspace) return MTS_ERR_NULL;
    if (workspace_bytes < mts_router_wide_bwd_workspace_bytes(T, H, E)) return MTS_ERR_WORKSPACE;
    if (!mts_aligned16(dlogits) || !mts_aligned16(dx) || !mts_aligned16(d_w_r) || !mts_aligned16(workspace)) return MTS_ERR_ALIGN;
    hipStream_t s = (hipStream_t)stream;
    const bool vec = E % 4 == 0;
    const dim3 grid_dx((unsigned)((T + 63) / 64 * ((H + 63) / 64)));
    const WideChunks c = wide_chunks(T, H, E);
    const dim3 grid_dw((unsigned)((H + 63) / 64), (unsigned)((E + 63) / 64), (unsigned)c.count);
    float* part = (float*)workspace;
    auto launch = [&](auto* kind) {
        typedef typename std::remove_pointer<decltype(kind)>::type XT;
        if (vec) {
            wide_dx_kernel<XT, true><<<grid_dx, kThreads, 0, s>>>(dlogits, w_r, T, H, E, (XT*)dx);
            wide_dw_kernel<XT, true><<<grid_dw, kThreads, 0, s>>>(dlogits, (const XT*)x, T, H, E, c.rows, part);
        } else {
            wide_dx_kernel<XT, false><<<grid_dx, kThreads, 0, s>>>(dlogits, w_r, T, H, E, (XT*)dx);
            wide_dw_kernel<XT, false><<<grid_dw, kThreads, 0, s>>>(dlogits, (const XT*)x, T, H, E, c.rows, part);
        }
    };
    if (act_dtype == MTS_BF16) launch((bf16_t*)nullptr);
    else if (act_dtype == MTS_F16) launch((mts_f16_t*)nullptr);
    else launch((float*)nullptr);
    MTS_CHECK_LAUNCH();
    return mts_launch_router_dw_reduce(part, c.count, (int64_t)E * H, d_w_r, s);
}
