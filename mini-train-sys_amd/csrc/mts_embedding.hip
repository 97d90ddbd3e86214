// The gradient of an embedding table: row r of dw is the fp32 sum, in token order, of the rows of g whose id is r, and zero where
// there is none.
//
// Bound by HBM at the table's size (50 257 x 768: 154 MB written, 38 MB of bf16 gradients read for 24 576 tokens), as long as the
// tokens are sorted by id cheaply: a block owns a range of ids and looks through all of them (200 KB out of an L2, two passes), so that
// nothing waits between blocks; its own tokens are then few.  The sum takes a wave a row, and all waves of a block for a row of more than
// kLongRow tokens.  24 576 tokens of 50 257 words: order 15 us, sum 26 us (7.3 TB/s); the stock operators (fp32 copy of the gradient,
// sort in six launches, sums in two, a pass that clears the table) took about 230 us, the training step around it 15.09 ms where it now takes 14.87.
#include "mts_common.h"

#include <type_traits>

namespace {

constexpr int kOrderThreads = 1024, kOrderWaves = kOrderThreads / MTS_WAVE;
constexpr int kOrderBlocks = 256;      // one a CU
constexpr int kMostIds = 1 << 20;      // a block's range of them has its counters in LDS
constexpr int kMostTokens = 1 << 18;   // every block reads all of them
constexpr int kInFlight = 8;

typedef volatile __attribute__((address_space(3))) int32_t* LdsCounters;

// row_start[r]: tokens with an id below r; order: the tokens by id, those of one id in ascending order.  found: scratch, as long as order.
// An id outside [0, V) belongs to no block's range; it takes a place in front of or behind the rows' and is not looked at.
__global__ __launch_bounds__(kOrderThreads) void embedding_order_kernel(const int64_t* __restrict__ ids, int T, int V, int per, int32_t* __restrict__ row_start,
                                                                        int32_t* __restrict__ found, int32_t* __restrict__ order) {
    extern __shared__ int32_t counters[];   // [per]
    __shared__ int32_t below_of[kOrderWaves], hits_of[kOrderWaves];
    const int wave = threadIdx.x / MTS_WAVE, lane = threadIdx.x % MTS_WAVE;
    const int lo = blockIdx.x * per, hi = min(lo + per, V);
    for (int i = threadIdx.x; i < per; i += kOrderThreads) counters[i] = 0;
    __syncthreads();
    const int share = ((T + kOrderWaves - 1) / kOrderWaves + MTS_WAVE - 1) / MTS_WAVE * MTS_WAVE;
    const int t0 = min(wave * share, T), t1 = min(t0 + share, T);
    int below = 0, hits = 0;
    for (int base = t0; base < t1; base += kInFlight * MTS_WAVE) {
        int64_t id[kInFlight];
#pragma unroll
        for (int u = 0; u < kInFlight; ++u) {
            const int t = base + u * MTS_WAVE + lane;
            id[u] = ids[t < t1 ? t : t1 - 1];
        }
#pragma unroll
        for (int u = 0; u < kInFlight; ++u) {
            const bool there = base + u * MTS_WAVE + lane < t1, in = there && id[u] >= lo && id[u] < hi;
            below += __popcll(__ballot(there && id[u] < lo));
            hits += __popcll(__ballot(in));
            if (in) atomicAdd(&counters[(int)id[u] - lo], 1);
        }
    }
    if (lane == 0) below_of[wave] = below, hits_of[wave] = hits;
    __syncthreads();
    int first = 0, total = 0, at = 0;   // where this block's tokens begin in the order, how many there are, where this wave's begin
    for (int w = 0; w < kOrderWaves; ++w) {
        first += below_of[w];
        if (w == wave) at = total;
        total += hits_of[w];
    }
    at += first;
    if (hits)
        for (int base = t0; base < t1; base += kInFlight * MTS_WAVE) {
            int64_t id[kInFlight];
#pragma unroll
            for (int u = 0; u < kInFlight; ++u) {
                const int t = base + u * MTS_WAVE + lane;
                id[u] = ids[t < t1 ? t : t1 - 1];
            }
#pragma unroll
            for (int u = 0; u < kInFlight; ++u) {
                const int t = base + u * MTS_WAVE + lane;
                const bool in = t < t1 && id[u] >= lo && id[u] < hi;
                const uint64_t mask = __ballot(in);
                if (in) found[at + __popcll(mask & lanemask_lt())] = t;
                at += __popcll(mask);
            }
        }
    if (wave == 0) {   // the counters become the places of each id's next token
        int32_t carry = first;
        for (int i0 = 0; i0 < hi - lo; i0 += MTS_WAVE) {
            const int i = i0 + lane;
            const int32_t n = i < hi - lo ? counters[i] : 0, incl = wave_scan(n);
            if (i < hi - lo) {
                counters[i] = carry + incl - n;
                row_start[lo + i] = carry + incl - n;
            }
            carry += __builtin_amdgcn_readlane(incl, MTS_WAVE - 1);
        }
        if (hi == V && lane == 0) row_start[V] = carry;
    }
    __syncthreads();
    if (wave != 0) return;
    // 64 tokens at a time: lanes with the same id find each other with a ballot a bit of it
    LdsCounters next = (LdsCounters)counters;
    int bits = 0;
    while ((1 << bits) < hi - lo) ++bits;
    for (int k = 0; k < total; k += MTS_WAVE) {
        const bool valid = k + lane < total;
        const int t = valid ? found[first + k + lane] : 0;
        const int id = valid ? (int)ids[t] - lo : 0;
        uint64_t same = __ballot(valid);
        for (int bit = 0; bit < bits; ++bit) {
            const uint64_t set = __ballot((id >> bit) & 1);
            same &= ((id >> bit) & 1) ? set : ~set;
        }
        if (valid) {
            const int place = next[id], rank = __popcll(same & lanemask_lt());   // every lane reads before the first of its group updates
            if (rank == 0) next[id] = place + __popcll(same);
            order[place + rank] = t;
        }
    }
}

constexpr int kSumWaves = 8, kSumThreads = kSumWaves * MTS_WAVE;
constexpr int kLongRow = 32;   // tokens

template <typename ET>
struct Quad;
template <>
struct Quad<bf16_t> { typedef bf16x4 type; };
template <>
struct Quad<mts_f16_t> { typedef mts_f16x4 type; };
template <>
struct Quad<float> { typedef f32x4 type; };

// acc += the rows of g that order[from .. to - 1] names; lane: 4 columns of every 256
template <typename ET, int NV>
__device__ __forceinline__ void add_rows(f32x4 (&acc)[NV], const ET* __restrict__ g, const int32_t* __restrict__ order, int from, int to, int H) {
    typedef typename Quad<ET>::type quad;
    constexpr int ROWS = NV <= 4 ? 4 : 2;   // in flight
    const int lane = threadIdx.x % MTS_WAVE, quads = H / 4;
    for (int k = from; k < to; k += ROWS) {
        quad v[ROWS][NV];
#pragma unroll
        for (int r = 0; r < ROWS; ++r) {
            const int t = __builtin_amdgcn_readfirstlane(order[k + r < to ? k + r : to - 1]);
            const quad* row = reinterpret_cast<const quad*>(g + (int64_t)t * H);
#pragma unroll
            for (int i = 0; i < NV; ++i) {
                const int c = i * MTS_WAVE + lane;
                v[r][i] = row[c < quads ? c : quads - 1];
            }
        }
#pragma unroll
        for (int r = 0; r < ROWS; ++r)
            if (k + r < to)
#pragma unroll
                for (int i = 0; i < NV; ++i)
#pragma unroll
                    for (int j = 0; j < 4; ++j) acc[i][j] += (float)v[r][i][j];
    }
}

template <typename ET, int NV>
__global__ __launch_bounds__(kSumThreads) void embedding_sum_kernel(const ET* __restrict__ g, const int32_t* __restrict__ row_start,
                                                                    const int32_t* __restrict__ order, int V, int H, float* __restrict__ dw) {
    extern __shared__ f32x4 sums[];   // [H / 4]
    const int wave = threadIdx.x / MTS_WAVE, lane = threadIdx.x % MTS_WAVE, quads = H / 4;
    const int row0 = blockIdx.x * kSumWaves;
    int start[kSumWaves + 1];
#pragma unroll
    for (int w = 0; w <= kSumWaves; ++w) start[w] = row_start[min(row0 + w, V)];
    auto store = [&](int row, const f32x4(&acc)[NV]) {
        f32x4* out = reinterpret_cast<f32x4*>(dw + (int64_t)row * H);
#pragma unroll
        for (int i = 0; i < NV; ++i)
            if (i * MTS_WAVE + lane < quads) out[i * MTS_WAVE + lane] = acc[i];
    };
    int from = start[0], to = start[1];
    bool any_long = false;
#pragma unroll
    for (int w = 0; w < kSumWaves; ++w) {
        if (w == wave) from = start[w], to = start[w + 1];
        any_long |= start[w + 1] - start[w] > kLongRow;
    }
    if (row0 + wave < V && to - from <= kLongRow) {
        f32x4 acc[NV] = {};
        add_rows<ET, NV>(acc, g, order, from, to, H);
        store(row0 + wave, acc);
    }
    if (!any_long) return;   // block-uniform
    for (int w = 0; w < kSumWaves; ++w) {
        const int beg = row_start[min(row0 + w, V)], end = row_start[min(row0 + w + 1, V)];
        if (end - beg <= kLongRow) continue;
        const int per = (end - beg + kSumWaves - 1) / kSumWaves;
        f32x4 acc[NV] = {};
        const int first = min(beg + wave * per, end), last = min(first + per, end);
        add_rows<ET, NV>(acc, g, order, first, last, H);
        for (int k = 0; k < kSumWaves; ++k) {   // in wave order
            if (wave == k) {
#pragma unroll
                for (int i = 0; i < NV; ++i) {
                    const int c = i * MTS_WAVE + lane;
                    if (c >= quads) continue;
                    if (k) {
                        const f32x4 before = sums[c];
#pragma unroll
                        for (int j = 0; j < 4; ++j) acc[i][j] = before[j] + acc[i][j];
                    }
                    sums[c] = acc[i];
                }
                if (k == kSumWaves - 1) store(row0 + w, acc);
            }
            __syncthreads();
        }
    }
}

int ids_per_block(int V) { return (V + kOrderBlocks - 1) / kOrderBlocks; }

template <typename ET>
void launch_sum(const void* g, const int32_t* row_start, const int32_t* order, int V, int H, float* dw, hipStream_t s) {
    const dim3 grid((unsigned)((V + kSumWaves - 1) / kSumWaves)), block(kSumThreads);
    const size_t lds = (size_t)H * sizeof(float);
    const int groups = (H / 4 + MTS_WAVE - 1) / MTS_WAVE;
    auto launch = [&](auto nv) { embedding_sum_kernel<ET, decltype(nv)::value><<<grid, block, lds, s>>>((const ET*)g, row_start, order, V, H, dw); };
    if (groups <= 1) launch(std::integral_constant<int, 1>());
    else if (groups <= 2) launch(std::integral_constant<int, 2>());
    else if (groups <= 3) launch(std::integral_constant<int, 3>());
    else if (groups <= 4) launch(std::integral_constant<int, 4>());
    else if (groups <= 8) launch(std::integral_constant<int, 8>());
    else launch(std::integral_constant<int, 16>());
}

}  // namespace

extern "C" int mts_embedding_bwd_supported(int64_t T, int64_t V, int64_t H) {
    return T > 0 && T <= kMostTokens && V > 0 && V <= kMostIds && H > 0 && H % 4 == 0 && H <= 16 * 4 * MTS_WAVE ? 1 : 0;
}

extern "C" int64_t mts_embedding_bwd_workspace_bytes(int64_t T, int64_t V) { return (V + 1 + 2 * T) * (int64_t)sizeof(int32_t); }

extern "C" int mts_embedding_bwd(const void* g, const int64_t* ids, int64_t T, int V, int H, int act_dtype, float* dw, void* workspace,
                                 int64_t workspace_bytes, void* stream) {
    if (!g || !ids || !dw || !workspace) return MTS_ERR_NULL;
    if (!mts_embedding_bwd_supported(T, V, H)) return MTS_ERR_SHAPE;
    if (act_dtype != MTS_BF16 && act_dtype != MTS_F16 && act_dtype != MTS_F32) return MTS_ERR_DTYPE;
    if (workspace_bytes < mts_embedding_bwd_workspace_bytes(T, V)) return MTS_ERR_WORKSPACE;
    if (!mts_aligned16(g) || !mts_aligned16(dw) || !mts_aligned16(workspace)) return MTS_ERR_ALIGN;
    hipStream_t s = (hipStream_t)stream;
    int32_t *row_start = (int32_t*)workspace, *found = row_start + V + 1, *order = found + T;
    const int per = ids_per_block(V);
    embedding_order_kernel<<<dim3((unsigned)((V + per - 1) / per)), kOrderThreads, (size_t)per * sizeof(int32_t), s>>>(ids, (int)T, V, per, row_start, found, order);
    MTS_CHECK_LAUNCH();
    if (act_dtype == MTS_BF16) launch_sum<bf16_t>(g, row_start, order, V, H, dw, s);
    else if (act_dtype == MTS_F16) launch_sum<mts_f16_t>(g, row_start, order, V, H, dw, s);
    else launch_sum<float>(g, row_start, order, V, H, dw, s);
    MTS_CHECK_LAUNCH();
    return MTS_OK;
}
