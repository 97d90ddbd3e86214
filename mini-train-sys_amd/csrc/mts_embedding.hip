// The gradient of an embedding table: row r of dw is the fp32 sum of the rows of g whose id is r, and zero where there is none.  Up to
// kLongRow tokens are added in token order.  Of more, each wave adds a share of those in front of the whole segments (below), one of those behind them
// and one of the segments' sums, and the waves' sums are added in turn: a fixed order for the same ids, which goes by where the row lies in the order.
//
// Bound by HBM at the table's size (50 257 x 768: 154 MB written, 38 MB of bf16 gradients read for 24 576 tokens), as long as the
// tokens are sorted by id cheaply: a block owns a range of ids and looks through all of them (200 KB out of an L2, two passes), so that
// nothing waits between blocks; its own tokens are then few.  The sum takes a wave a row, and all waves of a block for a row of more than
// kLongRow tokens, of which whole segments of the order have been added up by a block each before.  24 576 tokens of 50 257 words: 48 us in three launches where the
// stock operators (fp32 copy of the gradient, sort in six launches, sums in two, a pass that clears the table) took 225, the training step around
// it 15.09 ms where it now takes 14.87; with half or all of the tokens the same word 79 and 84 us (492 and 801 stock; 683 and 1348 by one wave that orders
// and one block that adds, which took 41 us of evenly spread words).
#include "mts_common.h"

#include <type_traits>

namespace {

constexpr int kOrderThreads = 1024, kOrderWaves = kOrderThreads / MTS_WAVE;
constexpr int kOrderBlocks = 256;      // one a CU
constexpr int kMostRange = 768;        // ids of a block, which have a counter for every wave in LDS
constexpr int kMostIds = 1 << 20;
constexpr int kMostTokens = 1 << 18;   // every block reads all of them
constexpr int kInFlight = 8;

typedef volatile __attribute__((address_space(3))) int32_t* LdsCounters;

// row_start[r]: tokens with an id below r; order: the tokens by id, those of one id in ascending order.  A wave takes a contiguous share of the
// tokens and counts its own, so that it knows their places when it comes by a second time.
// An id outside [0, V) belongs to no block's range; it takes a place in front of or behind the rows' and is not looked at.
__global__ __launch_bounds__(kOrderThreads) void embedding_order_kernel(const int64_t* __restrict__ ids, int T, int V, int per, int32_t* __restrict__ row_start,
                                                                        int32_t* __restrict__ order) {
    extern __shared__ int32_t counters[];   // [kOrderWaves][per], and [per] more
    __shared__ int32_t below_of[kOrderWaves], hits_of[kOrderWaves];
    const int wave = threadIdx.x / MTS_WAVE, lane = threadIdx.x % MTS_WAVE;
    const int lo = blockIdx.x * per, hi = min(lo + per, V);
    int32_t* mine = counters + wave * per;
    for (int i = lane; i < per; i += MTS_WAVE) mine[i] = 0;
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
            if (in) atomicAdd(&mine[(int)id[u] - lo], 1);
        }
    }
    if (lane == 0) below_of[wave] = below, hits_of[wave] = hits;
    __syncthreads();
    // The counters become those of the waves in front, and first[] the place of each id's first token.
    int32_t* first = counters + kOrderWaves * per;
    for (int i = threadIdx.x; i < per; i += kOrderThreads) {
        int32_t n[kOrderWaves], before = 0;
#pragma unroll
        for (int w = 0; w < kOrderWaves; ++w) n[w] = counters[w * per + i];
#pragma unroll
        for (int w = 0; w < kOrderWaves; ++w) {
            counters[w * per + i] = before;
            before += n[w];
        }
        first[i] = before;
    }
    __syncthreads();
    if (wave == 0) {
        int32_t carry = wave_sum(lane < kOrderWaves ? below_of[lane] : 0);
        for (int i0 = 0; i0 < hi - lo; i0 += MTS_WAVE) {
            const int i = i0 + lane;
            const int32_t n = i < hi - lo ? first[i] : 0, incl = wave_scan(n);
            if (i < hi - lo) first[i] = row_start[lo + i] = carry + incl - n;
            carry += __builtin_amdgcn_readlane(incl, MTS_WAVE - 1);
        }
        if (hi == V && lane == 0) row_start[V] = carry;
    }
    __syncthreads();
    if (hits == 0) return;
    // 64 tokens at a time: lanes with the same id find each other with a ballot a bit of it
    LdsCounters next = (LdsCounters)mine;
    int bits = 0;
    while ((1 << bits) < hi - lo) ++bits;
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
            const int at = in ? (int)id[u] - lo : 0;
            uint64_t same = __ballot(in);
            if (same == 0) continue;
            for (int bit = 0; bit < (same & (same - 1) ? bits : 0); ++bit) {   // one alone needs no search
                const uint64_t set = __ballot((at >> bit) & 1);
                same &= ((at >> bit) & 1) ? set : ~set;
            }
            if (in) {
                const int nth = next[at], rank = __popcll(same & lanemask_lt());   // every lane reads before the first of its group updates
                if (rank == 0) next[at] = nth + __popcll(same);
                order[first[at] + nth + rank] = t;
            }
        }
    }
}

constexpr int kSumWaves = 8, kSumThreads = kSumWaves * MTS_WAVE;
constexpr int kLongRow = 32;    // tokens
constexpr int kSegment = 128;   // tokens

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

// acc of all waves of a block, added in wave order, ends up in the last wave's
template <int NV>
__device__ __forceinline__ void add_waves(f32x4 (&acc)[NV], f32x4* sums, int quads) {
    const int wave = threadIdx.x / MTS_WAVE, lane = threadIdx.x % MTS_WAVE;
    for (int k = 0; k < kSumWaves; ++k) {
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
        }
        __syncthreads();
    }
}
template <int NV>
__device__ __forceinline__ void store_sums(float* __restrict__ row, const f32x4 (&acc)[NV], int quads) {
    f32x4* out = reinterpret_cast<f32x4*>(row);
    const int lane = threadIdx.x % MTS_WAVE;
#pragma unroll
    for (int i = 0; i < NV; ++i)
        if (i * MTS_WAVE + lane < quads) out[i * MTS_WAVE + lane] = acc[i];
}

// Rows of very many tokens (an id that fills short sequences up, say) would be the work of one block: where all of the order's places [s * kSegment, (s + 1) *
// kSegment) are of one row, this block adds them up before (part[s]).  In other batches its blocks leave at once.
template <typename ET, int NV>
__global__ __launch_bounds__(kSumThreads) void embedding_segment_kernel(const ET* __restrict__ g, const int64_t* __restrict__ ids, const int32_t* __restrict__ row_start,
                                                                        const int32_t* __restrict__ order, int V, int H, float* __restrict__ part) {
    extern __shared__ f32x4 sums[];   // [H / 4]
    const int first = blockIdx.x * kSegment, last = first + kSegment;
    const int from_row = row_start[0], to_row = row_start[V], t = order[first];
    if (first < from_row || last > to_row) return;   // places that belong to no row hold nothing
    if (last > row_start[ids[t] + 1]) return;
    constexpr int SHARE = kSegment / kSumWaves;
    const int from = first + threadIdx.x / MTS_WAVE * SHARE;
    f32x4 acc[NV] = {};
    add_rows<ET, NV>(acc, g, order, from, from + SHARE, H);
    add_waves(acc, sums, H / 4);
    if (threadIdx.x / MTS_WAVE == kSumWaves - 1) store_sums(part + (int64_t)blockIdx.x * H, acc, H / 4);
}

template <typename ET, int NV>
__global__ __launch_bounds__(kSumThreads) void embedding_sum_kernel(const ET* __restrict__ g, const int32_t* __restrict__ row_start,
                                                                    const int32_t* __restrict__ order, int V, int H, const float* __restrict__ part,
                                                                    float* __restrict__ dw) {
    extern __shared__ f32x4 sums[];   // [H / 4]
    const int wave = threadIdx.x / MTS_WAVE, lane = threadIdx.x % MTS_WAVE, quads = H / 4;
    const int row0 = blockIdx.x * kSumWaves;
    int start[kSumWaves + 1];
#pragma unroll
    for (int w = 0; w <= kSumWaves; ++w) start[w] = row_start[min(row0 + w, V)];
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
        store_sums(dw + (int64_t)(row0 + wave) * H, acc, quads);
    }
    if (!any_long) return;   // block-uniform
    for (int w = 0; w < kSumWaves; ++w) {
        const int beg = row_start[min(row0 + w, V)], end = row_start[min(row0 + w + 1, V)];
        if (end - beg <= kLongRow) continue;
        // the tokens in front of the whole segments and behind them, a share each
        const int s0 = (beg + kSegment - 1) / kSegment, s1 = max(end / kSegment, s0);
        const bool cut = s1 > s0;
        const int front = cut ? s0 * kSegment : end, back = cut ? s1 * kSegment : end;
        f32x4 acc[NV] = {};
        auto share = [&](int beg, int end) {
            const int per = (end - beg + kSumWaves - 1) / kSumWaves, first = min(beg + wave * per, end);
            add_rows<ET, NV>(acc, g, order, first, min(first + per, end), H);
        };
        share(beg, front);
        share(back, end);
        if (cut) {
            const int per = (s1 - s0 + kSumWaves - 1) / kSumWaves, first = min(s0 + wave * per, s1), last = min(first + per, s1);
#pragma unroll 4
            for (int k = first; k < last; ++k) {
                const f32x4* row = reinterpret_cast<const f32x4*>(part + (int64_t)k * H);
#pragma unroll
                for (int i = 0; i < NV; ++i) acc[i] += row[min(i * MTS_WAVE + lane, quads - 1)];
            }
        }
        add_waves(acc, sums, quads);
        if (wave == kSumWaves - 1) store_sums(dw + (int64_t)(row0 + w) * H, acc, quads);
    }
}

int ids_per_block(int V) {
    const int per = (V + kOrderBlocks - 1) / kOrderBlocks;
    return per < kMostRange ? per : kMostRange;
}
int64_t segments(int64_t T) { return T / kSegment; }

template <typename ET>
void launch_sum(const void* g, const int64_t* ids, int64_t T, const int32_t* row_start, const int32_t* order, int V, int H, float* part, float* dw, hipStream_t s) {
    const dim3 grid((unsigned)((V + kSumWaves - 1) / kSumWaves)), block(kSumThreads);
    const size_t lds = (size_t)H * sizeof(float);
    const int groups = (H / 4 + MTS_WAVE - 1) / MTS_WAVE;
    auto launch = [&](auto nv) {
        if (segments(T)) embedding_segment_kernel<ET, decltype(nv)::value><<<dim3((unsigned)segments(T)), block, lds, s>>>((const ET*)g, ids, row_start, order, V, H, part);
        embedding_sum_kernel<ET, decltype(nv)::value><<<grid, block, lds, s>>>((const ET*)g, row_start, order, V, H, part, dw);
    };
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

// Against the stock operators (conversion, sort, sums): ahead from 64 tokens on with tables of up to 65 536 rows (64 tokens 38 us, stock 45; 512 39 / 58).  More rows
// are more blocks that each read all tokens, and a launch over all rows, while the stock sums walk the tokens; us here / stock, 768 wide: 128 256 rows, 64 tokens
// 77 / 70; 262 144 rows, 64 tokens 172 / 130, 512 175 / 169, 4096 183 / 209; 300 001, 1024 tokens 204 / 230 (4 wide 63 / 62), 3000 209 / 401; 393 216, 4096 tokens
// 272 / 267, 65 536 411 / 757; 524 288, 65 536 tokens of 512 361 / 549, of 128 187 / 187; 2^20, 4096 tokens 728 / 560, 65 536 950 / 1062, 262 144 of 256 825 / 971,
// of 128 677 / 563.
extern "C" int mts_embedding_bwd_preferred(int64_t T, int64_t V, int64_t H) {
    if (!mts_embedding_bwd_supported(T, V, H)) return 0;
    if (V <= 65536) return 1;
    return V <= 327680 ? T >= V / 256 : T * H >= 64 * V;
}

extern "C" int64_t mts_embedding_bwd_workspace_bytes(int64_t T, int64_t V, int64_t H) {
    return (segments(T) * H + V + 1 + T) * (int64_t)sizeof(int32_t);   // sums of the segments first, on 16 bytes
}

extern "C" int mts_embedding_bwd(const void* g, const int64_t* ids, int64_t T, int V, int H, int act_dtype, float* dw, void* workspace,
                                 int64_t workspace_bytes, void* stream) {
    if (!g || !ids || !dw || !workspace) return MTS_ERR_NULL;
    if (!mts_embedding_bwd_supported(T, V, H)) return MTS_ERR_SHAPE;
    if (act_dtype != MTS_BF16 && act_dtype != MTS_F16 && act_dtype != MTS_F32) return MTS_ERR_DTYPE;
    if (workspace_bytes < mts_embedding_bwd_workspace_bytes(T, V, H)) return MTS_ERR_WORKSPACE;
    if (!mts_aligned16(g) || !mts_aligned16(dw) || !mts_aligned16(workspace)) return MTS_ERR_ALIGN;
    hipStream_t s = (hipStream_t)stream;
    float* part = (float*)workspace;
    int32_t *row_start = (int32_t*)(part + segments(T) * H), *order = row_start + V + 1;
    const int per = ids_per_block(V);
    embedding_order_kernel<<<dim3((unsigned)((V + per - 1) / per)), kOrderThreads, (size_t)per * (kOrderWaves + 1) * sizeof(int32_t), s>>>(ids, (int)T, V, per, row_start, order);
    MTS_CHECK_LAUNCH();
    if (act_dtype == MTS_BF16) launch_sum<bf16_t>(g, ids, T, row_start, order, V, H, part, dw, s);
    else if (act_dtype == MTS_F16) launch_sum<mts_f16_t>(g, ids, T, row_start, order, V, H, part, dw, s);
    else launch_sum<float>(g, ids, T, row_start, order, V, H, part, dw, s);
    MTS_CHECK_LAUNCH();
    return MTS_OK;
}
