// Attention of the decoder for heads of 64 elements, forward and backward, causal or not, without materialised scores.
//
// Every product runs on v_mfma_f32_32x32x16 and is laid out so that no score changes lanes.  An accumulator of that
// instruction holds, for column n = lane % 32, the rows 8 * (i / 4) + 4 * (lane / 32) + i % 4; its 16 x n operand wants
// 8 values of k per lane.  Which k those are is free as long as the other operand agrees, so eight consecutive
// accumulator registers serve as an operand as they are, and the other one is read from LDS with rows
// krow0 + 4 * (lane / 32) + {0..3, 8..11} by the transposing load.  The scores are therefore formed transposed (keys x
// queries) where they are summed over the keys (output, dQ), and as queries x keys where they are summed over the queries
// (dK, dV): the operand that a wave owns stays in registers, the other one streams through LDS in tiles of 64 rows.
//
// The vector pipe bounds it: for 32 x 64 scores the forward pass issues 512 cycles of MFMA and about 1000 of exponentials (a
// quarter of the rate), maxima, sums and conversions.  bf16, causal, 12 heads of 64, 1024 rows, against the stock operator:
// batch 8: 31 us forward (79) and 121 backward (308); batch 24: 72 us (534 TFLOP/s; 168) and 304 (445 TFLOP/s of the seven
// products that two separate kernels form, so that each gradient is summed by one block in a fixed order; 844).
//
// Between rotary encodings (the decoder's case) the queries are turned as they are read and the gradients turned back as they are written, straight into the
// gradient of the packed projection: a launch that turned queries and one that turned gradients and copied those of the values go (24 x 12 heads x
// 1024: 38 + 38 us), the keys keep theirs (20).  In turn the forward kernel takes 92 us where it took 78 (it leaves the turned queries for the
// backward pass; 32 for 31 without, batch 8), dQ 102 for 100, dK/dV 127 for 130.  Results leave through LDS, a line by eight lanes: with 8-byte
// pieces of 32 rows an instruction forward, dQ and dK/dV took 95, 116 and 144 us.  Training step of four layers 14.41 -> 14.27 ms, validation
// pass of 8 x 1024 tokens through twelve 3.92 -> 3.90; passes of 800 tokens, which wait for the host, 512 -> 470 us, training steps 1.81 -> 1.69 ms.
//
// Error against fp64 (2-norm, bf16, 24 heads x 1024): output 2.0e-3, dQ 2.5e-3, dK 2.4e-3, dV 2.3e-3, the stock operator's to
// three digits; likewise at 200 and 777 rows, for scores three times as far apart, and in fp16.
#include "mts_common.h"

namespace {

typedef __attribute__((ext_vector_type(4))) short s16x4;
typedef __attribute__((ext_vector_type(8))) short s16x8;

template <typename ET>
struct Mma;
template <>
struct Mma<bf16_t> {
    typedef bf16x8 frag;
    typedef bf16x4 quad;
    static __device__ __forceinline__ f32x16 mul(frag a, frag b, f32x16 c) { return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0); }
};
template <>
struct Mma<mts_f16_t> {
    typedef mts_f16x8 frag;
    typedef mts_f16x4 quad;
    static __device__ __forceinline__ f32x16 mul(frag a, frag b, f32x16 c) { return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0); }
};

constexpr int kHead = 64;               // elements of a head
constexpr int kTile = 64;               // rows of a streamed tile
constexpr int kWaves = 4;
constexpr int kThreads = kWaves * MTS_WAVE;
constexpr int kOwn = 32 * kWaves;       // rows a block owns, 32 a wave
constexpr int kTileElems = kTile * kHead;
constexpr int kCusPerXcd = 32;
constexpr float kLog2e = 1.4426950408889634f;

// [B, heads, S, 64], dense in the last dimension, strides in elements
template <typename T>
struct Heads {
    T* p;
    int64_t b, h, s;
    __device__ __forceinline__ T* row0(int64_t bh, int heads) const { return p + (bh / heads) * b + (bh % heads) * h; }
};

// 16-byte chunk of a row, exchanged so that 16 consecutive rows of one chunk (row fragments) and 4 rows of four chunks
// (transposed fragments) both fall on all 64 banks
__device__ __forceinline__ int chunk_off(int row, int chunk) { return row * kHead + ((chunk ^ (((row >> 1) & 1) << 2 | ((row >> 2) & 3))) << 3); }

// rows row0 + lane % 32, elements 16 * ks + 8 * (lane / 32) + 0..7
template <typename ET>
__device__ __forceinline__ typename Mma<ET>::frag row_frag(const ET* tile, int row0, int ks) {
    const int lane = threadIdx.x % MTS_WAVE;
    return *reinterpret_cast<const typename Mma<ET>::frag*>(tile + chunk_off(row0 + lane % 32, 2 * ks + lane / 32));
}

// columns col0 + lane % 32, rows krow0 + 4 * (lane / 32) + {0..3, 8..11}
template <typename ET>
__device__ __forceinline__ typename Mma<ET>::frag column_frag(const ET* tile, int krow0, int col0) {
    const int lane = threadIdx.x % MTS_WAVE;
    const int col = col0 + 16 * ((lane / 16) % 2) + 4 * (lane % 4);
    s16x4 h[2];
#pragma unroll
    for (int q = 0; q < 2; ++q) {
        const ET* src = tile + chunk_off(krow0 + 8 * q + 4 * (lane / 32) + (lane % 16) / 4, col / 8) + col % 8;
        h[q] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)(src));
    }
    const s16x8 v = {h[0][0], h[0][1], h[0][2], h[0][3], h[1][0], h[1][1], h[1][2], h[1][3]};
    return __builtin_bit_cast(typename Mma<ET>::frag, v);
}

// A tile on its way from memory to LDS through registers, so that its latency is covered by the tile before it; rows behind
// the end arrive as zeros.
template <typename ET>
struct TileCopy {
    u32x4 reg[kTileElems / 8 / kThreads];
    __device__ __forceinline__ void fetch(const ET* head, int64_t stride, int row0, int S) {
#pragma unroll
        for (int i = 0; i < (int)(sizeof(reg) / 16); ++i) {
            const int row = row0 + (threadIdx.x + i * kThreads) / 8, c = threadIdx.x % 8;
            reg[i] = row < S ? *reinterpret_cast<const u32x4*>(head + row * stride + c * 8) : u32x4{};
        }
    }
    __device__ __forceinline__ void commit(ET* tile) const {
#pragma unroll
        for (int i = 0; i < (int)(sizeof(reg) / 16); ++i)
            *reinterpret_cast<u32x4*>(tile + chunk_off((threadIdx.x + i * kThreads) / 8, threadIdx.x % 8)) = reg[i];
    }
};

// the 32 rows a wave owns, as an operand that stays in registers (row row, elements 16 * ks + 8 * (lane / 32) + 0..7)
template <typename ET>
__device__ __forceinline__ void own_frags(const ET* row, typename Mma<ET>::frag (&f)[4]) {
    const int lane = threadIdx.x % MTS_WAVE;
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) f[ks] = *reinterpret_cast<const typename Mma<ET>::frag*>(row + 16 * ks + 8 * (lane / 32));
}

template <typename ET>
__device__ __forceinline__ typename Mma<ET>::frag narrowed(const f32x16& v, int t) {
    typename Mma<ET>::frag f;
#pragma unroll
    for (int j = 0; j < 8; ++j) f[j] = (ET)v[8 * t + j];
    return f;
}

// Four elements of a row in two registers.  A lane of a transposed accumulator holds elements 8 * i + 4 * (lane / 32) + 0..3 of the row of its column, the
// lane 32 from it the other four of every eight; memory is asked in pieces of 16 bytes, of which a lane takes 16 * k + 8 * (lane / 32) + 0..7: twice
// the bytes an instruction.
typedef uint2 Quad;
__device__ __forceinline__ void load_quads(const void* row, Quad (&q)[8]) {
    const int lane = threadIdx.x % MTS_WAVE;
    u32x4 v[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) v[k] = *reinterpret_cast<const u32x4*>(static_cast<const char*>(row) + 32 * k + 16 * (lane / 32));
#pragma unroll
    for (int k = 0; k < 4; ++k) {   // each half hands the other the quad that it has a place for
        const auto x = __builtin_amdgcn_permlane32_swap(v[k][0], v[k][2], false, false), y = __builtin_amdgcn_permlane32_swap(v[k][1], v[k][3], false, false);
        q[2 * k] = {x[0], y[0]}, q[2 * k + 1] = {x[1], y[1]};
    }
}

// The 32 x 64 results of a wave go out through a tile of its own in LDS, where nothing is read any more: eight lanes then write a row, a whole line.
template <typename ET>
__device__ __forceinline__ void flush_rows(const ET* tile, ET* head, int64_t stride, int first, int S) {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    const int lane = threadIdx.x % MTS_WAVE;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int r = 8 * i + lane / 8;
        if (first + r < S) *reinterpret_cast<u32x4*>(head + (first + r) * stride + lane % 8 * 8) = *reinterpret_cast<const u32x4*>(tile + chunk_off(r, lane % 8));
    }
}
template <typename ET>
__device__ __forceinline__ void put_quad(ET* tile, int i, typename Mma<ET>::quad v) {
    const int lane = threadIdx.x % MTS_WAVE;
    *reinterpret_cast<typename Mma<ET>::quad*>(tile + chunk_off(lane % 32, i) + 4 * (lane / 32)) = v;
}
// transposed accumulators (64 x 32: two tiles)
template <typename ET>
__device__ __forceinline__ void store_rows(ET* tile, ET* head, int64_t stride, int first, int S, const f32x16 (&acc)[2], float scale) {
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        typename Mma<ET>::quad o;
#pragma unroll
        for (int r = 0; r < 4; ++r) o[r] = (ET)(acc[i / 4][i % 4 * 4 + r] * scale);
        put_quad<ET>(tile, i, o);
    }
    flush_rows(tile, head, stride, first, S);
}

// Rotary encoding (rope_kernel's pairs (d, d + 32) and its arithmetic) of a row that a lane holds as an operand: both elements of a pair are its own.
// cos, sin: the row's angles.
template <typename ET>
__device__ __forceinline__ void turn(typename Mma<ET>::frag (&f)[4], const ET* cos, const ET* sin) {
    typename Mma<ET>::frag c[4], s[4];
    own_frags<ET>(cos, c);
    own_frags<ET>(sin, s);
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const float x1 = (float)f[ks][j], x2 = (float)f[ks + 2][j];
            f[ks][j] = difference_of_rounded_products<ET>(x1, (float)c[ks][j], x2, (float)s[ks][j]);
            f[ks + 2][j] = sum_of_rounded_products<ET>(x2, (float)c[ks + 2][j], x1, (float)s[ks + 2][j]);
        }
}
// The same of a gradient turned back: in fp32, rounded once, on its way out.  cos, sin: the angles of the row of this lane's column.
template <typename ET>
__device__ __forceinline__ void store_rows_turned_back(ET* tile, ET* head, int64_t stride, int first, int S, const f32x16 (&acc)[2], float scale, const ET* cos,
                                                       const ET* sin) {
    typedef typename Mma<ET>::quad quad;
    Quad c[8], s[8];
    load_quads(cos, c);
    load_quads(sin, s);
#pragma unroll
    for (int g = 0; g < 4; ++g) {
        const quad c1 = __builtin_bit_cast(quad, c[g]), c2 = __builtin_bit_cast(quad, c[g + 4]);
        const quad s1 = __builtin_bit_cast(quad, s[g]), s2 = __builtin_bit_cast(quad, s[g + 4]);
        quad o1, o2;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const float g1 = acc[0][4 * g + r] * scale, g2 = acc[1][4 * g + r] * scale;
            o1[r] = (ET)fmaf(g1, (float)c1[r], g2 * (float)s2[r]);
            o2[r] = (ET)fmaf(g2, (float)c2[r], -(g1 * (float)s1[r]));
        }
        put_quad<ET>(tile, g, o1);
        put_quad<ET>(tile, g + 4, o2);
    }
    flush_rows(tile, head, stride, first, S);
}

// Blocks of one head on one XCD (its keys and values, or queries and gradients, are read by all of them); `order` counts the
// blocks of a head, the same for all heads before the next, so that the longest of a causal pass start first.  Every other
// round of an XCD's 32 CUs is dealt backwards, so that a CU that took the longest block of one takes the shortest of the next
// (batch 8: 33 -> 31 us forward, 127 -> 121 backward; 24: 75 -> 72 and 311 -> 304).
struct Where {
    int64_t bh;
    int order;
    __device__ __forceinline__ Where(int64_t BH) {
        const int64_t per = (BH + 7) / 8, total = gridDim.x / 8;
        int64_t j = blockIdx.x / 8;
        const int64_t round = j / kCusPerXcd;
        if (round % 2 && (round + 1) * kCusPerXcd <= total) j = (2 * round + 1) * kCusPerXcd - 1 - j;
        order = (int)(j / per);
        bh = (j % per) * 8 + blockIdx.x % 8;
    }
};

template <typename ET>
struct AttnArgs {
    Heads<const ET> q, k, v, o, dO;
    Heads<ET> out, dq, dk, dv;
    // Rotary angles [S, 64], or NULL: the forward kernel then turns the queries on their way in (and leaves them in q_turned, where that is
    // given), the backward kernels turn the gradients of queries and keys back on their way out.
    const ET *cos, *sin;
    Heads<ET> q_turned;
    float *lse, *delta;   // [BH, S]: log2 of the row's sum of exponentials; sum of dO * O
    int64_t BH;
    int heads, S, blocks;
    float scale;
};

// TURN: with rotary angles (AttnArgs::cos)
template <typename ET, bool CAUSAL, bool TURN>
__global__ __launch_bounds__(kThreads, 3) void attention_fwd_kernel(AttnArgs<ET> a) {
    typedef typename Mma<ET>::frag frag;
    __shared__ __align__(16) ET lds[2][2][kTileElems];
    const Where at(a.BH);
    if (at.bh >= a.BH) return;
    const int lane = threadIdx.x % MTS_WAVE, wave = threadIdx.x / MTS_WAVE, half = lane / 32;
    const int S = a.S, q0 = (CAUSAL ? a.blocks - 1 - at.order : at.order) * kOwn, first = q0 + 32 * wave, row = first + lane % 32;
    const ET *k = a.k.row0(at.bh, a.heads), *v = a.v.row0(at.bh, a.heads);
    TileCopy<ET> kc, vc;   // on their way before the queries are waited for
    kc.fetch(k, a.k.s, 0, S);
    vc.fetch(v, a.v.s, 0, S);
    frag q[4];
    own_frags<ET>(a.q.row0(at.bh, a.heads) + min(row, S - 1) * a.q.s, q);
    if constexpr (TURN) {
        const int64_t angle = (int64_t)min(row, S - 1) * kHead;
        turn<ET>(q, a.cos + angle, a.sin + angle);
    }
    const float sc = a.scale * kLog2e;
    float top = -INFINITY, sum = 0.f;
    f32x16 acc[2] = {};
    const int end = CAUSAL ? min(S, q0 + kOwn) : S, tiles = (end + kTile - 1) / kTile;
    kc.commit(lds[0][0]);
    vc.commit(lds[0][1]);
    __syncthreads();
    for (int t = 0; t < tiles; ++t) {
        const int kv0 = t * kTile;
        const ET *kt = lds[t & 1][0], *vt = lds[t & 1][1];
        if (t + 1 < tiles) {
            kc.fetch(k, a.k.s, kv0 + kTile, S);
            vc.fetch(v, a.v.s, kv0 + kTile, S);
        }
        if (!CAUSAL || kv0 <= first + 31) {
            f32x16 s[2] = {};
#pragma unroll
            for (int ks = 0; ks < 4; ++ks)
#pragma unroll
                for (int m = 0; m < 2; ++m) s[m] = Mma<ET>::mul(row_frag(kt, 32 * m, ks), q[ks], s[m]);
            if (kv0 + kTile > S || (CAUSAL && kv0 + kTile - 1 > first)) {
                const int last = CAUSAL ? min(row, S - 1) : S - 1;
#pragma unroll
                for (int m = 0; m < 2; ++m)
#pragma unroll
                    for (int i = 0; i < 16; ++i)
                        if (kv0 + 32 * m + 8 * (i / 4) + 4 * half + i % 4 > last) s[m][i] = -INFINITY;
            }
            float hi = s[0][0];
#pragma unroll
            for (int i = 0; i < 16; ++i) hi = fmaxf(hi, fmaxf(s[0][i], s[1][i]));
            hi = lane_pair<32>(hi, [](float a, float b) { return fmaxf(a, b); });
            if (__any(hi > top)) {
                const float next = fmaxf(top, hi), keep = next == top ? 1.f : __builtin_amdgcn_exp2f((top - next) * sc);
                top = next;
                sum *= keep;
#pragma unroll
                for (int dt = 0; dt < 2; ++dt)
#pragma unroll
                    for (int i = 0; i < 16; ++i) acc[dt][i] *= keep;
            }
            const float base = top == -INFINITY ? 0.f : -top * sc;   // nothing but -inf so far: every exponential is zero
#pragma unroll
            for (int m = 0; m < 2; ++m)
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    s[m][i] = __builtin_amdgcn_exp2f(fmaf(s[m][i], sc, base));
                    sum += s[m][i];
                }
#pragma unroll
            for (int m = 0; m < 2; ++m)
#pragma unroll
                for (int u = 0; u < 2; ++u) {
                    const frag p = narrowed<ET>(s[m], u);
#pragma unroll
                    for (int dt = 0; dt < 2; ++dt) acc[dt] = Mma<ET>::mul(column_frag(vt, 32 * m + 16 * u, 32 * dt), p, acc[dt]);
                }
        }
        if (t + 1 < tiles) {
            kc.commit(lds[(t + 1) & 1][0]);
            vc.commit(lds[(t + 1) & 1][1]);
        }
        __syncthreads();
    }
    sum = lane_pair<32>(sum, LaneSum());
    ET* tile = &lds[0][0][0] + wave * 32 * kHead;   // the loop has ended with a barrier
    store_rows(tile, a.out.row0(at.bh, a.heads), a.out.s, first, S, acc, 1.f / sum);
    if constexpr (TURN) {   // here and not where they are turned: a tile's loads would be waited for behind these stores
        if (a.q_turned.p) {
            tile += kOwn * kHead;
#pragma unroll
            for (int ks = 0; ks < 4; ++ks) *reinterpret_cast<frag*>(tile + chunk_off(lane % 32, 2 * ks + half)) = q[ks];
            flush_rows(tile, a.q_turned.row0(at.bh, a.heads), a.q_turned.s, first, S);
        }
    }
    if (half == 0 && row < S) a.lse[at.bh * S + row] = top * sc + log2f(sum);
}

// dQ of 128 queries; also delta, which the other kernel reads.  Three blocks a CU (at 171 registers and two of them 116 us for 102).
template <typename ET, bool CAUSAL, bool TURN>
__global__ __launch_bounds__(kThreads, 3) void attention_dq_kernel(AttnArgs<ET> a) {
    typedef typename Mma<ET>::frag frag;
    __shared__ __align__(16) ET lds[2][2][kTileElems];
    const Where at(a.BH);
    if (at.bh >= a.BH) return;
    const int lane = threadIdx.x % MTS_WAVE, wave = threadIdx.x / MTS_WAVE, half = lane / 32;
    const int S = a.S, q0 = (CAUSAL ? a.blocks - 1 - at.order : at.order) * kOwn, first = q0 + 32 * wave, row = first + lane % 32;
    const int64_t from = min(row, S - 1);
    const ET *k = a.k.row0(at.bh, a.heads), *v = a.v.row0(at.bh, a.heads);
    frag q[4], g[4];
    own_frags<ET>(a.q.row0(at.bh, a.heads) + from * a.q.s, q);
    own_frags<ET>(a.dO.row0(at.bh, a.heads) + from * a.dO.s, g);
    float delta = 0.f;
    {
        frag o[4];
        own_frags<ET>(a.o.row0(at.bh, a.heads) + from * a.o.s, o);
#pragma unroll
        for (int ks = 0; ks < 4; ++ks)
#pragma unroll
            for (int j = 0; j < 8; ++j) delta += (float)o[ks][j] * (float)g[ks][j];
        delta = lane_pair<32>(delta, LaneSum());
        if (half == 0 && row < S) a.delta[at.bh * S + row] = delta;
    }
    const float sc = a.scale * kLog2e, lse = a.lse[at.bh * S + from];
    f32x16 acc[2] = {};
    const int end = CAUSAL ? min(S, q0 + kOwn) : S, tiles = (end + kTile - 1) / kTile;
    TileCopy<ET> kc, vc;
    kc.fetch(k, a.k.s, 0, S);
    vc.fetch(v, a.v.s, 0, S);
    kc.commit(lds[0][0]);
    vc.commit(lds[0][1]);
    __syncthreads();
    for (int t = 0; t < tiles; ++t) {
        const int kv0 = t * kTile;
        const ET *kt = lds[t & 1][0], *vt = lds[t & 1][1];
        if (t + 1 < tiles) {
            kc.fetch(k, a.k.s, kv0 + kTile, S);
            vc.fetch(v, a.v.s, kv0 + kTile, S);
        }
#pragma unroll
        for (int m = 0; m < 2; ++m) {
            const int kvm = kv0 + 32 * m;
            if (CAUSAL && kvm > first + 31) continue;
            f32x16 s = {}, d = {};
#pragma unroll
            for (int ks = 0; ks < 4; ++ks) {
                s = Mma<ET>::mul(row_frag(kt, 32 * m, ks), q[ks], s);
                d = Mma<ET>::mul(row_frag(vt, 32 * m, ks), g[ks], d);
            }
#pragma unroll
            for (int i = 0; i < 16; ++i) s[i] = __builtin_amdgcn_exp2f(fmaf(s[i], sc, -lse));
            if (kvm + 32 > S || (CAUSAL && kvm + 31 > first)) {
                const int last = CAUSAL ? min(row, S - 1) : S - 1;
#pragma unroll
                for (int i = 0; i < 16; ++i)
                    if (kvm + 8 * (i / 4) + 4 * half + i % 4 > last) s[i] = 0.f;
            }
#pragma unroll
            for (int i = 0; i < 16; ++i) s[i] *= d[i] - delta;
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                const frag ds = narrowed<ET>(s, u);
#pragma unroll
                for (int dt = 0; dt < 2; ++dt) acc[dt] = Mma<ET>::mul(column_frag(kt, 32 * m + 16 * u, 32 * dt), ds, acc[dt]);
            }
        }
        if (t + 1 < tiles) {
            kc.commit(lds[(t + 1) & 1][0]);
            vc.commit(lds[(t + 1) & 1][1]);
        }
        __syncthreads();
    }
    ET *tile = &lds[0][0][0] + wave * 32 * kHead, *dq = a.dq.row0(at.bh, a.heads);
    if constexpr (TURN) store_rows_turned_back(tile, dq, a.dq.s, first, S, acc, a.scale, a.cos + from * kHead, a.sin + from * kHead);
    else store_rows(tile, dq, a.dq.s, first, S, acc, a.scale);
}

// dK and dV of 128 keys.
template <typename ET, bool CAUSAL, bool TURN>
__global__ __launch_bounds__(kThreads, 2) void attention_dkdv_kernel(AttnArgs<ET> a) {
    typedef typename Mma<ET>::frag frag;
    __shared__ __align__(16) ET lds[2][2][kTileElems];
    __shared__ __align__(16) float stats[2][2][kTile];
    const Where at(a.BH);
    if (at.bh >= a.BH) return;
    const int lane = threadIdx.x % MTS_WAVE, wave = threadIdx.x / MTS_WAVE, half = lane / 32;
    const int S = a.S, first = at.order * kOwn + 32 * wave, row = first + lane % 32;
    const int64_t from = min(row, S - 1);
    const ET *q = a.q.row0(at.bh, a.heads), *g = a.dO.row0(at.bh, a.heads);
    const float *lse = a.lse + at.bh * S, *delta = a.delta + at.bh * S;
    frag k[4], v[4];
    own_frags<ET>(a.k.row0(at.bh, a.heads) + from * a.k.s, k);
    own_frags<ET>(a.v.row0(at.bh, a.heads) + from * a.v.s, v);
    const float sc = a.scale * kLog2e;
    f32x16 dk[2] = {}, dv[2] = {};
    const int t0 = CAUSAL ? at.order * kOwn / kTile : 0, tiles = (S + kTile - 1) / kTile;
    TileCopy<ET> qc, gc;
    float stat = 0.f;
    auto fetch = [&](int t) {
        qc.fetch(q, a.q.s, t * kTile, S);
        gc.fetch(g, a.dO.s, t * kTile, S);
        if (threadIdx.x < 2 * kTile) {   // queries behind the end: the exponential of -inf
            const int r = t * kTile + threadIdx.x % kTile;
            stat = threadIdx.x < kTile ? (r < S ? lse[r] : INFINITY) : (r < S ? delta[r] : 0.f);
        }
    };
    auto commit = [&](int buf) {
        qc.commit(lds[buf][0]);
        gc.commit(lds[buf][1]);
        if (threadIdx.x < 2 * kTile) stats[buf][threadIdx.x / kTile][threadIdx.x % kTile] = stat;
    };
    fetch(t0);
    commit(t0 & 1);
    __syncthreads();
    for (int t = t0; t < tiles; ++t) {
        const ET *qt = lds[t & 1][0], *gt = lds[t & 1][1];
        if (t + 1 < tiles) fetch(t + 1);
#pragma unroll
        for (int m = 0; m < 2; ++m) {
            const int qm = t * kTile + 32 * m;
            if (CAUSAL && qm + 31 < first) continue;
            f32x16 s = {}, d = {};
#pragma unroll
            for (int ks = 0; ks < 4; ++ks) {
                s = Mma<ET>::mul(row_frag(qt, 32 * m, ks), k[ks], s);
                d = Mma<ET>::mul(row_frag(gt, 32 * m, ks), v[ks], d);
            }
            const float *l = stats[t & 1][0] + 32 * m + 4 * half, *dl = stats[t & 1][1] + 32 * m + 4 * half;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const f32x4 l4 = *reinterpret_cast<const f32x4*>(l + 8 * j);
#pragma unroll
                for (int r = 0; r < 4; ++r) s[4 * j + r] = __builtin_amdgcn_exp2f(fmaf(s[4 * j + r], sc, -l4[r]));
            }
            if (CAUSAL && qm < first + 31) {
#pragma unroll
                for (int i = 0; i < 16; ++i)
                    if (qm + 8 * (i / 4) + 4 * half + i % 4 < row) s[i] = 0.f;
            }
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                const frag p = narrowed<ET>(s, u);
#pragma unroll
                for (int dt = 0; dt < 2; ++dt) dv[dt] = Mma<ET>::mul(column_frag(gt, 32 * m + 16 * u, 32 * dt), p, dv[dt]);
            }
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const f32x4 d4 = *reinterpret_cast<const f32x4*>(dl + 8 * j);
#pragma unroll
                for (int r = 0; r < 4; ++r) s[4 * j + r] *= d[4 * j + r] - d4[r];
            }
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                const frag ds = narrowed<ET>(s, u);
#pragma unroll
                for (int dt = 0; dt < 2; ++dt) dk[dt] = Mma<ET>::mul(column_frag(qt, 32 * m + 16 * u, 32 * dt), ds, dk[dt]);
            }
        }
        if (t + 1 < tiles) commit((t + 1) & 1);
        __syncthreads();
    }
    ET *tile = &lds[0][0][0] + wave * 32 * kHead, *to = a.dk.row0(at.bh, a.heads);
    store_rows(tile, a.dv.row0(at.bh, a.heads), a.dv.s, first, S, dv, 1.f);
    tile += kOwn * kHead;
    if constexpr (TURN) store_rows_turned_back(tile, to, a.dk.s, first, S, dk, a.scale, a.cos + from * kHead, a.sin + from * kHead);
    else store_rows(tile, to, a.dk.s, first, S, dk, a.scale);
}

template <typename T>
Heads<T> heads_of(const MtsHeads& t) {
    return {(T*)t.data, t.batch_stride, t.head_stride, t.row_stride};
}

bool heads_ok(const MtsHeads& t) {
    return t.data && mts_aligned16(t.data) && t.batch_stride % 8 == 0 && t.head_stride % 8 == 0 && t.row_stride % 8 == 0;
}

int attention_shape(const MtsHeads* const* tensors, int count, int64_t B, int heads, int64_t S, int act_dtype) {
    for (int i = 0; i < count; ++i) {
        if (!tensors[i] || !tensors[i]->data) return MTS_ERR_NULL;
        if (!heads_ok(*tensors[i])) return MTS_ERR_ALIGN;
    }
    if (act_dtype != MTS_BF16 && act_dtype != MTS_F16) return MTS_ERR_DTYPE;
    if (!mts_attention_supported(B, heads, S, kHead)) return MTS_ERR_SHAPE;
    return MTS_OK;
}

template <typename ET>
AttnArgs<ET> attention_args(const MtsHeads* q, const MtsHeads* k, const MtsHeads* v, int64_t B, int heads, int64_t S) {
    AttnArgs<ET> a = {};
    a.q = heads_of<const ET>(*q), a.k = heads_of<const ET>(*k), a.v = heads_of<const ET>(*v);
    a.BH = B * heads, a.heads = heads, a.S = (int)S, a.blocks = (int)((S + kOwn - 1) / kOwn);
    a.scale = 0.125f;   // 1 / sqrt(64)
    return a;
}

template <typename ET>
dim3 attention_grid(const AttnArgs<ET>& a) { return dim3((unsigned)((a.BH + 7) / 8 * 8 * a.blocks)); }

#define MTS_ATTENTION_LAUNCH(KERNEL)                                                                  \
    if (a.cos && causal) KERNEL<ET, true, true><<<attention_grid(a), kThreads, 0, st>>>(a);           \
    else if (a.cos) KERNEL<ET, false, true><<<attention_grid(a), kThreads, 0, st>>>(a);               \
    else if (causal) KERNEL<ET, true, false><<<attention_grid(a), kThreads, 0, st>>>(a);              \
    else KERNEL<ET, false, false><<<attention_grid(a), kThreads, 0, st>>>(a);

template <typename ET>
int attention_fwd(const MtsHeads* q, const MtsHeads* k, const MtsHeads* v, int64_t B, int heads, int64_t S, int causal, const MtsHeads* out, float* lse,
                  const void* cos, const void* sin, const MtsHeads* q_turned, hipStream_t st) {
    AttnArgs<ET> a = attention_args<ET>(q, k, v, B, heads, S);
    a.out = heads_of<ET>(*out), a.lse = lse;
    a.cos = (const ET*)cos, a.sin = (const ET*)sin;
    if (q_turned) a.q_turned = heads_of<ET>(*q_turned);
    MTS_ATTENTION_LAUNCH(attention_fwd_kernel)
    MTS_CHECK_LAUNCH();
    return MTS_OK;
}

template <typename ET>
int attention_bwd(const MtsHeads* q, const MtsHeads* k, const MtsHeads* v, const MtsHeads* out, const MtsHeads* d_out, const float* lse, int64_t B,
                  int heads, int64_t S, int causal, const MtsHeads* dq, const MtsHeads* dk, const MtsHeads* dv, float* delta,
                  const void* cos, const void* sin, hipStream_t st) {
    AttnArgs<ET> a = attention_args<ET>(q, k, v, B, heads, S);
    a.cos = (const ET*)cos, a.sin = (const ET*)sin;
    a.o = heads_of<const ET>(*out), a.dO = heads_of<const ET>(*d_out);
    a.dq = heads_of<ET>(*dq), a.dk = heads_of<ET>(*dk), a.dv = heads_of<ET>(*dv);
    a.lse = const_cast<float*>(lse), a.delta = delta;
    MTS_ATTENTION_LAUNCH(attention_dq_kernel)
    MTS_CHECK_LAUNCH();
    MTS_ATTENTION_LAUNCH(attention_dkdv_kernel)
    MTS_CHECK_LAUNCH();
    return MTS_OK;
}

}  // namespace

extern "C" int mts_attention_supported(int64_t B, int heads, int64_t S, int head_dim) {
    if (B <= 0 || heads <= 0 || S <= 0 || head_dim != kHead || S > (1 << 24) || B >= (1LL << 31)) return 0;
    return (B * heads + 7) / 8 * 8 * ((S + kOwn - 1) / kOwn) * kThreads < (1LL << 32);
}

static int attention_fwd_any(const MtsHeads* q, const MtsHeads* k, const MtsHeads* v, int64_t B, int heads, int64_t S, int causal, int act_dtype, const MtsHeads* out,
                             float* lse, const void* cos, const void* sin, const MtsHeads* q_turned, void* stream) {
    const MtsHeads* all[] = {q, k, v, out, q_turned};
    if (!lse) return MTS_ERR_NULL;
    if (int e = attention_shape(all, q_turned ? 5 : 4, B, heads, S, act_dtype)) return e;
    if (!mts_aligned16(cos) || !mts_aligned16(sin)) return MTS_ERR_ALIGN;
    if (act_dtype == MTS_BF16) return attention_fwd<bf16_t>(q, k, v, B, heads, S, causal, out, lse, cos, sin, q_turned, (hipStream_t)stream);
    return attention_fwd<mts_f16_t>(q, k, v, B, heads, S, causal, out, lse, cos, sin, q_turned, (hipStream_t)stream);
}
static int attention_bwd_any(const MtsHeads* q, const MtsHeads* k, const MtsHeads* v, const MtsHeads* out, const MtsHeads* d_out, const float* lse, int64_t B, int heads,
                             int64_t S, int causal, int act_dtype, const MtsHeads* dq, const MtsHeads* dk, const MtsHeads* dv, float* delta, const void* cos,
                             const void* sin, void* stream) {
    const MtsHeads* all[] = {q, k, v, out, d_out, dq, dk, dv};
    if (!lse || !delta) return MTS_ERR_NULL;
    if (int e = attention_shape(all, 8, B, heads, S, act_dtype)) return e;
    if (!mts_aligned16(cos) || !mts_aligned16(sin)) return MTS_ERR_ALIGN;
    if (act_dtype == MTS_BF16) return attention_bwd<bf16_t>(q, k, v, out, d_out, lse, B, heads, S, causal, dq, dk, dv, delta, cos, sin, (hipStream_t)stream);
    return attention_bwd<mts_f16_t>(q, k, v, out, d_out, lse, B, heads, S, causal, dq, dk, dv, delta, cos, sin, (hipStream_t)stream);
}

extern "C" int mts_attention_fwd(const MtsHeads* q, const MtsHeads* k, const MtsHeads* v, int64_t B, int heads, int64_t S, int causal, int act_dtype,
                                 const MtsHeads* out, float* lse, void* stream) {
    return attention_fwd_any(q, k, v, B, heads, S, causal, act_dtype, out, lse, nullptr, nullptr, nullptr, stream);
}

extern "C" int mts_attention_bwd(const MtsHeads* q, const MtsHeads* k, const MtsHeads* v, const MtsHeads* out, const MtsHeads* d_out, const float* lse,
                                 int64_t B, int heads, int64_t S, int causal, int act_dtype, const MtsHeads* dq, const MtsHeads* dk, const MtsHeads* dv,
                                 float* delta, void* stream) {
    return attention_bwd_any(q, k, v, out, d_out, lse, B, heads, S, causal, act_dtype, dq, dk, dv, delta, nullptr, nullptr, stream);
}

extern "C" int mts_attention_turned_fwd(const MtsHeads* q, const MtsHeads* k_turned, const MtsHeads* v, const void* cos, const void* sin, int64_t B, int heads,
                                        int64_t S, int causal, int act_dtype, const MtsHeads* q_turned, const MtsHeads* out, float* lse, void* stream) {
    if (!cos || !sin) return MTS_ERR_NULL;
    return attention_fwd_any(q, k_turned, v, B, heads, S, causal, act_dtype, out, lse, cos, sin, q_turned, stream);
}

extern "C" int mts_attention_turned_bwd(const MtsHeads* q_turned, const MtsHeads* k_turned, const MtsHeads* v, const MtsHeads* out, const MtsHeads* d_out,
                                        const float* lse, const void* cos, const void* sin, int64_t B, int heads, int64_t S, int causal, int act_dtype,
                                        const MtsHeads* dq, const MtsHeads* dk, const MtsHeads* dv, float* delta, void* stream) {
    if (!cos || !sin) return MTS_ERR_NULL;
    return attention_bwd_any(q_turned, k_turned, v, out, d_out, lse, B, heads, S, causal, act_dtype, dq, dk, dv, delta, cos, sin, stream);
}
