// attention_bwd_mfma.hip -- the gradient of the attention core for heads up to
// 128, on the bf16 matrix cores with fp32 operands held as three bf16 terms
// (split.hpp).
//
// Reference: the per-head part of backward_self_attention (Model.cpp:
// 6892-7028) and backward_cross_attention (:7122-7246).  With s = scale q . k
// (causal j > i masked), p = exp(s - max) / (sum + 1e-9), dp = dout . v:
//   dV = P^T dO,  dS = P (dP - delta),  dQ = scale dS K,  dK = scale dS^T Q,
// delta_i = sum_j p_ij dp_ij.  Only visible 32 x 32 tiles are computed, and P is
// never stored:
// 1. attention_bwd_stats: each query's max, 1 / (sum + 1e-9) and delta, from the
//    scores and dP, both with the bits that step 2 computes again: where one key
//    has all the weight, dP - delta cancels to what the other keys leave, and to 0
//    where there is no other.  (out . dout, from the forward's output, is the
//    same number with another rounding: it left 1e-7 of dP there, up to a
//    hundred times dQ itself.)  A layer's output comes from it too, or, heads over
//    kOutDim, from the forward.
// 2. attention_bwd_kv: a workgroup owns 128 keys and streams tiles of 32
//    queries.  Its eight waves are four pairs, a pair for 32 keys: one wave
//    holds the K rows and computes S, then P, then dV += dO P; the other holds
//    the V rows and computes dP, takes P from its partner through LDS, forms
//    dS, and computes dK += Q dS.  So each holds one operand (96 registers at
//    128 dimensions) and one result (64) where a single wave for both would
//    need twice that and run alone on its SIMD; a pair shares a SIMD, and both
//    do the same two products per tile, so the code is one.  S and dP come
//    out with the queries as rows and the wave's keys as columns, the layout
//    of the second product's operand.  dS goes to memory in blocks of 32 x 32,
//    [key][query], for
// 3. attention_bwd_q: dQ += K dS^T, a wave for 32 queries, streaming 32 keys.
// dS is the only matrix in memory (the (sequence, head) pairs run in groups
// whose blocks fit kDsBytes), written and read once.
//
// Bound by latency and the barriers as much as by the matrix cores: at 8 x 32
// heads x 1024 x 128, causal, 1550 to 1680 us = 102 to 111 TFLOP/s of the five
// products counted (seven are run: S and dP in steps 1 and 2, then dV, dK and dQ).
// The kernels alone, traced: step 1 450 us, step 2 950 us with the matrix pipes
// busy 45% of the cycles (10% more with its tile in one buffer and three
// barriers), step 3 250 us.  Step 1 as the forward with out . dout took as long.
// 3.30 ms for the same products as library fp32 GEMMs with P and dS in memory; 4 x
// 16 heads x 512 x 128 causal 202 us, 96 x 333 x 777 x 80 273 us, against 1.2 ms (the
// GEMMs ran sequence by sequence).
//
// LDS of step 2: Q rows, dO rows, Q^T and dO^T of one tile in bf16 planes
// (114 KB at 128 dimensions), the pairs' P (16 KB) and the tile's max / sum /
// delta.  One buffer, each half refilled while the other is read.
#include "attention_tile.hpp"
#include "internal.hpp"

#include <float.h>
#include <math.h>

#include <algorithm>
#include <cmath>

using namespace mimir;

namespace {

constexpr int kWaves = 8;
constexpr int kThreads = kWaves * kWave;
constexpr int kKeysPerBlock = 128;
constexpr int kXcds = 8;
constexpr float kLog2e = 1.4426950408889634f;
constexpr int kBlockFloats = kTileRows * kTileRows;
// Heads up to this have their output from attention_bwd_stats too, where a layer
// wants it; at 96 dimensions a hundred registers would spill.  Layer backward, us (the
// forward beside the statistics / this): 2048 tokens, 16 heads of 64 713 / 624, 300 tokens,
// 8 heads of 64 115 / 103, 777 tokens, 8 heads of 32 107 / 93.
constexpr int kOutDim = 64;

struct BwdArgs {
    CoreBwd c;
    int32_t q_len, kv_len, heads, head_dim;
    // A product q . k times `sign` (of the scale) orders like the scores, and qscale
    // = |scale| log2(e) takes a difference of two to base-2 units.
    float qscale, sign;
    // Per query of each (sequence, head), in rows of stats_ld queries: the max of
    // its signed products, 1 / (sum + 1e-9) and delta, three planes
    // [n_bh][stats_ld] (rows past q_len zero).
    float* stats;
    int64_t stats_ld;
    // The keys of attention_bwd_stats dealt to several workgroups: max, sum and
    // sum_j e_j dp_j of each, [split][3][n_bh][stats_ld]; null: one workgroup.  Then,
    // where the output is wanted (c.att), sum_j e_j v_j, [split][n_bh][q_len][head_dim].
    float* stats_part;
    int32_t stats_splits;
    float* ds;                 // [n_bh][key tile][query tile][32 keys][32 queries]
    int32_t q_tiles, k_tiles;
    uint32_t bh0, n_bh;
    uint32_t blocks;           // blocks of queries (keys) per (sequence, head)
    // The queries (attention_bwd_kv) or keys (attention_bwd_q) dealt to
    // several workgroups: partial dV and dK, or dQ, [split][n_bh][rows]
    // [head_dim] each; null: one workgroup.
    int32_t splits, q_splits;
    float* part[3];            // dV, dK, dQ
};

// Workgroup (without its split) -> (sequence, head) and its block, the longest
// first; unsplit, each XCD keeps whole (sequence, head) pairs where they divide by
// the XCDs.
__device__ __forceinline__ void coords(const BwdArgs& a, uint32_t bid, uint32_t* bh, uint32_t* block) {
    uint32_t first = 0, owned = a.n_bh, idx = bid;
    if (a.n_bh % kXcds == 0) {
        owned = a.n_bh / kXcds;
        first = bid % kXcds * owned;
        idx = bid / kXcds;
    }
    *block = idx / owned;
    *bh = first + idx % owned;
}

// exp(score - max) of a product with its query's max: the difference is taken before
// it is scaled, so its error is relative to it and not to the two scores, and the
// largest of a row gives exactly 1.
__device__ __forceinline__ float weight(const BwdArgs& a, float product, float max) {
    return __builtin_amdgcn_exp2f((product * a.sign - max) * a.qscale);
}

// Running max, sum and sum of e dP of a query; a lane half holds its own share of
// the sums.
struct RowStats {
    float m, l, d;
    // One tile: products s, which become weights, and dP, of which the first `lim` of
    // the lane's half count.  Returns what earlier weights are scaled by.
    __device__ __forceinline__ float add(const BwdArgs& a, f16v& s, const f16v& dp, int lim) {
        f16v x;
#pragma unroll
        for (int r = 0; r < 16; ++r) x[r] = 8 * (r / 4) + r % 4 < lim ? s[r] * a.sign : -INFINITY;
        float top = fmaxf(fmaxf(fmaxf(x[0], x[1]), fmaxf(x[2], x[3])), fmaxf(fmaxf(x[4], x[5]), fmaxf(x[6], x[7])));
        top = fmaxf(top, fmaxf(fmaxf(fmaxf(x[8], x[9]), fmaxf(x[10], x[11])),
                               fmaxf(fmaxf(x[12], x[13]), fmaxf(x[14], x[15]))));
        top = fmaxf(m, fmaxf(top, __shfl_xor(top, 32)));
        const float alpha = __builtin_amdgcn_exp2f((m - top) * a.qscale);
        m = top;
        float sum = 0.f, dot = 0.f;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const bool sees = 8 * (r / 4) + r % 4 < lim;
            s[r] = sees ? weight(a, s[r], top) : 0.f;
            sum += s[r];
            dot += sees ? s[r] * dp[r] : 0.f;
        }
        l = l * alpha + sum;
        d = d * alpha + dot;
        return alpha;
    }
};

// Step 1: a wave for 32 queries (their rows of Q and dO in registers), streaming 32
// keys and values.  The scores come out as S^T = K Q^T, dP as V dO^T, the products
// of step 2 transposed.  OUT: and the output, out += V P^T as in attention.hip, from
// the same weights; heads up to kOutDim, above which the registers do not hold it
// (the forward runs beside this kernel there).
template <int DP, bool VEC, bool OUT>
__global__ __launch_bounds__(kThreads, 2) void attention_bwd_stats(BwdArgs a) {
    using Rows = RowTile<DP, kThreads, VEC>;
    using Cols = ColTile<DP, kThreads>;
    constexpr int kC = DP / 16, kDb = DP / 32;
    constexpr int kBuf = 2 * Rows::kBytes + (OUT ? Cols::kBytes : 0);  // K and V rows of a tile, V^T
    __shared__ __attribute__((aligned(16))) char lds[2 * kBuf];

    uint32_t bh, qblock;
    const int split = static_cast<int>(blockIdx.x % static_cast<uint32_t>(a.stats_splits));
    coords(a, blockIdx.x / static_cast<uint32_t>(a.stats_splits), &bh, &qblock);
    if (a.c.causal) qblock = a.blocks - 1 - qblock;  // the last queries see the most keys
    const uint32_t head = a.bh0 + bh;
    const int64_t b = head / static_cast<uint32_t>(a.heads);
    const int64_t hd = static_cast<int64_t>(head % static_cast<uint32_t>(a.heads)) * a.head_dim;
    const float* k = a.c.k + b * a.kv_len * a.c.ld_kv + hd;
    const float* v = a.c.v + b * a.kv_len * a.c.ld_kv + hd;
    const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;
    const int li = lane % 32, hf = lane / 32;
    const int qt = static_cast<int>(qblock) * kWaves + wave;  // this wave's query tile
    const int my_q = qt * kTileRows + li;
    const int last_qt = min(static_cast<int>(qblock) * kWaves + kWaves, a.q_tiles) - 1;
    const int all_tiles = a.c.causal ? min(a.k_tiles, last_qt + 1) : a.k_tiles;
    const int per = (all_tiles + a.stats_splits - 1) / a.stats_splits;
    const int t0 = min(split * per, all_tiles), n_tiles = min(t0 + per, all_tiles);
    const int wave_tiles = qt >= a.q_tiles ? 0 : min(n_tiles, a.c.causal ? qt + 1 : a.k_tiles);
    const int end = a.c.causal ? min(a.kv_len, my_q + 1) : a.kv_len;  // this lane's keys
    const int64_t row = min(my_q, a.q_len - 1);
    const float* q = a.c.q + (b * a.q_len + row) * a.c.ld_q + hd;
    const float* dout = a.c.dout + (b * a.q_len + row) * a.c.ld_dout + hd;

    Rows keys, values;
    Cols cols;
    keys.init(a.c.ld_kv, a.head_dim);
    values.init(a.c.ld_kv, a.head_dim);
    if constexpr (OUT) cols.init(a.c.ld_kv, a.head_dim);
    auto load = [&](int t) {
        keys.load(k, t, a.c.ld_kv, a.kv_len, a.head_dim);
        values.load(v, t, a.c.ld_kv, a.kv_len, a.head_dim);
        if constexpr (OUT) cols.load(v, t, a.c.ld_kv, a.kv_len, a.head_dim);
    };
    auto stash = [&](char* to) {
        keys.stash(to);
        values.stash(to + Rows::kBytes);
        if constexpr (OUT) cols.stash(to + 2 * Rows::kBytes);
    };
    if (t0 < n_tiles) load(t0);
    Split8 qx[kC], ox[kC];
    row_operand<DP, VEC>(q, hf, a.head_dim, 1.0f, qx);
    row_operand<DP, VEC>(dout, hf, a.head_dim, 1.0f, ox);
    // A masked key counts in the max with its score of -1e9 (Model.cpp:6906-6920);
    // the max starts at -1e30 (LayerOps.hpp:1052).
    const RowStats none{fmaxf((end < a.kv_len ? -1e9f : -1e30f) * kLog2e / a.qscale, -FLT_MAX), 0.f, 0.f};
    RowStats st = none;
    auto add = [&](RowStats& to, f16v& s, const f16v& dp, int t) {
        if ((t + 1) * kTileRows > a.kv_len || (a.c.causal && t == qt))
            return to.add(a, s, dp, end - t * kTileRows - 4 * hf);
        return to.add(a, s, dp, kTileRows);
    };
    f16v o[OUT ? kDb : 1];
#pragma unroll
    for (int d = 0; d < (OUT ? kDb : 1); ++d) o[d] = f16v{};
    if (t0 < n_tiles) {
        stash(lds);
        load(min(t0 + 1, n_tiles - 1));
    }
    __syncthreads();
    for (int t = t0; t < n_tiles; ++t) {
        const char* cur = lds + ((t - t0) & 1) * kBuf;
        char* const next = lds + ((t - t0 + 1) & 1) * kBuf;
        f16v s = f16v{}, dp = f16v{};
        if (t < wave_tiles) {
#pragma unroll
            for (int c = 0; c < kC; ++c) s = mfma_split_mirror(Rows::at(cur, li, hf, c), qx[c], s);
        }
        // Past the last tile the stash rewrites a buffer that is not read again,
        // and the load repeats the last tile.
        stash(next);
        load(min(t + 2, n_tiles - 1));
        if (t < wave_tiles) {
#pragma unroll
            for (int c = 0; c < kC; ++c) dp = mfma_split_mirror(Rows::at(cur + Rows::kBytes, li, hf, c), ox[c], dp);
            const float alpha = add(st, s, dp, t);
            if constexpr (OUT) {
                if (__any(alpha != 1.f)) {
#pragma unroll
                    for (int d = 0; d < kDb; ++d) o[d] *= alpha;
                }
#pragma unroll
                for (int c = 0; c < 2; ++c) {
                    float x[8];
#pragma unroll
                    for (int e = 0; e < 8; ++e) x[e] = s[8 * c + e];
                    const Split8 p = split8(x);
#pragma unroll
                    for (int d = 0; d < kDb; ++d) o[d] = mfma_split(Cols::at(cur + 2 * Rows::kBytes, li, hf, d, c), p, o[d]);
                }
            }
        }
        __syncthreads();
    }
    const bool in = my_q < a.q_len;
    // Queries whose sums are not finite: again on the fp32 matrix cores (split.hpp).
    // The others keep theirs, whose rounding is that of step 2.
    if (const uint32_t bad = bad_rows((st.l - st.l) + (st.d - st.d), in)) {
        RowStats redo = none;
#pragma unroll 1
        for (int t = t0; t < wave_tiles; ++t) {
            f16v s = f32_scores(k, a.c.ld_kv, t * kTileRows, a.kv_len, a.head_dim, q, 1.0f);
            const f16v dp = f32_scores(v, a.c.ld_kv, t * kTileRows, a.kv_len, a.head_dim, dout, 1.0f);
            add(redo, s, dp, t);
        }
        if (bad >> li & 1) st = redo;
    }
    st.l += __shfl_xor(st.l, 32);
    st.d += __shfl_xor(st.d, 32);
    const int64_t plane = a.n_bh * a.stats_ld;
    const float inv = 1.0f / (st.l + 1e-9f);
    if constexpr (OUT) {
        float* to = a.stats_part ? a.stats_part + 3 * a.stats_splits * plane + ((split * int64_t{a.n_bh} + bh) * a.q_len + row) * a.head_dim
                                 : a.c.att + (b * a.q_len + row) * a.c.ld_att + hd;
        const float scale = a.stats_part ? 1.0f : inv;
        const float check = store_columns<DP, VEC>(o, scale, to, in, hf, a.head_dim);
        // Not finite: with the final max, in fp32.
        if (const uint32_t bad = bad_rows(check, in)) {
#pragma unroll 1
            for (int d0 = 0; d0 < a.head_dim; d0 += 32) {
                f16v x = f16v{};
#pragma unroll 1
                for (int t = t0; t < wave_tiles; ++t) {
                    f16v s = f32_scores(k, a.c.ld_kv, t * kTileRows, a.kv_len, a.head_dim, q, 1.0f);
#pragma unroll
                    for (int r = 0; r < 16; ++r)
                        s[r] = t * kTileRows + 8 * (r / 4) + 4 * hf + r % 4 < end ? weight(a, s[r], st.m) : 0.f;
                    f32_accumulate<1>(v + d0, a.c.ld_kv, t * kTileRows, a.kv_len, a.head_dim - d0, s, 0, end, &x);
                }
                store_columns<32, VEC>(&x, scale, to + d0, in && (bad >> li & 1), hf, a.head_dim - d0);
            }
        }
    }
    if (hf || my_q >= a.stats_ld) return;
    float* out = a.stats + bh * a.stats_ld + my_q;
    if (a.stats_part) out = a.stats_part + (split * 3ll * a.n_bh + bh) * a.stats_ld + my_q;
    // Rows past the sequence, up to the tile's end: no weight.
    out[0] = in ? st.m : 0.f;
    out[plane] = in ? (a.stats_part ? st.l : inv) : 0.f;
    out[2 * plane] = in ? (a.stats_part ? st.d : st.d * inv) : 0.f;
}

// The splits' results of one query each, brought to one max; W floats of the
// output a thread (0: none is wanted).
template <int W>
__global__ __launch_bounds__(256) void attention_bwd_stats_sum(BwdArgs a) {
    const int64_t plane = a.n_bh * a.stats_ld, id = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
    const int per = W ? a.head_dim / W : 1;
    const int64_t at = id / per;
    if (at >= plane) return;
    const float* p = a.stats_part + at;
    float m = p[0], l = 0.f, d = 0.f;
    for (int s = 1; s < a.stats_splits; ++s) m = fmaxf(m, p[3 * s * plane]);
    for (int s = 0; s < a.stats_splits; ++s) {
        const float f = __builtin_amdgcn_exp2f((p[3 * s * plane] - m) * a.qscale);
        l += p[(3 * s + 1) * plane] * f;
        d += p[(3 * s + 2) * plane] * f;
    }
    const int64_t bh = at / a.stats_ld, i = at % a.stats_ld;
    const bool in = i < a.q_len;
    const float inv = 1.0f / (l + 1e-9f);
    const int col = static_cast<int>(id % per) * W;
    if (col == 0) {
        a.stats[at] = in ? m : 0.f;
        a.stats[plane + at] = in ? inv : 0.f;
        a.stats[2 * plane + at] = in ? d * inv : 0.f;
    }
    if constexpr (W > 0) {
        if (!in) return;
        const int64_t head = a.bh0 + bh, next = a.n_bh * int64_t{a.q_len} * a.head_dim;
        const float* x = a.stats_part + 3 * a.stats_splits * plane + (bh * a.q_len + i) * a.head_dim + col;
        float* to = a.c.att + (head / a.heads * a.q_len + i) * a.c.ld_att + head % a.heads * a.head_dim + col;
        typedef float fw __attribute__((ext_vector_type(W)));
        fw sum = fw(0.f);
        for (int s = 0; s < a.stats_splits; ++s)
            sum += *reinterpret_cast<const fw*>(x + s * next) * __builtin_amdgcn_exp2f((p[3 * s * plane] - m) * a.qscale);
        *reinterpret_cast<fw*>(to) = sum * inv;
    }
}

// The gradient of a wave's 32 keys on the fp32 matrix cores (attention_tile.hpp),
// over query tiles t0 .. t1 - 1, for 32 NB dimensions from d0 on: dV (role 0) or dK /
// scale (role 1).
template <int NB>
__device__ __forceinline__ void keys_f32(const BwdArgs& a, int role, int key, int t0, int t1, int d0, const float* q,
                                         const float* k, const float* v, const float* dout, const float* stats, int64_t plane,
                                         f16v* acc) {
    const int hf = threadIdx.x % kWave / 32;
    const int lo = a.c.causal ? key : 0;
    const float* const rows = role ? q : dout;
    const int64_t ld = role ? a.c.ld_q : a.c.ld_dout;
#pragma unroll
    for (int d = 0; d < NB; ++d) acc[d] = f16v{};
#pragma unroll 1
    for (int t = t0; t < t1; ++t) {
        const int row0 = t * kTileRows;
        f16v w = f32_scores(q, a.c.ld_q, row0, a.q_len, a.head_dim, k + key * a.c.ld_kv, 1.0f), dp = f16v{};
        if (role) dp = f32_scores(dout, a.c.ld_dout, row0, a.q_len, a.head_dim, v + key * a.c.ld_kv, 1.0f);
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int i = row0 + 8 * (r / 4) + 4 * hf + r % 4;  // below stats_ld
            float p = weight(a, w[r], stats[i]) * stats[plane + i];
            if (role) p *= dp[r] - stats[2 * plane + i];
            w[r] = i >= lo && i < a.q_len ? p : 0.f;
        }
        f32_accumulate<NB>(rows + d0, ld, row0, a.q_len, a.head_dim - d0, w, lo, a.q_len, acc);
    }
}

// The same for a wave's 32 queries, over key tiles t0 .. t1 - 1, for 32
// dimensions: dQ / scale.  stats: the lane's query's.
__device__ __forceinline__ void queries_f32(const BwdArgs& a, int end, int t0, int t1, int d0, const float* q, const float* k,
                                            const float* v, const float* dout, const float* stats, int64_t plane, f16v& acc) {
    const int hf = threadIdx.x % kWave / 32;
    const float m = stats[0], inv = stats[plane], delta = stats[2 * plane];
    acc = f16v{};
#pragma unroll 1
    for (int t = t0; t < t1; ++t) {
        const int row0 = t * kTileRows;
        f16v w = f32_scores(k, a.c.ld_kv, row0, a.kv_len, a.head_dim, q, 1.0f);
        const f16v dp = f32_scores(v, a.c.ld_kv, row0, a.kv_len, a.head_dim, dout, 1.0f);
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const float ds = weight(a, w[r], m) * inv * (dp[r] - delta);
            w[r] = row0 + 8 * (r / 4) + 4 * hf + r % 4 < end ? ds : 0.f;
        }
        f32_accumulate<1>(k + d0, a.c.ld_kv, row0, a.kv_len, a.head_dim - d0, w, 0, end, &acc);
    }
}

template <int DP, bool VEC>
__global__ __launch_bounds__(kThreads, 2) void attention_bwd_kv(BwdArgs a) {
    using Rows = RowTile<DP, kThreads, VEC>;
    using Cols = ColTile<DP, kThreads>;
    constexpr int kC = DP / 16, kDb = DP / 32;
    constexpr int kRole = Rows::kBytes + Cols::kBytes;  // the rows and columns one role reads
    __shared__ __attribute__((aligned(16))) char lds[2 * kRole];
    __shared__ __attribute__((aligned(16))) f4 pshare[kWaves / 2][4][kWave];
    __shared__ __attribute__((aligned(16))) float tstats[2][3][kTileRows];

    uint32_t bh, kblock;
    const uint32_t split = blockIdx.x % static_cast<uint32_t>(a.splits);
    coords(a, blockIdx.x / static_cast<uint32_t>(a.splits), &bh, &kblock);
    const uint32_t head = a.bh0 + bh;
    const int64_t b = head / static_cast<uint32_t>(a.heads);
    const int64_t hd = static_cast<int64_t>(head % static_cast<uint32_t>(a.heads)) * a.head_dim;
    const float* q = a.c.q + b * a.q_len * a.c.ld_q + hd;
    const float* dout = a.c.dout + b * a.q_len * a.c.ld_dout + hd;
    const float* k = a.c.k + b * a.kv_len * a.c.ld_kv + hd;
    const float* v = a.c.v + b * a.kv_len * a.c.ld_kv + hd;
    const float* stats = a.stats + bh * a.stats_ld;
    const int64_t plane = a.n_bh * a.stats_ld;

    const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;
    const int li = lane % 32, hf = lane / 32;
    const int pair = wave % 4, role = __builtin_amdgcn_readfirstlane(wave / 4);
    const int k0 = static_cast<int>(kblock) * kKeysPerBlock + pair * kTileRows;
    const int key = k0 + li;
    const int ktile = k0 / kTileRows;
    // Query tiles the workgroup streams, and the first that this pair sees.
    const int first_t = a.c.causal ? min(static_cast<int>(kblock) * (kKeysPerBlock / kTileRows), a.q_tiles) : 0;
    const int per = (a.q_tiles - first_t + a.splits - 1) / a.splits;
    const int t0 = min(first_t + static_cast<int>(split) * per, a.q_tiles), t_end = min(t0 + per, a.q_tiles);
    const int pair_t0 = a.c.causal ? ktile : 0;
    const bool pair_in = k0 < a.kv_len;

    Rows qrows, drows;
    Cols qcols, dcols;
    qrows.init(a.c.ld_q, a.head_dim);
    qcols.init(a.c.ld_q, a.head_dim);
    drows.init(a.c.ld_dout, a.head_dim);
    dcols.init(a.c.ld_dout, a.head_dim);
    float stat = 0.f;
    // Role 0 reads Q rows and dO columns, role 1 dO rows and Q columns.
    auto load_rows = [&](int t) {
        qrows.load(q, t, a.c.ld_q, a.q_len, a.head_dim);
        drows.load(dout, t, a.c.ld_dout, a.q_len, a.head_dim);
        if (threadIdx.x < 3 * kTileRows) stat = stats[threadIdx.x / kTileRows * plane + t * kTileRows + threadIdx.x % kTileRows];
    };
    auto load_cols = [&](int t) {
        dcols.load(dout, t, a.c.ld_dout, a.q_len, a.head_dim);
        qcols.load(q, t, a.c.ld_q, a.q_len, a.head_dim);
    };
    auto stash_rows = [&](int t) {
        qrows.stash(lds);
        drows.stash(lds + kRole);
        if (threadIdx.x < 3 * kTileRows) tstats[t & 1][threadIdx.x / kTileRows][threadIdx.x % kTileRows] = stat;
    };
    auto stash_cols = [&]() {
        dcols.stash(lds + Rows::kBytes);
        qcols.stash(lds + kRole + Rows::kBytes);
    };
    if (t0 < t_end) {
        load_rows(t0);
        load_cols(t0);
    }
    Split8 own[kC];
    row_operand<DP, VEC>((role ? v : k) + static_cast<int64_t>(min(key, a.kv_len - 1)) * a.c.ld_kv, hf, a.head_dim, 1.0f, own);
    f16v acc[kDb];
#pragma unroll
    for (int d = 0; d < kDb; ++d) acc[d] = f16v{};
    const char* const rows = lds + role * kRole;
    const char* const cols = rows + Rows::kBytes;

    if (t0 < t_end) {
        stash_rows(t0);
        load_rows(min(t0 + 1, t_end - 1));
    }
    __syncthreads();
    // A tile has two phases, the first reading its rows and the second its
    // columns, so each phase's half of LDS is refilled during the other.  Of the
    // two waves of a SIMD one refills before its products and one after, so one's
    // vector work runs beside the other's MFMAs.  Past the last tile the refills
    // repeat it.
    for (int t = t0; t < t_end; ++t) {
        const float(*const ts)[kTileRows] = tstats[t & 1];
        const bool work = pair_in && t >= pair_t0;
        f16v x = f16v{};
        if (role) {
            stash_cols();
            load_cols(min(t + 1, t_end - 1));
        }
        if (work) {
#pragma unroll
            for (int c = 0; c < kC; ++c) x = mfma_split(Rows::at(rows, li, hf, c), own[c], x);
            if (role == 0) {
                // A tile that the diagonal or the last key crosses.
                const bool edge = k0 + kTileRows > a.kv_len || (a.c.causal && t == ktile);
#pragma unroll
                for (int r = 0; r < 16; r += 4) {
                    const f4 m = *reinterpret_cast<const f4*>(&ts[0][8 * (r / 4) + 4 * hf]);
                    const f4 inv = *reinterpret_cast<const f4*>(&ts[1][8 * (r / 4) + 4 * hf]);
                    f4 p;
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        p[e] = weight(a, x[r + e], m[e]) * inv[e];
                        if (edge && (key >= a.kv_len || (a.c.causal && key > t * kTileRows + 8 * (r / 4) + 4 * hf + e)))
                            p[e] = 0.f;
                        x[r + e] = p[e];
                    }
                    pshare[pair][r / 4][lane] = p;
                }
            }
        }
        if (!role) {
            stash_cols();
            load_cols(min(t + 1, t_end - 1));
        }
        __syncthreads();
        if (role) {
            stash_rows(t + 1);
            load_rows(min(t + 2, t_end - 1));
        }
        if (work) {
            if (role == 1) {
                float* block = a.ds + ((static_cast<int64_t>(bh) * a.k_tiles + ktile) * a.q_tiles + t) * kBlockFloats;
#pragma unroll
                for (int r = 0; r < 16; r += 4) {
                    const f4 p = pshare[pair][r / 4][lane];
                    const f4 delta = *reinterpret_cast<const f4*>(&ts[2][8 * (r / 4) + 4 * hf]);
                    f4 ds;
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        ds[e] = p[e] * (x[r + e] - delta[e]);
                        if (key >= a.kv_len) ds[e] = 0.f;
                        x[r + e] = ds[e];
                    }
                    *reinterpret_cast<f4*>(block + li * kTileRows + 8 * (r / 4) + 4 * hf) = ds;
                }
            }
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                float w[8];
#pragma unroll
                for (int e = 0; e < 8; ++e) w[e] = x[8 * c + e];
                const Split8 s = split8(w);
#pragma unroll
                for (int d = 0; d < kDb; ++d) acc[d] = mfma_split(Cols::at(cols, li, hf, d, c), s, acc[d]);
            }
        }
        if (!role) {
            stash_rows(t + 1);
            load_rows(min(t + 2, t_end - 1));
        }
        __syncthreads();
    }
    const bool in = key < a.kv_len;
    float* grad = (role ? a.c.dk : a.c.dv) + b * a.kv_len * a.c.ld_dkv + hd;
    int64_t ld = a.c.ld_dkv;
    if (a.part[role]) {
        ld = a.head_dim;
        grad = a.part[role] + (split * static_cast<int64_t>(a.n_bh) + bh) * a.kv_len * ld;
    }
    const int own_key = min(key, a.kv_len - 1);
    const float scale = role ? a.c.scale : 1.0f;
    grad += own_key * ld;
    const float check = store_columns<DP, VEC>(acc, scale, grad, in, hf, a.head_dim);
    // Keys whose result is not finite, in fp32 (split.hpp).
    if (const uint32_t bad = bad_rows(check, in)) {
        constexpr int kNb = kRedoBlocks<DP>;
#pragma unroll 1
        for (int d0 = 0; d0 < a.head_dim; d0 += 32 * kNb) {
            f16v x[kNb];
            keys_f32<kNb>(a, role, own_key, max(t0, pair_t0), t_end, d0, q, k, v, dout, stats, plane, x);
            store_columns<32 * kNb, VEC>(x, scale, grad + d0, in && (bad >> li & 1), hf, a.head_dim - d0);
        }
    }
}

// The splits' partial results added up, in order: grid.y chooses dV, dK or dQ.
template <bool VEC>
__global__ __launch_bounds__(256) void attention_bwd_sum(BwdArgs a) {
    constexpr uint32_t kW = VEC ? 4 : 1;
    const int which = blockIdx.y;
    const float* part = a.part[which];
    if (!part) return;
    const uint32_t len = which == 2 ? a.q_len : a.kv_len, row = a.head_dim / kW;
    const int splits = which == 2 ? a.q_splits : a.splits;
    const int64_t ld = which == 2 ? a.c.ld_dq : a.c.ld_dkv, one = static_cast<int64_t>(a.n_bh) * len * a.head_dim;
    float* out = which == 0 ? a.c.dv : which == 1 ? a.c.dk : a.c.dq;
    const uint32_t x = blockIdx.x * 256 + threadIdx.x;
    if (x >= a.n_bh * len * row) return;
    const uint32_t at = x / row, d = x % row * kW, head = a.bh0 + at / len, i = at % len;
    float* o = out + (static_cast<int64_t>(head / a.heads) * len + i) * ld + static_cast<int64_t>(head % a.heads) * a.head_dim + d;
    const float* p = part + static_cast<int64_t>(x) * kW;
    if constexpr (VEC) {
        f4 sum = *reinterpret_cast<const f4*>(p);
        for (int s = 1; s < splits; ++s) sum += *reinterpret_cast<const f4*>(p + s * one);
        *reinterpret_cast<f4*>(o) = sum;
    } else {
        float sum = *p;
        for (int s = 1; s < splits; ++s) sum += p[s * one];
        *o = sum;
    }
}

// dQ from dS: a wave for 32 queries; K^T tiles through LDS, dS blocks straight
// to registers (lane = query).
template <int DP, bool VEC>
__global__ __launch_bounds__(kThreads, 2) void attention_bwd_q(BwdArgs a) {
    using Cols = ColTile<DP, kThreads>;
    constexpr int kDb = DP / 32;
    __shared__ __attribute__((aligned(16))) char lds[2 * Cols::kBytes];

    uint32_t bh, qblock;
    const int split = static_cast<int>(blockIdx.x % static_cast<uint32_t>(a.q_splits));
    coords(a, blockIdx.x / static_cast<uint32_t>(a.q_splits), &bh, &qblock);
    if (a.c.causal) qblock = a.blocks - 1 - qblock;  // the last queries see the most keys
    const uint32_t head = a.bh0 + bh;
    const int64_t b = head / static_cast<uint32_t>(a.heads);
    const int64_t hd = static_cast<int64_t>(head % static_cast<uint32_t>(a.heads)) * a.head_dim;
    const float* k = a.c.k + b * a.kv_len * a.c.ld_kv + hd;
    const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;
    const int li = lane % 32, hf = lane / 32;
    const int qt = static_cast<int>(qblock) * kWaves + wave;  // this wave's query tile
    const int my_q = qt * kTileRows + li;
    const int last_qt = min(static_cast<int>(qblock) * kWaves + kWaves, a.q_tiles) - 1;
    const int all_tiles = a.c.causal ? min(a.k_tiles, last_qt + 1) : a.k_tiles;
    const int per = (all_tiles + a.q_splits - 1) / a.q_splits;
    const int t0 = min(split * per, all_tiles), n_tiles = min(t0 + per, all_tiles);
    const int wave_tiles = qt >= a.q_tiles ? 0 : min(n_tiles, a.c.causal ? qt + 1 : a.k_tiles);
    const float* ds = a.ds + (static_cast<int64_t>(bh) * a.k_tiles * a.q_tiles + min(qt, a.q_tiles - 1)) * kBlockFloats;

    Cols kcols;
    kcols.init(a.c.ld_kv, a.head_dim);
    float w[16];
    auto load_ds = [&](int t) {
        const float* block = ds + static_cast<int64_t>(min(t, max(wave_tiles - 1, 0))) * a.q_tiles * kBlockFloats + li;
#pragma unroll
        for (int r = 0; r < 16; ++r) w[r] = __builtin_nontemporal_load(block + (8 * (r / 4) + 4 * hf + r % 4) * kTileRows);
    };
    f16v acc[kDb];
#pragma unroll
    for (int d = 0; d < kDb; ++d) acc[d] = f16v{};
    if (t0 < n_tiles) {
        kcols.load(k, t0, a.c.ld_kv, a.kv_len, a.head_dim);
        if (t0 < wave_tiles) load_ds(t0);
        kcols.stash(lds);
        kcols.load(k, min(t0 + 1, n_tiles - 1), a.c.ld_kv, a.kv_len, a.head_dim);
    }
    __syncthreads();
    for (int t = t0; t < n_tiles; ++t) {
        const char* cur = lds + ((t - t0) & 1) * Cols::kBytes;
        if (t < wave_tiles) {
            Split8 s[2];
            s[0] = split8(w);
            s[1] = split8(w + 8);
            load_ds(t + 1);
#pragma unroll
            for (int c = 0; c < 2; ++c)
#pragma unroll
                for (int d = 0; d < kDb; ++d) acc[d] = mfma_split(Cols::at(cur, li, hf, d, c), s[c], acc[d]);
        }
        kcols.stash(lds + ((t - t0 + 1) & 1) * Cols::kBytes);
        kcols.load(k, min(t + 2, n_tiles - 1), a.c.ld_kv, a.kv_len, a.head_dim);
        __syncthreads();
    }
    const bool in = my_q < a.q_len;
    float* dq = a.c.dq + b * a.q_len * a.c.ld_dq + hd;
    int64_t ld = a.c.ld_dq;
    if (a.part[2]) {
        ld = a.head_dim;
        dq = a.part[2] + (split * static_cast<int64_t>(a.n_bh) + bh) * a.q_len * ld;
    }
    const int64_t row = min(my_q, a.q_len - 1);
    dq += row * ld;
    const float check = store_columns<DP, VEC>(acc, a.c.scale, dq, in, hf, a.head_dim);
    // Queries whose result is not finite, in fp32 (split.hpp); 32 dimensions a pass,
    // so that the kernel stays at 128 registers and two workgroups a CU.
    if (const uint32_t bad = bad_rows(check, in)) {
#pragma unroll 1
        for (int d0 = 0; d0 < a.head_dim; d0 += 32) {
            f16v x;
            queries_f32(a, a.c.causal ? min(a.kv_len, static_cast<int>(row) + 1) : a.kv_len, t0, wave_tiles, d0,
                        a.c.q + (b * a.q_len + row) * a.c.ld_q + hd, k, a.c.v + b * a.kv_len * a.c.ld_kv + hd,
                        a.c.dout + (b * a.q_len + row) * a.c.ld_dout + hd, a.stats + bh * a.stats_ld + row,
                        a.n_bh * a.stats_ld, x);
            store_columns<32, VEC>(&x, a.c.scale, dq + d0, in && (bad >> li & 1), hf, a.head_dim - d0);
        }
    }
}

int64_t tiles(int64_t n) { return (n + kTileRows - 1) / kTileRows; }
int64_t key_blocks(const CoreBwd& c) { return (c.kv_len + kKeysPerBlock - 1) / kKeysPerBlock; }
int64_t query_blocks(const CoreBwd& c) { return (tiles(c.q_len) + kWaves - 1) / kWaves; }

template <int DP>
int launch(mimir_ctx* ctx, BwdArgs a, bool vec) {
    a.blocks = static_cast<uint32_t>(query_blocks(a.c));
    const int64_t w = static_cast<int64_t>(a.n_bh) * a.blocks * a.stats_splits;
    const int per = !a.c.att ? 1 : vec ? a.head_dim / 4 : a.head_dim;  // threads a query in the sum
    const int64_t sums = (a.n_bh * a.stats_ld * per + 255) / 256;
    MIMIR_REQUIRE(ctx, dispatch_fits(w, kThreads) && dispatch_fits(sums, 256), "attention backward: grid too large");
    const auto wgs = static_cast<unsigned>(w);
    if (a.c.att) {
        if constexpr (DP <= kOutDim) {
            if (vec) attention_bwd_stats<DP, true, true><<<wgs, kThreads, 0, ctx->stream>>>(a);
            else attention_bwd_stats<DP, false, true><<<wgs, kThreads, 0, ctx->stream>>>(a);
        }
    } else if (vec) {
        attention_bwd_stats<DP, true, false><<<wgs, kThreads, 0, ctx->stream>>>(a);
    } else {
        attention_bwd_stats<DP, false, false><<<wgs, kThreads, 0, ctx->stream>>>(a);
    }
    if (int st = launched(ctx, "attention_bwd_stats")) return st;
    if (a.stats_part) {
        const auto blocks = static_cast<unsigned>(sums);
        if (!a.c.att) attention_bwd_stats_sum<0><<<blocks, 256, 0, ctx->stream>>>(a);
        else if (vec) attention_bwd_stats_sum<4><<<blocks, 256, 0, ctx->stream>>>(a);
        else attention_bwd_stats_sum<1><<<blocks, 256, 0, ctx->stream>>>(a);
        if (int st = launched(ctx, "attention_bwd_stats_sum")) return st;
    }
    a.blocks = static_cast<uint32_t>(key_blocks(a.c));
    const int64_t n = static_cast<int64_t>(a.n_bh) * a.blocks * a.splits;
    const int64_t m = static_cast<int64_t>(a.n_bh) * query_blocks(a.c) * a.q_splits;
    MIMIR_REQUIRE(ctx, dispatch_fits(std::max(n, m), kThreads), "attention backward: grid too large");
    if (vec) attention_bwd_kv<DP, true><<<static_cast<unsigned>(n), kThreads, 0, ctx->stream>>>(a);
    else attention_bwd_kv<DP, false><<<static_cast<unsigned>(n), kThreads, 0, ctx->stream>>>(a);
    if (int st = launched(ctx, "attention_bwd_kv")) return st;
    a.blocks = static_cast<uint32_t>(query_blocks(a.c));
    if (vec) attention_bwd_q<DP, true><<<static_cast<unsigned>(m), kThreads, 0, ctx->stream>>>(a);
    else attention_bwd_q<DP, false><<<static_cast<unsigned>(m), kThreads, 0, ctx->stream>>>(a);
    if (int st = launched(ctx, "attention_bwd_q")) return st;
    if (!a.part[0] && !a.part[2]) return MIMIR_OK;
    const int64_t rows = std::max(a.part[0] ? a.kv_len : 0, a.part[2] ? a.q_len : 0);
    const int64_t items = a.n_bh * rows * (vec ? a.head_dim / 4 : a.head_dim);
    MIMIR_REQUIRE(ctx, dispatch_fits((items + 255) / 256, 256), "attention backward: grid too large");
    const dim3 grid(static_cast<unsigned>((items + 255) / 256), 3);
    if (vec) attention_bwd_sum<true><<<grid, 256, 0, ctx->stream>>>(a);
    else attention_bwd_sum<false><<<grid, 256, 0, ctx->stream>>>(a);
    return launched(ctx, "attention_bwd_sum");
}

// (sequence, head) pairs per group: their dS blocks stay below kDsBytes.
// Measured at 8 x 32 heads x 1024 x 128, causal (us): 128 MiB 2599, 256 MiB
// 1998, 512 MiB 1703, 1 GiB 1710.
constexpr int64_t kDsBytes = int64_t{1} << 29;
int64_t group_of(const mimir_ctx* ctx, const CoreBwd& c) {
    const int64_t one = tiles(c.q_len) * tiles(c.kv_len) * kBlockFloats * static_cast<int64_t>(sizeof(float));
    int64_t n = std::min(c.batch * c.heads, std::max<int64_t>(1, kDsBytes / one));
    if (n < c.batch * c.heads && n > kXcds) n -= n % kXcds;
    if (ctx->tune.attn_bwd_heads > 0) n = std::min<int64_t>(n, ctx->tune.attn_bwd_heads);
    return n;
}

// Workgroups per block of 128 keys or 256 queries: the other side is split
// until the workgroups fill the GPU, four tiles each at least.  The target of
// 512 against 256 / 1024 (us): 16 heads x 2048 x 64 causal 304 / 349 / 330, 16 x
// 1024 x 128 218 / 210 / 267 (unsplit 364), 64 x 512 x 64 120 / 116 / 143.
int64_t splits_of(int64_t blocks, int64_t steps, int64_t target = 512) {
    return std::max<int64_t>(1, std::min<int64_t>(target / blocks, steps / 4));
}
int64_t kv_splits(const CoreBwd& c, int64_t n_bh) { return splits_of(n_bh * key_blocks(c), tiles(c.q_len)); }
int64_t q_splits(const CoreBwd& c, int64_t n_bh) { return splits_of(n_bh * query_blocks(c), tiles(c.kv_len)); }
// The statistics' workgroups run one to a CU: 256 fill it, and only a causal call's
// uneven blocks gain from more.  256 / 512, whole backward, us: 16 x 4 heads x 40 x 1500
// x 64 91 / 98, 8 x 16 x 512 x 512 x 128 390 / 408; causal, 2 x 16 x 2048 x 128 823 / 761,
// 4 x 12 x 700 x 80 195 / 182, 4 x 16 x 512 x 128 200 / 211.
int64_t stats_splits(const CoreBwd& c, int64_t n_bh) {
    return splits_of(n_bh * query_blocks(c), tiles(c.kv_len), c.causal ? 512 : 256);
}
// Floats of one partial result (rounded so that the next is 16-byte aligned).
int64_t part_floats(int64_t splits, int64_t n_bh, int64_t rows, int64_t head_dim) {
    return splits > 1 ? (splits * n_bh * rows * head_dim + 3) / 4 * 4 : 0;
}
int64_t ds_floats(const CoreBwd& c, int64_t n_bh) { return n_bh * tiles(c.q_len) * tiles(c.kv_len) * kBlockFloats; }
int64_t stats_floats(const CoreBwd& c, int64_t n_bh) { return 3 * n_bh * tiles(c.q_len) * kTileRows; }
int64_t parts_floats(const CoreBwd& c, int64_t n_bh) {
    // The statistics' partial results are gone before the others are written.
    const int64_t s = stats_splits(c, n_bh);
    return std::max(2 * part_floats(kv_splits(c, n_bh), n_bh, c.kv_len, c.head_dim) +
                        part_floats(q_splits(c, n_bh), n_bh, c.q_len, c.head_dim),
                    s > 1 ? s * (stats_floats(c, n_bh) + (c.head_dim <= kOutDim ? n_bh * c.q_len * c.head_dim : 0)) : 0);
}

}  // namespace

namespace mimir {

bool attention_bwd_mfma_takes(const CoreBwd& c) {
    const int64_t lim = (int64_t{1} << 31) / (4 * kTileRows);
    return c.head_dim <= 128 && c.kv_len > 0 && c.q_len > 0 && c.ld_q < lim && c.ld_kv < lim && c.ld_dout < lim;
}

int64_t attention_bwd_mfma_floats(const mimir_ctx* ctx, const CoreBwd& c) {
    const int64_t n = group_of(ctx, c), rest = c.batch * c.heads % n;  // the last group may be smaller and split more
    return ds_floats(c, n) + stats_floats(c, n) + std::max(parts_floats(c, n), rest ? parts_floats(c, rest) : 0);
}

int attention_bwd_mfma(mimir_ctx* ctx, const CoreBwd& c, float* work) {
    const int64_t group = group_of(ctx, c), total = c.batch * c.heads;
    const int64_t stats_ld = tiles(c.q_len) * kTileRows;
    auto vec4 = [](const float* p, int64_t ld) { return ld % 4 == 0 && aligned16(p); };
    const bool vec = c.head_dim % 4 == 0 && vec4(c.q, c.ld_q) && vec4(c.k, c.ld_kv) && vec4(c.v, c.ld_kv) &&
                     vec4(c.dout, c.ld_dout) && vec4(c.dq, c.ld_dq) && vec4(c.dk, c.ld_dkv) && vec4(c.dv, c.ld_dkv) &&
                     (!c.att || vec4(c.att, c.ld_att));
    BwdArgs a{};
    a.c = c;
    if (c.att && c.head_dim > kOutDim) {
        if (int st = mimir_attention_fwd(ctx, c.q, c.ld_q, c.k, c.v, c.ld_kv, c.att, c.ld_att, c.batch, c.q_len, c.kv_len,
                                         c.heads, c.head_dim, c.scale, c.causal))
            return st;
        a.c.att = nullptr;
    }
    a.q_len = static_cast<int32_t>(c.q_len);
    a.kv_len = static_cast<int32_t>(c.kv_len);
    a.heads = static_cast<int32_t>(c.heads);
    a.head_dim = static_cast<int32_t>(c.head_dim);
    a.qscale = std::max(std::fabs(c.scale) * kLog2e, FLT_MIN);  // a scale of 0: all weights the same
    a.sign = c.scale < 0 ? -1.0f : 1.0f;
    a.ds = work;  // 16-byte aligned blocks first
    a.stats = work + ds_floats(c, group);
    a.stats_ld = stats_ld;
    a.q_tiles = static_cast<int32_t>(tiles(c.q_len));
    a.k_tiles = static_cast<int32_t>(tiles(c.kv_len));
    for (int64_t h0 = 0; h0 < total; h0 += group) {
        a.bh0 = static_cast<uint32_t>(h0);
        a.n_bh = static_cast<uint32_t>(std::min(group, total - h0));
        float* const parts = a.stats + stats_floats(c, group);
        a.splits = static_cast<int32_t>(kv_splits(c, a.n_bh));
        a.q_splits = static_cast<int32_t>(q_splits(c, a.n_bh));
        a.stats_splits = static_cast<int32_t>(stats_splits(c, a.n_bh));
        a.stats_part = a.stats_splits > 1 ? parts : nullptr;
        const int64_t one = part_floats(a.splits, a.n_bh, c.kv_len, c.head_dim);
        a.part[0] = a.splits > 1 ? parts : nullptr;
        a.part[1] = a.splits > 1 ? parts + one : nullptr;
        a.part[2] = a.q_splits > 1 ? parts + 2 * one : nullptr;
        int e = MIMIR_OK;
        if (c.head_dim <= 32) e = launch<32>(ctx, a, vec);
        else if (c.head_dim <= 64) e = launch<64>(ctx, a, vec);
        else if (c.head_dim <= 96) e = launch<96>(ctx, a, vec);
        else e = launch<128>(ctx, a, vec);
        if (e) return e;
    }
    return MIMIR_OK;
}

}  // namespace mimir
