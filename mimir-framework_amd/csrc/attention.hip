// attention.hip -- the attention core softmax(Q K^T * scale) V with the
// softmax fused between the two products, on the gfx950 matrix cores.
//
// Reference: the core of LayerOps::self_attention_forward (LayerOps.hpp:
// 1045-1089) and cross_attention_forward (:1163-1209), which materialise one
// score row per query (s = dot * scale; causal j > i masked to -1e9; max from
// -1e30; e = exp(s - max); p = e / (sum + 1e-9); out = sum_j p_j V_j).  Here
// no score row is ever stored: each workgroup streams K / V tiles through LDS
// and keeps a running max / sum per query ("online softmax"; Milakov and
// Gimelshein 2018, as used by FlashAttention, Dao et al. 2022), rescaling its
// partial output when the max grows, and divides by (sum + 1e-9) at the end.
// Q is multiplied by scale * log2(e) once, so the scores come out of the
// matrix core in base-2 units and each probability is one v_exp_f32.
//
// Products.  Every fp32 operand (Q, K, V and the probabilities) is held as
// three bf16 terms and every product is six bf16 MFMAs (split.hpp): 6/16 of
// the fp32 matrix time.  v_mfma_f32_32x32x16_bf16 computes D[32x32] +=
// A[32x16] B[16x32]; lane l supplies A[l%32][8(l/32) + i], B[8(l/32) + i][l%32]
// (i = 0..7) and receives D[8(r/4) + 4(l/32) + r%4][l%32] in register r.
// - Scores: S^T = K Q^T, keys as rows, queries as columns.  Lane l owns query
//   l%32 (its share of Q split once, in registers for the whole kernel) and
//   16 of the 32 keys of the tile.
// - Softmax: per lane over its 16 keys; the max is shared with the other half
//   (lane l ^ 32, same query).
// - Output: O^T = V^T P^T.  Registers 8c .. 8c+7 of S^T hold P^T at the keys
//   16c + 4(l/32) + {0..3, 8..11}: the B operand of a product over 16 keys in
//   that order, so the probabilities feed it without a lane exchange, and V is
//   laid out in LDS in the same order.
//
// LDS: K planes [3][32 keys][DP] and V^T planes [3][DP][32 keys] in bf16, rows
// padded by 16 bytes (eight rows' 16-byte reads touch every bank once).  The
// tile is split on its way in, once for all queries of the workgroup: K in
// groups of eight dimensions of a row, V in groups of eight keys of a column.
// Two buffers: iteration t computes tile t while tile t+1 moves from registers
// to the other one and tile t+2 is on its way to the registers; one barrier.
//
// Workgroup: WAVES waves, 32 queries each, of one (sequence, head).
// Causal: a workgroup stops at its last query's diagonal, a wave skips the
// tiles past its own diagonal and masks inside its last tile only (the
// diagonal, or the sequence's ragged end).
// Grid: the hardware deals workgroups to the 8 XCDs round-robin.  When the
// (sequence, head) count divides by 8, each XCD owns an eighth of them (their
// K and V stay in that XCD's L2) and runs its query blocks longest first
// across all of its heads, so the short causal blocks fill the tail.
//
// Bound by the power the matrix cores draw: at 8 x 32 heads x 1024 tokens x 128,
// causal, the bf16 MFMAs hold the matrix pipes 51% of the cycles at 1.9 GHz (a
// loop of nothing else runs at 1.6 GHz), beside 350 VALU operations per 96
// MFMAs.  Measured there 404 to 413 us = 167 to 170 TFLOP/s of fp32 work, against
// 627 us on the fp32 MFMAs (157 TFLOP/s peak); 16 heads x 1024 x 128 70 / 152 us, 96
// heads x 333 x 777 x 80 80 / 213 us.  Within noise of that: two accumulators in
// turns, LDS reads ordered ahead of the MFMAs, the split interleaved with them,
// raised priority for half the waves; four waves with two workgroups' worth of
// LDS are slower (the tile is split twice as often).
#include "attention_tile.hpp"
#include "common.hpp"
#include "internal.hpp"

#include <math.h>

#include <algorithm>
#include <cmath>

using namespace mimir;

namespace {

constexpr int kQPerWave = 32;
constexpr int kKeyTile = 32;
constexpr int kXcds = 8;
constexpr float kLog2e = 1.4426950408889634f;
// The running max follows a growing score only past this many base-2 units:
// probabilities up to 2^8 of the final scale lose nothing in fp32, and the
// rescale of the output (DP / 2 multiplies) runs in few tiles instead of most.
constexpr float kMaxSlack = 8.0f;
// Workgroups of eight waves that fill the GPU.
constexpr int64_t kSplitTarget = 256;

struct AttnArgs {
    const float* q;
    const float* k;
    const float* v;
    float* out;
    int64_t ld_q, ld_kv, ld_out;  // row strides (floats)
    int32_t q_len, kv_len, heads, head_dim;
    int32_t n_qblocks;            // query blocks of one (sequence, head)
    uint32_t total_blocks;        // batch * heads * n_qblocks
    float qscale;                 // scale * log2(e), applied to Q
    int32_t causal;
    // Keys dealt to several workgroups: partial results [split][n_bh][q_len]
    // [head_dim | max | sum], null: one workgroup per query block.
    int32_t splits;
    float* part;
};

// Key tiles that a query block (queries q0 .. q0 + n) streams, and how many a
// split takes.
__device__ __forceinline__ int tiles_of(const AttnArgs& a, int q0, int n) {
    const int end = a.causal ? min(a.kv_len, min(q0 + n, a.q_len)) : a.kv_len;
    return (end + kKeyTile - 1) / kKeyTile;
}

// Workgroup (without its split) -> (sequence * heads + head, query block): see the
// file comment; the XCDs own whole (sequence, head) pairs where keys are not split.
__device__ __forceinline__ void block_coords(const AttnArgs& a, uint32_t bid, uint32_t* bh, int* qb) {
    const uint32_t n_bh = a.total_blocks / static_cast<uint32_t>(a.n_qblocks);
    uint32_t first = 0, owned = n_bh, idx = bid;
    if (n_bh % kXcds == 0) {
        owned = n_bh / kXcds;
        first = (bid % kXcds) * owned;
        idx = bid / kXcds;
    }
    *qb = a.n_qblocks - 1 - static_cast<int>(idx / owned);
    *bh = first + idx % owned;
}

// A wave's 32 queries on the fp32 matrix cores (attention_tile.hpp), over key
// tiles t0 .. t1 - 1, for 32 NB dimensions of the output (vbase and head_dim from
// the first of them on): the same online softmax.  `end`: where the lane's keys end.
template <int NB>
__device__ __forceinline__ void queries_f32(const AttnArgs& a, const float* qrow, const float* kbase, const float* vbase,
                                            int head_dim, int t0, int t1, int end, float* m, float* l, f16v* o) {
    const int hf = threadIdx.x % kWave / 32;
#pragma unroll
    for (int d = 0; d < NB; ++d) o[d] = f16v{};
    float m_run = -1e30f, l_run = 0.f;
#pragma unroll 1
    for (int t = t0; t < t1; ++t) {
        f16v s = f32_scores(kbase, a.ld_kv, t * kKeyTile, a.kv_len, a.head_dim, qrow, a.qscale);
        float m_new = m_run;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            s[r] = t * kKeyTile + 8 * (r / 4) + 4 * hf + r % 4 < end ? s[r] : -INFINITY;
            m_new = fmaxf(m_new, s[r]);
        }
        m_new = fmaxf(m_new, __shfl_xor(m_new, 32));
        const float alpha = __builtin_amdgcn_exp2f(m_run - m_new);
        m_run = m_new;
        l_run *= alpha;
#pragma unroll
        for (int d = 0; d < NB; ++d) o[d] *= alpha;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            s[r] = __builtin_amdgcn_exp2f(s[r] - m_run);
            l_run += s[r];
        }
        f32_accumulate<NB>(vbase, a.ld_kv, t * kKeyTile, a.kv_len, head_dim, s, 0, end, o);
    }
    *m = m_run;
    *l = l_run + __shfl_xor(l_run, 32);
}

template <int DP, int WAVES, bool VEC>
__global__ __launch_bounds__(WAVES * kWave, WAVES == 4 ? 1 : DP == 32 && VEC ? 4 : 2) void attention_fwd_mfma(AttnArgs a) {
    using Keys = RowTile<DP, WAVES * kWave, VEC>;
    using Values = ColTile<DP, WAVES * kWave>;
    constexpr int kBuf = Keys::kBytes + Values::kBytes;
    constexpr int kC = DP / 16;   // MFMA steps of a score
    constexpr int kDb = DP / 32;  // output dimension blocks
    __shared__ __attribute__((aligned(16))) char lds[2 * kBuf];

    uint32_t bh;
    int qb;
    const int split = static_cast<int>(blockIdx.x % static_cast<uint32_t>(a.splits));
    block_coords(a, blockIdx.x / static_cast<uint32_t>(a.splits), &bh, &qb);
    const int64_t b = bh / static_cast<uint32_t>(a.heads);
    const int64_t hd_off = static_cast<int64_t>(bh % static_cast<uint32_t>(a.heads)) * a.head_dim;
    const float* qbase = a.q + b * a.q_len * a.ld_q + hd_off;
    const float* kbase = a.k + b * a.kv_len * a.ld_kv + hd_off;
    const float* vbase = a.v + b * a.kv_len * a.ld_kv + hd_off;
    float* obase = a.out + b * a.q_len * a.ld_out + hd_off;

    const int wave = threadIdx.x / kWave;
    const int lane = threadIdx.x % kWave;
    const int li = lane % 32, hf = lane / 32;
    const int q0 = qb * kQPerWave * WAVES;
    const int qw0 = q0 + wave * kQPerWave;
    const int my_q = qw0 + li;

    // Tiles this workgroup streams, and the ones this wave computes.
    int wave_key_end = a.causal ? min(a.kv_len, min(qw0 + kQPerWave, a.q_len)) : a.kv_len;
    if (qw0 >= a.q_len) wave_key_end = 0;
    const int all_tiles = tiles_of(a, q0, kQPerWave * WAVES);
    const int per = (all_tiles + a.splits - 1) / a.splits;
    const int t0 = split * per;
    const int n_tiles = min(t0 + per, all_tiles);
    if (split > 0 && t0 >= n_tiles) return;
    const int wave_tiles = min(n_tiles, (wave_key_end + kKeyTile - 1) / kKeyTile);
    // Keys of this lane's query: the rest of its last tile is masked
    // (causal: key > query; all: key >= kv_len).
    const int lane_key_end = min(a.kv_len, a.causal ? my_q + 1 : a.kv_len);

    Keys keys;
    Values values;
    keys.init(a.ld_kv, a.head_dim);
    values.init(a.ld_kv, a.head_dim);
    auto load = [&](int t) {
        keys.load(kbase, t, a.ld_kv, a.kv_len, a.head_dim);
        values.load(vbase, t, a.ld_kv, a.kv_len, a.head_dim);
    };
    auto stash = [&](char* buf) {
        keys.stash(buf);
        values.stash(buf + Keys::kBytes);
    };
    if (n_tiles > t0) load(t0);

    // This lane's Q values, times scale*log2(e).
    Split8 q[kC];
    row_operand<DP, VEC>(qbase + static_cast<int64_t>(min(my_q, a.q_len - 1)) * a.ld_q, hf, a.head_dim, a.qscale, q);
    f16v o[kDb];
#pragma unroll
    for (int d = 0; d < kDb; ++d) o[d] = f16v{};
    float m_run = -1e30f;  // running max (base-2 units); the reference starts at -1e30 (LayerOps.hpp:1052)
    float m_top = -1e30f;  // the max itself: m_run lags behind it by up to kMaxSlack
    float l_run = 0.f;     // this half's share of the running sum

    if (n_tiles > t0) {
        stash(lds);
        load(min(t0 + 1, n_tiles - 1));
    }
    __syncthreads();

    for (int t = t0; t < n_tiles; ++t) {
        const char* cur = lds + ((t - t0) & 1) * kBuf;
        char* const next = lds + ((t - t0 + 1) & 1) * kBuf;
        if (t < wave_tiles) {
            f16v s = f16v{};
            __builtin_amdgcn_s_setprio(1);
#pragma unroll
            for (int c = 0; c < kC; ++c) s = mfma_split(Keys::at(cur, li, hf, c), q[c], s);
            // Past the last tile the stash rewrites a buffer that is not read
            // again, and the load repeats the last tile.
            stash(next);
            __builtin_amdgcn_s_setprio(0);
            load(min(t + 2, n_tiles - 1));
            if ((t + 1) * kKeyTile > a.kv_len || (a.causal && (t + 1) * kKeyTile - 1 > qw0)) {
                const int lim = lane_key_end - t * kKeyTile - 4 * hf;
#pragma unroll
                for (int r = 0; r < 16; ++r) s[r] = 8 * (r / 4) + (r % 4) < lim ? s[r] : -INFINITY;
            }
            float tmax = fmaxf(fmaxf(fmaxf(s[0], s[1]), fmaxf(s[2], s[3])), fmaxf(fmaxf(s[4], s[5]), fmaxf(s[6], s[7])));
            tmax = fmaxf(tmax, fmaxf(fmaxf(fmaxf(s[8], s[9]), fmaxf(s[10], s[11])),
                                     fmaxf(fmaxf(s[12], s[13]), fmaxf(s[14], s[15]))));
            tmax = fmaxf(tmax, __shfl_xor(tmax, 32));
            m_top = fmaxf(m_top, tmax);
            if (__any(tmax > m_run + kMaxSlack)) {
                const float m_new = fmaxf(m_run, tmax);
                const float alpha = __builtin_amdgcn_exp2f(m_run - m_new);
                m_run = m_new;
                l_run *= alpha;
#pragma unroll
                for (int d = 0; d < kDb; ++d) o[d] *= alpha;
            }
            float psum = 0.f;
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                s[r] = __builtin_amdgcn_exp2f(s[r] - m_run);  // exp2(-inf) = 0: masked keys
                psum += s[r];
            }
            l_run += psum;
            __builtin_amdgcn_s_setprio(1);
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                float x[8];
#pragma unroll
                for (int e = 0; e < 8; ++e) x[e] = s[8 * c + e];
                const Split8 p = split8(x);
#pragma unroll
                for (int d = 0; d < kDb; ++d) o[d] = mfma_split(Values::at(cur + Keys::kBytes, li, hf, d, c), p, o[d]);
            }
            __builtin_amdgcn_s_setprio(0);
        } else {
            stash(next);
            load(min(t + 2, n_tiles - 1));
        }
        __syncthreads();
    }

    // out = O / (sum + 1e-9) (LayerOps.hpp:1076-1079); a split's share in units of
    // the true max, so that the shares' sum stays below what one workgroup without
    // lag would hold.
    const float lag = __builtin_amdgcn_exp2f(m_run - m_top);
    const float l_tot = l_run + __shfl_xor(l_run, 32);
    const float inv = 1.0f / (l_tot + 1e-9f);
    const bool in = my_q < a.q_len;
    const int64_t row = min(my_q, a.q_len - 1);
    const int64_t n_bh = a.total_blocks / static_cast<uint32_t>(a.n_qblocks);
    float* const part = a.part ? a.part + ((split * n_bh + bh) * a.q_len + row) * (a.head_dim + 2) : nullptr;
    float* const out = obase + row * a.ld_out;
    float check;
    if (part) {
        check = store_columns<DP, false>(o, lag, part, in, hf, a.head_dim);
        if (in && hf == 0) {
            part[a.head_dim] = m_top;
            part[a.head_dim + 1] = l_tot * lag;
        }
    } else {
        check = store_columns<DP, VEC>(o, inv, out, in, hf, a.head_dim);
    }
    // Queries that came out NaN or infinite, again in fp32: their operands may have
    // had no bf16 split (split.hpp), or the lag of the max an overflow.
    if (const uint32_t bad = bad_rows(check + (l_tot - l_tot), in)) {
        constexpr int kNb = kRedoBlocks<DP>;
        const bool mine = in && (bad >> li & 1);
#pragma unroll 1
        for (int d0 = 0; d0 < a.head_dim; d0 += 32 * kNb) {
            f16v x[kNb];
            float m, l;
            queries_f32<kNb>(a, qbase + row * a.ld_q, kbase, vbase + d0, a.head_dim - d0, t0, wave_tiles, lane_key_end, &m, &l, x);
            if (part) {
                store_columns<32 * kNb, false>(x, 1.0f, part + d0, mine, hf, a.head_dim - d0);
                if (mine && hf == 0) {
                    part[a.head_dim] = m;
                    part[a.head_dim + 1] = l;
                }
            } else {
                store_columns<32 * kNb, VEC>(x, 1.0f / (l + 1e-9f), out + d0, mine, hf, a.head_dim - d0);
            }
        }
    }
}

// The splits of one query, one wave per query: their sums brought to one max,
// then what attention_fwd_mfma does with the whole.
__global__ __launch_bounds__(4 * kWave) void attention_fwd_combine(AttnArgs a, int queries_per_block) {
    constexpr int kCh = 2;  // heads up to 128
    const uint32_t n_bh = a.total_blocks / static_cast<uint32_t>(a.n_qblocks);
    const int64_t at = static_cast<int64_t>(blockIdx.x) * 4 + threadIdx.x / kWave;
    if (at >= static_cast<int64_t>(n_bh) * a.q_len) return;  // whole waves
    const int lane = threadIdx.x & (kWave - 1);
    const uint32_t bh = static_cast<uint32_t>(at / a.q_len);
    const int64_t i = at % a.q_len;
    const int64_t b = bh / static_cast<uint32_t>(a.heads);
    const int64_t hd_off = static_cast<int64_t>(bh % static_cast<uint32_t>(a.heads)) * a.head_dim;
    const int w = a.head_dim + 2;
    const float* p = a.part + at * w;
    const int64_t next = static_cast<int64_t>(n_bh) * a.q_len * w;
    const int all = tiles_of(a, static_cast<int>(i / queries_per_block) * queries_per_block, queries_per_block);
    const int per = (all + a.splits - 1) / a.splits, n = max(1, (all + per - 1) / max(per, 1));
    float m = -1e30f, l = 0.f, acc[kCh] = {0.f, 0.f};
    for (int s = 0; s < n; ++s) m = fmaxf(m, p[s * next + a.head_dim]);
    for (int s = 0; s < n; ++s) {
        const float* x = p + s * next;
        const float f = __builtin_amdgcn_exp2f(x[a.head_dim] - m);
        l += x[a.head_dim + 1] * f;
#pragma unroll
        for (int c = 0; c < kCh; ++c)
            if (lane + c * kWave < a.head_dim) acc[c] += x[lane + c * kWave] * f;
    }
    const float inv = 1.0f / (l + 1e-9f);
    float* const out = a.out + (b * a.q_len + i) * a.ld_out + hd_off;
#pragma unroll
    for (int c = 0; c < kCh; ++c)
        if (lane + c * kWave < a.head_dim) out[lane + c * kWave] = acc[c] * inv;
}

// Heads wider than 128 (up to 2048): one wave per query, the head's
// dimensions spread over the lanes (CH per lane, lane + 64 c), each score a
// DPP wave sum, the same online softmax (base-2 scores, running max and
// sum) and the same division by (sum + 1e-9).  Plain fp32 vector code: the
// reference accepts any head size, the matrix-core kernel's register layout
// stops at 128.  Keys are read row by row through L2 by all four waves of a
// workgroup (four queries).
constexpr int kGenericWaves = 4;
template <int CH>
__global__ __launch_bounds__(kGenericWaves * kWave) void attention_fwd_generic(AttnArgs a) {
    const int lane = threadIdx.x % kWave;
    const int64_t qi = static_cast<int64_t>(blockIdx.y) * kGenericWaves + threadIdx.x / kWave;
    if (qi >= a.q_len) return;  // whole waves leave: no barrier below
    const uint32_t bh = blockIdx.x;
    const int64_t b = bh / static_cast<uint32_t>(a.heads);
    const int64_t hd_off = static_cast<int64_t>(bh % static_cast<uint32_t>(a.heads)) * a.head_dim;
    const float* qrow = a.q + (b * a.q_len + qi) * a.ld_q + hd_off;
    const float* kb = a.k + b * a.kv_len * a.ld_kv + hd_off;
    const float* vb = a.v + b * a.kv_len * a.ld_kv + hd_off;
    float q[CH], acc[CH];
#pragma unroll
    for (int c = 0; c < CH; ++c) {
        const int d = lane + c * kWave;
        q[c] = d < a.head_dim ? qrow[d] * a.qscale : 0.f;
        acc[c] = 0.f;
    }
    const int64_t key_end = a.causal ? (qi + 1 < a.kv_len ? qi + 1 : a.kv_len) : a.kv_len;
    float m_run = -1e30f, l_run = 0.f;
    for (int64_t j = 0; j < key_end; ++j) {
        const float* krow = kb + j * a.ld_kv;
        const float* vrow = vb + j * a.ld_kv;
        float part = 0.f;
#pragma unroll
        for (int c = 0; c < CH; ++c) {
            const int d = lane + c * kWave;
            if (d < a.head_dim) part += q[c] * krow[d];
        }
        const float s = wave_sum(part);  // wave-uniform
        const float m_new = fmaxf(m_run, s);
        const float alpha = __builtin_amdgcn_exp2f(m_run - m_new);
        const float p = __builtin_amdgcn_exp2f(s - m_new);
        m_run = m_new;
        l_run = l_run * alpha + p;
#pragma unroll
        for (int c = 0; c < CH; ++c) {
            const int d = lane + c * kWave;
            acc[c] = acc[c] * alpha + (d < a.head_dim ? p * vrow[d] : 0.f);
        }
    }
    const float inv = 1.0f / (l_run + 1e-9f);
    float* orow = a.out + (b * a.q_len + qi) * a.ld_out + hd_off;
#pragma unroll
    for (int c = 0; c < CH; ++c) {
        const int d = lane + c * kWave;
        if (d < a.head_dim) orow[d] = acc[c] * inv;
    }
}

template <int CH>
int launch_generic(mimir_ctx* ctx, const AttnArgs& a, int64_t batch, int64_t heads) {
    const dim3 grid(static_cast<unsigned>(batch * heads),
                    static_cast<unsigned>((a.q_len + kGenericWaves - 1) / kGenericWaves));
    attention_fwd_generic<CH><<<grid, kGenericWaves * kWave, 0, ctx->stream>>>(a);
    return launched(ctx, "attention_fwd_generic");
}

template <int DP, int WAVES>
int launch(mimir_ctx* ctx, AttnArgs a, int64_t bh, bool vec) {
    constexpr int kThreads = WAVES * kWave;
    a.n_qblocks = (a.q_len + kQPerWave * WAVES - 1) / (kQPerWave * WAVES);
    const int64_t blocks = bh * a.n_qblocks;
    MIMIR_REQUIRE(ctx, dispatch_fits(blocks * a.splits, kThreads), "attention: grid of %lld workgroups exceeds the limit",
                  (long long)blocks);
    a.total_blocks = static_cast<uint32_t>(blocks);
    const auto n = static_cast<unsigned>(blocks * a.splits);
    if (vec) attention_fwd_mfma<DP, WAVES, true><<<n, kThreads, 0, ctx->stream>>>(a);
    else attention_fwd_mfma<DP, WAVES, false><<<n, kThreads, 0, ctx->stream>>>(a);
    if (int st = launched(ctx, "attention_fwd_mfma")) return st;
    if (!a.part) return MIMIR_OK;
    const int64_t rows = bh * a.q_len;
    MIMIR_REQUIRE(ctx, dispatch_fits((rows + 3) / 4, 4 * kWave), "attention: grid exceeds the limit");
    attention_fwd_combine<<<static_cast<unsigned>((rows + 3) / 4), 4 * kWave, 0, ctx->stream>>>(a, kQPerWave * WAVES);
    return launched(ctx, "attention_fwd_combine");
}

// Splits of the keys: until the workgroups fill the GPU, with partial results
// within `floats`.  Only for 24 tiles and more: below that the combine costs
// what the shorter chains give.  Measured (1 / 2 / 4 splits, us): 16 heads x
// 1024 x 128 causal 106 / 86 / 70, 32 heads 107 / 101 / 112, 48 heads x 333 x
// 777 x 80 69 / 61 / 73, 8 heads x 40 x 1500 x 128 125 / 73 / 45 (8: 34); 64
// heads x 512 x 128 59 / 75 / 93, 8 heads x 300 x 64 20 / 23 / 21.
int64_t splits_for(const mimir_ctx* ctx, int64_t bh, int64_t q_len, int64_t kv_len, int64_t head_dim, int64_t floats) {
    const int64_t blocks = bh * ((q_len + 8 * kQPerWave - 1) / (8 * kQPerWave));
    const int64_t tiles = (kv_len + kKeyTile - 1) / kKeyTile;
    int64_t s = tiles >= 24 ? std::min<int64_t>(kSplitTarget / blocks, tiles / 4) : 1;
    if (ctx->tune.attn_splits > 0) s = ctx->tune.attn_splits;
    s = std::min(s, floats / (bh * q_len * (head_dim + 2)));
    return std::max<int64_t>(s, 1);
}

template <int DP>
int launch_mfma(mimir_ctx* ctx, const AttnArgs& a, int64_t bh, bool vec) {
    // Eight waves split a tile once for 256 queries; four keep more of the
    // GPU busy while one workgroup per CU holds all of them.  Measured on
    // MI355X (4 / 8 waves, us): 8 x 32 heads x 1024 x 128 causal 508 / 395,
    // 16 heads x 1024 x 128 causal 99 / 120, 16 x 2048 x 64 causal 107 / 134,
    // 96 x 333 x 777 x 80 136 / 78.  Few queries (40 against 1500 keys): the
    // tile's way in is the work, 142 / 122.
    const int64_t blocks4 = bh * ((a.q_len + 4 * kQPerWave - 1) / (4 * kQPerWave));
    int waves = a.splits == 1 && blocks4 <= 256 && a.q_len > 64 ? 4 : 8;
    // A grid holds twice the workgroups of four waves.
    if (!dispatch_fits(bh * ((a.q_len + 8 * kQPerWave - 1) / (8 * kQPerWave)) * a.splits, 8 * kWave)) waves = 4;
    if (ctx->tune.attn_waves == 4 || ctx->tune.attn_waves == 8) waves = ctx->tune.attn_waves;
    return waves == 4 ? launch<DP, 4>(ctx, a, bh, vec) : launch<DP, 8>(ctx, a, bh, vec);
}

// Whether heads and strides are what the matrix-core kernels take: the tiles'
// buffer descriptors span 32 rows of ld floats, below 2^31 bytes.
bool mfma_takes(int64_t head_dim, int64_t ld) { return head_dim <= 128 && ld < (int64_t{1} << 31) / (4 * kKeyTile); }

int launch_any(mimir_ctx* ctx, const AttnArgs& a, int64_t bh, bool vec) {
    if (a.head_dim <= 32) return launch_mfma<32>(ctx, a, bh, vec);
    if (a.head_dim <= 64) return launch_mfma<64>(ctx, a, bh, vec);
    if (a.head_dim <= 96) return launch_mfma<96>(ctx, a, bh, vec);
    return launch_mfma<128>(ctx, a, bh, vec);
}

}  // namespace

extern "C" {

int mimir_attention_fwd(mimir_ctx* ctx, const float* q, int64_t ld_q, const float* k, const float* v,
                        int64_t ld_kv, float* out, int64_t ld_out, int64_t batch, int64_t q_len,
                        int64_t kv_len, int64_t heads, int64_t head_dim, float scale, int causal) {
    if (!ctx) return MIMIR_EINVAL;
    MIMIR_REQUIRE(ctx, batch >= 0 && q_len >= 0 && kv_len >= 0 && heads >= 1 && head_dim >= 1,
                  "attention: invalid shape (batch=%lld q_len=%lld kv_len=%lld heads=%lld head_dim=%lld)",
                  (long long)batch, (long long)q_len, (long long)kv_len, (long long)heads, (long long)head_dim);
    MIMIR_REQUIRE(ctx, head_dim <= 2048, "attention: head_dim %lld > 2048 is not supported", (long long)head_dim);
    const int64_t width = heads * head_dim;
    MIMIR_REQUIRE(ctx, ld_q >= width && ld_kv >= width && ld_out >= width,
                  "attention: row strides (%lld, %lld, %lld) below heads * head_dim = %lld", (long long)ld_q,
                  (long long)ld_kv, (long long)ld_out, (long long)width);
    MIMIR_REQUIRE(ctx, q_len < (int64_t{1} << 30) && kv_len < (int64_t{1} << 30) && heads < (int64_t{1} << 30),
                  "attention: sequence or head count too large");
    MIMIR_REQUIRE(ctx, std::isfinite(scale), "attention: scale must be finite");
    if (batch == 0 || q_len == 0) return MIMIR_OK;
    MIMIR_REQUIRE(ctx, q && out && (kv_len == 0 || (k && v)), "attention: null pointer");
    if (int st = enter(ctx)) return st;
    AttnArgs a{};
    a.q = q;
    a.k = kv_len ? k : q;  // never read when kv_len == 0
    a.v = kv_len ? v : q;
    a.out = out;
    a.ld_q = ld_q;
    a.ld_kv = ld_kv;
    a.ld_out = ld_out;
    a.q_len = static_cast<int32_t>(q_len);
    a.kv_len = static_cast<int32_t>(kv_len);
    a.heads = static_cast<int32_t>(heads);
    a.head_dim = static_cast<int32_t>(head_dim);
    a.qscale = scale * kLog2e;
    a.causal = causal ? 1 : 0;
    const bool vec = head_dim % 4 == 0 && ld_q % 4 == 0 && ld_kv % 4 == 0 && ld_out % 4 == 0 && aligned16(q) &&
                     aligned16(a.k) && aligned16(a.v) && aligned16(out);
    // Few queries: each key row is read once by vector code, where the
    // matrix-core kernel would use one of its waves (attention_decode.hip).
    if (attention_decode_applies(batch * heads, q_len, kv_len, head_dim, a.causal))
        return attention_decode_launch(ctx, q, ld_q, a.k, a.v, ld_kv, out, ld_out, batch, q_len, kv_len, heads, head_dim,
                                       a.qscale, vec);
    if (mfma_takes(head_dim, ld_kv)) {
        a.splits = static_cast<int32_t>(splits_for(ctx, batch * heads, q_len, kv_len, head_dim, kFixedWorkBytes / 4));
        a.part = a.splits > 1 ? fixed_work(ctx) : nullptr;
        if (!a.part) a.splits = 1;
        return launch_any(ctx, a, batch * heads, vec);
    }
    MIMIR_REQUIRE(ctx, dispatch_fits(batch * heads, kGenericWaves * kWave) && (q_len + kGenericWaves - 1) / kGenericWaves <= 65535,
                  "attention: grid exceeds the limit of the wide-head kernel");
    if (head_dim <= 256) return launch_generic<4>(ctx, a, batch, heads);
    if (head_dim <= 512) return launch_generic<8>(ctx, a, batch, heads);
    if (head_dim <= 1024) return launch_generic<16>(ctx, a, batch, heads);
    return launch_generic<32>(ctx, a, batch, heads);
}

// The attention layers (Model.cpp:5904-5934, 5936-5990): the projections as
// fp32 products (gemm.hip), the fused core between them on the projection's
// output in place (no split copies).  Scratch: the projections' outputs and
// the attended heads, reused in stream order.
int mimir_self_attention_fwd(mimir_ctx* ctx, const float* input, int64_t seq_len, int64_t embed_dim,
                             int64_t num_heads, int causal, const float* weights, int64_t weights_len, float* out) {
    if (!ctx) return MIMIR_EINVAL;
    MIMIR_REQUIRE(ctx, embed_dim >= 1 && num_heads >= 1 && embed_dim % num_heads == 0,
                  "SelfAttention: embed_dim must be divisible by num_heads");
    MIMIR_REQUIRE(ctx, seq_len >= 0, "SelfAttention: input size mismatch");
    const int64_t e = embed_dim;
    MIMIR_REQUIRE(ctx, weights_len >= 4 * e * e, "SelfAttention: weight block of %lld floats, %lld needed",
                  (long long)weights_len, (long long)(4 * e * e));
    MIMIR_REQUIRE(ctx, e / num_heads <= 2048, "attention: head_dim %lld > 2048 is not supported",
                  (long long)(e / num_heads));
    if (seq_len == 0) return MIMIR_OK;
    MIMIR_REQUIRE(ctx, input && weights && out, "SelfAttention: null pointer");
    MIMIR_ENTER(ctx);
    void* s = nullptr;
    if (int st = ensure_scratch(ctx, sizeof(float) * static_cast<size_t>(seq_len) * 4 * e, &s)) return st;
    float* qkv = static_cast<float*>(s);  // [seq, 3E]: Q | K | V
    float* att = qkv + seq_len * 3 * e;   // [seq, E]
    const int64_t hd = e / num_heads;
    if (int st = gemm_f32(ctx, seq_len, 3 * e, e, input, e, weights, 3 * e, qkv, 3 * e)) return st;  // :1027-1028
    if (int st = mimir_attention_fwd(ctx, qkv, 3 * e, qkv + e, qkv + 2 * e, 3 * e, att, e, 1, seq_len, seq_len,
                                     num_heads, hd, 1.0f / std::sqrt(static_cast<float>(hd)), causal))
        return st;
    return gemm_f32(ctx, seq_len, e, e, att, e, weights + 3 * e * e, e, out, e);  // :1093-1094
}

int mimir_cross_attention_fwd(mimir_ctx* ctx, const float* query_input, int64_t query_len, const float* kv_input,
                              int64_t kv_len, int64_t embed_dim, int64_t num_heads, int causal,
                              const float* weights, int64_t weights_len, float* out) {
    if (!ctx) return MIMIR_EINVAL;
    MIMIR_REQUIRE(ctx, embed_dim >= 1 && num_heads >= 1 && embed_dim % num_heads == 0,
                  "CrossAttention: embed_dim must be divisible by num_heads");
    MIMIR_REQUIRE(ctx, query_len > 0 && kv_len > 0, "CrossAttention: invalid dimensions");
    const int64_t e = embed_dim;
    MIMIR_REQUIRE(ctx, weights_len >= 4 * e * e, "CrossAttention: weight block of %lld floats, %lld needed",
                  (long long)weights_len, (long long)(4 * e * e));
    MIMIR_REQUIRE(ctx, e / num_heads <= 2048, "attention: head_dim %lld > 2048 is not supported",
                  (long long)(e / num_heads));
    MIMIR_REQUIRE(ctx, query_input && kv_input && weights && out, "CrossAttention: null pointer");
    MIMIR_ENTER(ctx);
    void* s = nullptr;
    if (int st = ensure_scratch(ctx, sizeof(float) * static_cast<size_t>(2 * query_len + 2 * kv_len) * e, &s))
        return st;
    float* qp = static_cast<float*>(s);  // [query_len, E]
    float* kv = qp + query_len * e;      // [kv_len, 2E]: K | V
    float* att = kv + kv_len * 2 * e;    // [query_len, E]
    const int64_t hd = e / num_heads;
    if (int st = gemm_f32(ctx, query_len, e, e, query_input, e, weights, e, qp, e)) return st;  // :1146-1147
    if (int st = gemm_f32(ctx, kv_len, 2 * e, e, kv_input, e, weights + e * e, 2 * e, kv, 2 * e)) return st;
    if (int st = mimir_attention_fwd(ctx, qp, e, kv, kv + e, 2 * e, att, e, 1, query_len, kv_len, num_heads, hd,
                                     1.0f / std::sqrt(static_cast<float>(hd)), causal))
        return st;
    return gemm_f32(ctx, query_len, e, e, att, e, weights + 3 * e * e, e, out, e);  // :1213-1214
}

}  // extern "C"
