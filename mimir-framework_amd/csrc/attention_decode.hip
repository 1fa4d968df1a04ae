// attention_decode.hip -- the attention core for a few queries per sequence
// against many keys (a decoding step over cached keys and values), the same
// softmax(Q K^T * scale) V as attention.hip (LayerOps.hpp:1045-1089).
//
// Bound by HBM: every key and value row is read once and used for NQ dot
// products of head_dim.  A group of LPK lanes owns a key at a time and holds
// NV 16-byte vectors of its row per lane, so a load instruction of the wave
// covers whole 64-byte lines of 64 / LPK rows; a group keeps the running max,
// sum and output of the keys it saw (fp32 vector code: no matrix core, no
// LDS in the loop) and reads kKeys rows of K and V ahead of their use.  The
// groups meet once, at the end: by lane exchanges in the wave, through LDS in
// the workgroup, and, when a (sequence, head) is dealt to several workgroups
// because there are too few of them to fill the GPU, through the context's
// workspace and a second small kernel.
//
// Measured on MI355X: 16 sequences x 32 heads, one query against 4000 keys of
// 128 (2.1 GB), 309 us = 6.8 TB/s, the rate of a large copy; the kernel for
// whole prompts (a wave of queries per workgroup, three of four waves idle)
// took 580 us there, 1118 us for one sequence of 8 heads and 8000 keys (here
// 37 us), 82 us for 48 heads of 64 and 1000 keys (12 us).  Eight queries read
// the rows twice (128 heads x 4096 keys: 174 us, against 577 us).
#include "common.hpp"
#include "internal.hpp"

#include <math.h>

#include <algorithm>

using namespace mimir;

namespace {

constexpr int kThreads = 256;
constexpr int kWaves = kThreads / kWave;
constexpr int kKeys = 4;  // rows of K and of V in flight per group
constexpr int kMaxDim = 128;

struct DecodeArgs {
    const float* q;
    const float* k;
    const float* v;
    float* out;
    float* part;  // [workgroup's split][query][2 + head_dim], null: one split
    int64_t ld_q, ld_kv, ld_out;
    int32_t q_len, kv_len, heads, head_dim;
    int32_t q_blocks;        // ceil(q_len / NQ)
    int32_t splits, span;    // workgroups per (sequence, head, query block), keys of each
    float qscale;            // scale * log2(e)
};

// NV vectors of one row: floats 4 (lane + LPK i) .. + 3, or, !VEC, float
// lane + LPK e of the row; past head_dim zero.
template <int LPK, int NV, bool VEC>
__device__ __forceinline__ void row_load(const float* row, int lane, int head_dim, f4* x) {
#pragma unroll
    for (int i = 0; i < NV; ++i) {
        if constexpr (VEC) {
            const int d = 4 * (lane + LPK * i);
            x[i] = d < head_dim ? __builtin_nontemporal_load(reinterpret_cast<const f4*>(row + d)) : f4{0.f, 0.f, 0.f, 0.f};
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int d = lane + LPK * (4 * i + e);
                x[i][e] = d < head_dim ? row[d] : 0.f;
            }
        }
    }
}

template <int LPK>
__device__ __forceinline__ float lanes_sum(float v) {
    v += dpp<kDppQuadXor1>(v);
    v += dpp<kDppQuadXor2>(v);
    if constexpr (LPK >= 8) v += dpp<kDppRowHalfMirror>(v);
    if constexpr (LPK >= 16) v += dpp<kDppRowMirror>(v);
    if constexpr (LPK >= 32) v += __shfl_xor(v, 16);
    return v;
}

// Running state of one query over some keys: output so far, max and sum.
template <int NV>
struct Partial {
    f4 acc[NV];
    float m, l;
    __device__ __forceinline__ void scale_to(float m_new) {
        const float f = __builtin_amdgcn_exp2f(m - m_new);
        m = m_new;
        l *= f;
#pragma unroll
        for (int i = 0; i < NV; ++i) acc[i] *= f;
    }
};

template <int LPK, int NV, int NQ, bool VEC>
__global__ __launch_bounds__(kThreads, 2) void attention_decode(DecodeArgs a) {
    constexpr int kGroups = kThreads / LPK;
    __shared__ float share[kWaves][NQ][4 * NV * LPK + 2];
    const int lane = threadIdx.x % LPK, group = threadIdx.x / LPK;
    const int wave = threadIdx.x / kWave;
    const uint32_t split = blockIdx.x % static_cast<uint32_t>(a.splits), rest = blockIdx.x / static_cast<uint32_t>(a.splits);
    const uint32_t qb = rest % static_cast<uint32_t>(a.q_blocks), bh = rest / static_cast<uint32_t>(a.q_blocks);
    const int64_t b = bh / static_cast<uint32_t>(a.heads);
    const int64_t hd_off = static_cast<int64_t>(bh % static_cast<uint32_t>(a.heads)) * a.head_dim;
    const int q0 = static_cast<int>(qb) * NQ, nq = min(NQ, a.q_len - q0);
    const float* kb = a.k + b * a.kv_len * a.ld_kv + hd_off;
    const float* vb = a.v + b * a.kv_len * a.ld_kv + hd_off;
    const int first = static_cast<int>(split) * a.span;  // keys of this workgroup
    const int last = min(a.kv_len, first + a.span);

    f4 q[NQ][NV];
    Partial<NV> st[NQ];
#pragma unroll
    for (int i = 0; i < NQ; ++i) {
        row_load<LPK, NV, VEC>(a.q + (b * a.q_len + min(q0 + i, a.q_len - 1)) * a.ld_q + hd_off, lane, a.head_dim, q[i]);
#pragma unroll
        for (int j = 0; j < NV; ++j) {
            q[i][j] *= a.qscale;
            st[i].acc[j] = f4{0.f, 0.f, 0.f, 0.f};
        }
        st[i].m = -1e30f;  // the reference's start (LayerOps.hpp:1052)
        st[i].l = 0.f;
    }

    auto step = [&](int key0, bool edge) {
        f4 k[kKeys][NV], v[kKeys][NV];
#pragma unroll
        for (int u = 0; u < kKeys; ++u) {
            const int key = key0 + u * kGroups + group;
            const int64_t off = static_cast<int64_t>(edge ? min(key, last - 1) : key) * a.ld_kv;
            row_load<LPK, NV, VEC>(kb + off, lane, a.head_dim, k[u]);
            row_load<LPK, NV, VEC>(vb + off, lane, a.head_dim, v[u]);
        }
        if (edge) {  // a key past the end adds nothing, whatever its row holds
#pragma unroll
            for (int u = 0; u < kKeys; ++u)
                if (key0 + u * kGroups + group >= last)
#pragma unroll
                    for (int j = 0; j < NV; ++j) v[u][j] = f4{0.f, 0.f, 0.f, 0.f};
        }
#pragma unroll
        for (int i = 0; i < NQ; ++i) {
            float s[kKeys];
#pragma unroll
            for (int u = 0; u < kKeys; ++u) {
                float d = 0.f;
#pragma unroll
                for (int j = 0; j < NV; ++j)
#pragma unroll
                    for (int e = 0; e < 4; ++e) d += q[i][j][e] * k[u][j][e];
                s[u] = lanes_sum<LPK>(d);
            }
            float m_new = st[i].m;
#pragma unroll
            for (int u = 0; u < kKeys; ++u) {
                if (edge && key0 + u * kGroups + group >= last) s[u] = -INFINITY;
                m_new = fmaxf(m_new, s[u]);
            }
            st[i].scale_to(m_new);
#pragma unroll
            for (int u = 0; u < kKeys; ++u) {
                const float p = __builtin_amdgcn_exp2f(s[u] - m_new);
                st[i].l += p;
#pragma unroll
                for (int j = 0; j < NV; ++j) st[i].acc[j] += p * v[u][j];
            }
        }
    };
    int key0 = first;
    for (; key0 + kKeys * kGroups <= last; key0 += kKeys * kGroups) step(key0, false);
    if (key0 < last) step(key0, true);

    // The groups of a wave (each ends with the sum over all of them), then
    // the waves of the workgroup.
#pragma unroll
    for (int i = 0; i < NQ; ++i) {
#pragma unroll
        for (int x = LPK; x < kWave; x *= 2) {
            const float m_new = fmaxf(st[i].m, __shfl_xor(st[i].m, x));
            st[i].scale_to(m_new);
            st[i].l += __shfl_xor(st[i].l, x);
#pragma unroll
            for (int j = 0; j < NV; ++j)
#pragma unroll
                for (int e = 0; e < 4; ++e) st[i].acc[j][e] += __shfl_xor(st[i].acc[j][e], x);
        }
        if (threadIdx.x % kWave < LPK) {
#pragma unroll
            for (int j = 0; j < NV; ++j)
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    share[wave][i][VEC ? 4 * (lane + LPK * j) + e : lane + LPK * (4 * j + e)] = st[i].acc[j][e];
            if (lane == 0) {
                share[wave][i][4 * NV * LPK] = st[i].m;
                share[wave][i][4 * NV * LPK + 1] = st[i].l;
            }
        }
    }
    __syncthreads();
    for (int x = threadIdx.x; x < nq * a.head_dim; x += kThreads) {
        const int i = x / a.head_dim, d = x % a.head_dim;
        float m = share[0][i][4 * NV * LPK];
#pragma unroll
        for (int w = 1; w < kWaves; ++w) m = fmaxf(m, share[w][i][4 * NV * LPK]);
        float l = 0.f, o = 0.f;
#pragma unroll
        for (int w = 0; w < kWaves; ++w) {
            const float f = __builtin_amdgcn_exp2f(share[w][i][4 * NV * LPK] - m);
            l += share[w][i][4 * NV * LPK + 1] * f;
            o += share[w][i][d] * f;
        }
        if (a.part) {
            float* p = a.part + ((static_cast<int64_t>(bh) * a.q_len + q0 + i) * a.splits + split) * (a.head_dim + 2);
            p[2 + d] = o;
            if (d == 0) {
                p[0] = m;
                p[1] = l;
            }
        } else {
            a.out[(b * a.q_len + q0 + i) * a.ld_out + hd_off + d] = o * (1.0f / (l + 1e-9f));
        }
    }
}

// The splits of one query of one head: one wave per row.
__global__ __launch_bounds__(kWave) void attention_decode_combine(DecodeArgs a) {
    const uint32_t bh = blockIdx.x / static_cast<uint32_t>(a.q_len);
    const int qi = static_cast<int>(blockIdx.x % static_cast<uint32_t>(a.q_len));
    const int w = a.head_dim + 2;
    const float* p = a.part + static_cast<int64_t>(blockIdx.x) * a.splits * w;
    float m = -1e30f;
    for (int s = 0; s < a.splits; ++s) m = fmaxf(m, p[s * w]);
    float l = 0.f;
    for (int s = 0; s < a.splits; ++s) l += p[s * w + 1] * __builtin_amdgcn_exp2f(p[s * w] - m);
    const float inv = 1.0f / (l + 1e-9f);
    const int64_t b = bh / static_cast<uint32_t>(a.heads);
    const int64_t hd_off = static_cast<int64_t>(bh % static_cast<uint32_t>(a.heads)) * a.head_dim;
    for (int d = threadIdx.x; d < a.head_dim; d += kWave) {
        float o = 0.f;
        for (int s = 0; s < a.splits; ++s) o += p[s * w + 2 + d] * __builtin_amdgcn_exp2f(p[s * w] - m);
        a.out[(b * a.q_len + qi) * a.ld_out + hd_off + d] = o * inv;
    }
}

template <int NQ>
void launch_nq(const DecodeArgs& a, unsigned grid, bool vec, hipStream_t s) {
    if (!vec) attention_decode<16, 2, NQ, false><<<grid, kThreads, 0, s>>>(a);
    else if (a.head_dim <= 32) attention_decode<8, 1, NQ, true><<<grid, kThreads, 0, s>>>(a);
    else if (a.head_dim <= 64) attention_decode<16, 1, NQ, true><<<grid, kThreads, 0, s>>>(a);
    else attention_decode<16, 2, NQ, true><<<grid, kThreads, 0, s>>>(a);
}

}  // namespace

namespace mimir {

// More (sequence, head) pairs than the grid holds at a workgroup per query go to
// the matrix-core kernel, which needs fewer workgroups.
bool attention_decode_applies(int64_t bh, int64_t q_len, int64_t kv_len, int64_t head_dim, bool causal) {
    return q_len <= kDecodeQueries && kv_len > 0 && head_dim <= kMaxDim && !causal && dispatch_fits(bh * q_len, kThreads);
}

int attention_decode_launch(mimir_ctx* ctx, const float* q, int64_t ld_q, const float* k, const float* v, int64_t ld_kv,
                            float* out, int64_t ld_out, int64_t batch, int64_t q_len, int64_t kv_len, int64_t heads,
                            int64_t head_dim, float qscale, bool vec) {
    const int nq = q_len >= 3 ? 4 : static_cast<int>(q_len);
    const int64_t q_blocks = (q_len + nq - 1) / nq, rows = batch * heads * q_blocks;
    // Two workgroups per CU fill the GPU: a (sequence, head) is dealt to more
    // only below that.  Measured (1 / 2 / 4 / 8 workgroups each, us): 512
    // pairs of 4000 keys 309 / 318 / 323 / 321, 128 of 4096 108 / 69 / 68 / 70,
    // 48 of 1000 18 / 15 / 12 / 13, 8 of 8000 168 / 95 / 55 / 38 (31: 37).
    constexpr int64_t kTarget = 512;
    int64_t splits = std::max<int64_t>(1, std::min<int64_t>(kTarget / std::max<int64_t>(rows, 1), (kv_len + 255) / 256));
    const int tuned = ctx->tune.decode_splits;
    if (tuned > 0) splits = std::min<int64_t>(tuned, kv_len);
    const int64_t floats = batch * heads * q_len * splits * (head_dim + 2);
    float* part = splits > 1 && floats * 4 <= static_cast<int64_t>(kFixedWorkBytes) ? fixed_work(ctx) : nullptr;
    if (!part) splits = 1;
    int64_t span = (kv_len + splits - 1) / splits;
    splits = (kv_len + span - 1) / span;
    MIMIR_REQUIRE(ctx, dispatch_fits(rows * splits, kThreads) && dispatch_fits(batch * heads * q_len, kWave),
                  "attention: grid of %lld workgroups exceeds the limit", (long long)(rows * splits));
    DecodeArgs a{q, k, v, out, splits > 1 ? part : nullptr, ld_q, ld_kv, ld_out,
                 static_cast<int32_t>(q_len), static_cast<int32_t>(kv_len), static_cast<int32_t>(heads),
                 static_cast<int32_t>(head_dim), static_cast<int32_t>(q_blocks), static_cast<int32_t>(splits),
                 static_cast<int32_t>(span), qscale};
    const auto grid = static_cast<unsigned>(rows * splits);
    if (nq == 1) launch_nq<1>(a, grid, vec, ctx->stream);
    else if (nq == 2) launch_nq<2>(a, grid, vec, ctx->stream);
    else launch_nq<4>(a, grid, vec, ctx->stream);
    if (int st = launched(ctx, "attention_decode")) return st;
    if (splits == 1) return MIMIR_OK;
    attention_decode_combine<<<static_cast<unsigned>(batch * heads * q_len), kWave, 0, ctx->stream>>>(a);
    return launched(ctx, "attention_decode_combine");
}

}  // namespace mimir
