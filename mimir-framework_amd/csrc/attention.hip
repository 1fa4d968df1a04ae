// attention.hip -- the attention core softmax(Q K^T * scale) V with the
// softmax fused between the two products, fp32 on the gfx950 matrix cores.
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
// MFMAs.  Measured there 400 us = 172 TFLOP/s of fp32 work, against 627 us on
// the fp32 MFMAs (157 TFLOP/s peak); 16 heads x 1024 x 128 99 / 152 us, 96 heads
// x 333 x 777 x 80 77 / 213 us.  Within noise of that: two accumulators in
// turns, LDS reads ordered ahead of the MFMAs, the split interleaved with them,
// raised priority for half the waves; four waves with two workgroups' worth of
// LDS are slower (the tile is split twice as often).
#include "common.hpp"
#include "internal.hpp"
#include "split.hpp"

#include <math.h>

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
};

// Workgroup -> (sequence * heads + head, query block): see the file comment.
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

// One query by one wave in plain fp32, the head's dimensions spread over the
// lanes (CH per lane, lane + 64 c): each score a DPP wave sum, the same online
// softmax and the same division by (sum + 1e-9).
template <int CH>
__device__ __forceinline__ void one_query(const float* qrow, const float* kb, const float* vb, float* orow,
                                          int64_t ld_kv, int64_t keys, int head_dim, float qscale) {
    const int lane = threadIdx.x % kWave;
    float q[CH], acc[CH];
#pragma unroll
    for (int c = 0; c < CH; ++c) {
        const int d = lane + c * kWave;
        q[c] = d < head_dim ? qrow[d] * qscale : 0.f;
        acc[c] = 0.f;
    }
    float m_run = -1e30f, l_run = 0.f;
    for (int64_t j = 0; j < keys; ++j) {
        const float* krow = kb + j * ld_kv;
        const float* vrow = vb + j * ld_kv;
        float part = 0.f;
#pragma unroll
        for (int c = 0; c < CH; ++c) {
            const int d = lane + c * kWave;
            if (d < head_dim) part += q[c] * krow[d];
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
            acc[c] = acc[c] * alpha + (d < head_dim ? p * vrow[d] : 0.f);
        }
    }
    const float inv = 1.0f / (l_run + 1e-9f);
#pragma unroll
    for (int c = 0; c < CH; ++c) {
        const int d = lane + c * kWave;
        if (d < head_dim) orow[d] = acc[c] * inv;
    }
}

// A tile of 32 keys on its way from memory to LDS.  Items of eight values: K
// item = (key, eight dimensions), V item = (dimension, eight keys in the order
// of the file comment); 4 * DP of each, dealt to THREADS threads.  Loads go
// through a descriptor that starts at the tile's first row and ends after the
// sequence's last, so rows past kv_len read as zeros; columns are clamped into
// the head (past head_dim, Q is zero and the output is not stored).
// VEC: K moves in 16-byte loads (head_dim, the stride and the base pointer are
// 16-byte multiples).
template <int DP, int THREADS, bool VEC>
struct KvTile {
    static constexpr int kKeyBytes = 2 * DP + 16, kDimBytes = 2 * kKeyTile + 16;
    static constexpr int kKPlane = kKeyTile * kKeyBytes, kVPlane = DP * kDimBytes;
    static constexpr int kBytes = 3 * (kKPlane + kVPlane);
    static constexpr int kKind = 4 * DP;  // items of each kind
    static constexpr int kItems = (kKind + THREADS - 1) / THREADS;
    static constexpr int kSpare = kItems * THREADS - kKind;  // threads without an item of one kind
    float k[kItems][8], v[kItems][8];
    uint32_t koff[kItems], voff[kItems];  // byte offsets of an item's first element
    int32_t kstep[kItems];                // VEC: bytes from the first four to the second four of a K item
    uint32_t ld4;

    // Where the items do not fill the threads, the first ones take K and the
    // last ones V.
    static __device__ __forceinline__ int k_item(int j) { return static_cast<int>(threadIdx.x) + j * THREADS; }
    static __device__ __forceinline__ int v_item(int j) { return k_item(j) - kSpare; }
    static __device__ __forceinline__ int wave_start() {
        return __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x)) & ~(kWave - 1);
    }
    static __device__ __forceinline__ bool has_k(int j) { return kSpare == 0 || wave_start() + j * THREADS < kKind; }
    static __device__ __forceinline__ bool has_v(int j) { return kSpare == 0 || wave_start() + j * THREADS >= kSpare; }

    __device__ __forceinline__ void init(int64_t ld, int head_dim) {
        ld4 = static_cast<uint32_t>(ld * 4);
#pragma unroll
        for (int j = 0; j < kItems; ++j) {
            const int ki = min(k_item(j), kKind - 1), key = ki / (DP / 8), d = 8 * (ki % (DP / 8));
            if constexpr (VEC) {
                koff[j] = key * ld4 + 4 * min(d, head_dim - 4);
                kstep[j] = 4 * (min(d + 4, head_dim - 4) - min(d, head_dim - 4));
            } else {
                koff[j] = key * ld4 + 4 * d;
            }
            const int vi = max(v_item(j), 0), group = vi / DP;
            voff[j] = 4 * min(vi % DP, head_dim - 1) + (16 * (group / 2) + 4 * (group % 2)) * ld4;
        }
    }
    __device__ __forceinline__ void load(const float* kbase, const float* vbase, int tile, int64_t ld, int kv_len,
                                         int head_dim) {
        const int64_t first = static_cast<int64_t>(tile) * kKeyTile * ld;
        const int rows = min(kKeyTile, kv_len - tile * kKeyTile);
        // The last row ends with the head, not with the stride.
        const int bytes = static_cast<int>((rows - 1) * ld4 + 4 * head_dim);
        const __amdgpu_buffer_rsrc_t rk = buffer_of(kbase + first, bytes), rv = buffer_of(vbase + first, bytes);
#pragma unroll
        for (int j = 0; j < kItems; ++j) {
            if (has_k(j)) {
                if constexpr (VEC) {
                    const f4 a = buffer_f4(rk, koff[j]), b = buffer_f4(rk, koff[j] + kstep[j]);
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        k[j][e] = a[e];
                        k[j][4 + e] = b[e];
                    }
                } else {
                    const int d = 8 * (k_item(j) % (DP / 8));
#pragma unroll
                    for (int e = 0; e < 8; ++e) k[j][e] = buffer_f1(rk, koff[j] + 4 * (min(d + e, head_dim - 1) - d));
                }
            }
            if (has_v(j)) {
#pragma unroll
                for (int e = 0; e < 8; ++e) v[j][e] = buffer_f1(rv, voff[j] + ((e & 3) + 8 * (e >> 2)) * ld4);
            }
        }
    }
    __device__ __forceinline__ void stash(char* lds) const {
#pragma unroll
        for (int j = 0; j < kItems; ++j) {
            if (has_k(j)) {
                const int id = k_item(j);
                char* p = lds + id / (DP / 8) * kKeyBytes + id % (DP / 8) * 16;
                const Split8 s = split8(k[j]);
                *reinterpret_cast<u4*>(p) = s.h;
                *reinterpret_cast<u4*>(p + kKPlane) = s.m;
                *reinterpret_cast<u4*>(p + 2 * kKPlane) = s.l;
            }
            if (has_v(j)) {
                const int id = v_item(j);
                char* p = lds + 3 * kKPlane + id % DP * kDimBytes + id / DP * 16;
                const Split8 s = split8(v[j]);
                *reinterpret_cast<u4*>(p) = s.h;
                *reinterpret_cast<u4*>(p + kVPlane) = s.m;
                *reinterpret_cast<u4*>(p + 2 * kVPlane) = s.l;
            }
        }
    }
    // MFMA operands: dimensions 16 c + 8 hf .. + 7 of key li; the eight keys
    // (c, hf) of dimension 32 db + li.
    static __device__ __forceinline__ Split8 key_rows(const char* lds, int li, int hf, int c) {
        const char* p = lds + li * kKeyBytes + 32 * c + 16 * hf;
        return Split8{*reinterpret_cast<const u4*>(p), *reinterpret_cast<const u4*>(p + kKPlane),
                      *reinterpret_cast<const u4*>(p + 2 * kKPlane)};
    }
    static __device__ __forceinline__ Split8 value_cols(const char* lds, int li, int hf, int db, int c) {
        const char* p = lds + 3 * kKPlane + (32 * db + li) * kDimBytes + 32 * c + 16 * hf;
        return Split8{*reinterpret_cast<const u4*>(p), *reinterpret_cast<const u4*>(p + kVPlane),
                      *reinterpret_cast<const u4*>(p + 2 * kVPlane)};
    }
};

template <int DP, int WAVES, bool VEC>
__global__ __launch_bounds__(WAVES * kWave, WAVES > 4 ? 2 : 1) void attention_fwd_mfma(AttnArgs a) {
    using Tile = KvTile<DP, WAVES * kWave, VEC>;
    constexpr int kC = DP / 16;   // MFMA steps of a score
    constexpr int kDb = DP / 32;  // output dimension blocks
    __shared__ __attribute__((aligned(16))) char lds[2 * Tile::kBytes];

    uint32_t bh;
    int qb;
    block_coords(a, blockIdx.x, &bh, &qb);
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
    int key_end = a.kv_len;
    int wave_key_end = a.kv_len;
    if (a.causal) {
        key_end = min(key_end, min(q0 + kQPerWave * WAVES, a.q_len));
        wave_key_end = min(wave_key_end, min(qw0 + kQPerWave, a.q_len));
    }
    if (qw0 >= a.q_len) wave_key_end = 0;
    const int n_tiles = (key_end + kKeyTile - 1) / kKeyTile;
    const int wave_tiles = (wave_key_end + kKeyTile - 1) / kKeyTile;
    // Keys of this lane's query: the rest of its last tile is masked
    // (causal: key > query; all: key >= kv_len).
    const int lane_key_end = min(a.kv_len, a.causal ? my_q + 1 : a.kv_len);

    Tile tile;
    tile.init(a.ld_kv, a.head_dim);
    if (n_tiles > 0) tile.load(kbase, vbase, 0, a.ld_kv, a.kv_len, a.head_dim);

    // This lane's Q values, times scale*log2(e), zero past head_dim.
    Split8 q[kC];
    {
        const float* qrow = qbase + static_cast<int64_t>(min(my_q, a.q_len - 1)) * a.ld_q;
#pragma unroll
        for (int c = 0; c < kC; ++c) {
            float x[8];
#pragma unroll
            for (int v = 0; v < 2; ++v) {
                const int d = 16 * c + 8 * hf + 4 * v;
                if constexpr (VEC) {
                    const f4 t = d < a.head_dim ? *reinterpret_cast<const f4*>(qrow + d) : f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                    for (int e = 0; e < 4; ++e) x[4 * v + e] = t[e] * a.qscale;
                } else {
#pragma unroll
                    for (int e = 0; e < 4; ++e) x[4 * v + e] = d + e < a.head_dim ? qrow[d + e] * a.qscale : 0.f;
                }
            }
            q[c] = split8(x);
        }
    }
    f16v o[kDb];
#pragma unroll
    for (int d = 0; d < kDb; ++d) o[d] = f16v{};
    float m_run = -1e30f;  // running max (base-2 units); the reference starts at -1e30 (LayerOps.hpp:1052)
    float l_run = 0.f;     // this half's share of the running sum

    if (n_tiles > 0) tile.stash(lds);
    if (n_tiles > 0) tile.load(kbase, vbase, min(1, n_tiles - 1), a.ld_kv, a.kv_len, a.head_dim);
    __syncthreads();

    for (int t = 0; t < n_tiles; ++t) {
        const char* cur = lds + (t & 1) * Tile::kBytes;
        char* const next = lds + ((t + 1) & 1) * Tile::kBytes;
        if (t < wave_tiles) {
            f16v s = f16v{};
            __builtin_amdgcn_s_setprio(1);
#pragma unroll
            for (int c = 0; c < kC; ++c) s = mfma_split(Tile::key_rows(cur, li, hf, c), q[c], s);
            // Past the last tile the stash rewrites a buffer that is not read
            // again, and the load repeats the last tile.
            tile.stash(next);
            
            __builtin_amdgcn_s_setprio(0);
            tile.load(kbase, vbase, min(t + 2, n_tiles - 1), a.ld_kv, a.kv_len, a.head_dim);
            if ((t + 1) * kKeyTile > a.kv_len || (a.causal && (t + 1) * kKeyTile - 1 > qw0)) {
                const int lim = lane_key_end - t * kKeyTile - 4 * hf;
#pragma unroll
                for (int r = 0; r < 16; ++r) s[r] = 8 * (r / 4) + (r % 4) < lim ? s[r] : -INFINITY;
            }
            float tmax = fmaxf(fmaxf(fmaxf(s[0], s[1]), fmaxf(s[2], s[3])), fmaxf(fmaxf(s[4], s[5]), fmaxf(s[6], s[7])));
            tmax = fmaxf(tmax, fmaxf(fmaxf(fmaxf(s[8], s[9]), fmaxf(s[10], s[11])),
                                     fmaxf(fmaxf(s[12], s[13]), fmaxf(s[14], s[15]))));
            tmax = fmaxf(tmax, __shfl_xor(tmax, 32));
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
                for (int d = 0; d < kDb; ++d) o[d] = mfma_split(Tile::value_cols(cur, li, hf, d, c), p, o[d]);
            }
            
            __builtin_amdgcn_s_setprio(0);
        } else {
            tile.stash(next);
            tile.load(kbase, vbase, min(t + 2, n_tiles - 1), a.ld_kv, a.kv_len, a.head_dim);
        }
        __syncthreads();
    }

    // out = O / (sum + 1e-9) (LayerOps.hpp:1076-1079).
    const float l_tot = l_run + __shfl_xor(l_run, 32);
    const float inv = 1.0f / (l_tot + 1e-9f);
    float check = l_tot - l_tot;
    float* orow = obase + static_cast<int64_t>(min(my_q, a.q_len - 1)) * a.ld_out;
#pragma unroll
    for (int d = 0; d < kDb; ++d) {
#pragma unroll
        for (int r = 0; r < 16; r += 4) {
            const int d0 = 32 * d + 8 * (r / 4) + 4 * hf;
            const f4 val{o[d][r] * inv, o[d][r + 1] * inv, o[d][r + 2] * inv, o[d][r + 3] * inv};
#pragma unroll
            for (int e = 0; e < 4; ++e) check += val[e] - val[e];
            if (my_q >= a.q_len) continue;
            if constexpr (VEC) {
                if (d0 < a.head_dim) *reinterpret_cast<f4*>(orow + d0) = val;
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (d0 + e < a.head_dim) orow[d0 + e] = val[e];
            }
        }
    }
    // Queries that came out NaN or infinite, again in fp32: their operands
    // may have had no bf16 split (split.hpp).
    uint64_t redo = __ballot(check != check && my_q < a.q_len);
    redo = (redo | redo >> 32) & 0xffffffffu;
    while (redo) {
        const int64_t i = qw0 + __builtin_ctzll(redo);
        redo &= redo - 1;
        one_query<(DP + kWave - 1) / kWave>(qbase + i * a.ld_q, kbase, vbase, obase + i * a.ld_out, a.ld_kv,
                                            a.causal ? min(static_cast<int64_t>(a.kv_len), i + 1) : a.kv_len, a.head_dim,
                                            a.qscale);
    }
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
    const int64_t qi = static_cast<int64_t>(blockIdx.y) * kGenericWaves + threadIdx.x / kWave;
    if (qi >= a.q_len) return;  // whole waves leave: no barrier below
    const uint32_t bh = blockIdx.x;
    const int64_t b = bh / static_cast<uint32_t>(a.heads);
    const int64_t hd_off = static_cast<int64_t>(bh % static_cast<uint32_t>(a.heads)) * a.head_dim;
    one_query<CH>(a.q + (b * a.q_len + qi) * a.ld_q + hd_off, a.k + b * a.kv_len * a.ld_kv + hd_off,
                  a.v + b * a.kv_len * a.ld_kv + hd_off, a.out + (b * a.q_len + qi) * a.ld_out + hd_off, a.ld_kv,
                  a.causal ? (qi + 1 < a.kv_len ? qi + 1 : a.kv_len) : a.kv_len, a.head_dim, a.qscale);
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
    MIMIR_REQUIRE(ctx, dispatch_fits(blocks, kThreads), "attention: grid of %lld workgroups exceeds the limit",
                  (long long)blocks);
    a.total_blocks = static_cast<uint32_t>(blocks);
    if (vec) attention_fwd_mfma<DP, WAVES, true><<<a.total_blocks, kThreads, 0, ctx->stream>>>(a);
    else attention_fwd_mfma<DP, WAVES, false><<<a.total_blocks, kThreads, 0, ctx->stream>>>(a);
    return launched(ctx, "attention_fwd_mfma");
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
    int waves = blocks4 <= 256 && a.q_len > 64 ? 4 : 8;
    if (ctx->tune.attn_waves == 4 || ctx->tune.attn_waves == 8) waves = ctx->tune.attn_waves;
    return waves == 4 ? launch<DP, 4>(ctx, a, bh, vec) : launch<DP, 8>(ctx, a, bh, vec);
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
    AttnArgs a;
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
    a.n_qblocks = 0;
    a.total_blocks = 0;
    a.qscale = scale * kLog2e;
    a.causal = causal ? 1 : 0;
    const bool vec = head_dim % 4 == 0 && ld_q % 4 == 0 && ld_kv % 4 == 0 && ld_out % 4 == 0 && aligned16(q) &&
                     aligned16(a.k) && aligned16(a.v) && aligned16(out);
    // Few queries: each key row is read once by vector code, where the
    // matrix-core kernel would use one of its waves (attention_decode.hip).
    if (attention_decode_applies(q_len, kv_len, head_dim, a.causal))
        return attention_decode_launch(ctx, q, ld_q, a.k, a.v, ld_kv, out, ld_out, batch, q_len, kv_len, heads, head_dim,
                                       a.qscale, vec);
    // The tile's buffer descriptors span 32 rows of ld_kv floats: below 2^31
    // bytes, or the wide-head kernel.
    if (ld_kv < (int64_t{1} << 31) / (4 * kKeyTile)) {
        if (head_dim <= 32) return launch_mfma<32>(ctx, a, batch * heads, vec);
        if (head_dim <= 64) return launch_mfma<64>(ctx, a, batch * heads, vec);
        if (head_dim <= 96) return launch_mfma<96>(ctx, a, batch * heads, vec);
        if (head_dim <= 128) return launch_mfma<128>(ctx, a, batch * heads, vec);
    }
    MIMIR_REQUIRE(ctx, dispatch_fits(batch * heads, kGenericWaves * kWave) && (q_len + kGenericWaves - 1) / kGenericWaves <= 65535,
                  "attention: grid exceeds the limit of the wide-head kernel");
    if (head_dim <= 256) return launch_generic<4>(ctx, a, batch, heads);
    if (head_dim <= 512) return launch_generic<8>(ctx, a, batch, heads);
    if (head_dim <= 1024) return launch_generic<16>(ctx, a, batch, heads);
    return launch_generic<32>(ctx, a, batch, heads);
}

// The attention layers (Model.cpp:5904-5934, 5936-5990): the projections as
// library GEMMs (gemm.hip), the fused core between them on the projection's
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
