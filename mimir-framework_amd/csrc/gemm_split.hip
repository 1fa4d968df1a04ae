// gemm_split.hip -- the fp32 matrix products around the attention core (the
// QKV and output projections of the attention layers, their gradients, and
// the per-head products of wide heads' backward) on the bf16 matrix cores, each
// fp32 operand held exactly as three bf16 terms (split.hpp): the small and the
// very large ones, where this is faster than the library (pick).
//
// The reference computes them with LayerOps::matmul (LayerOps.hpp:977-1001)
// and the loops of backward_self_attention (Model.cpp:6847-7062): row-major
// float32.
//
// gemm_tile: a workgroup of four waves computes a T x T tile of C (T = 128),
// each wave a quarter.  A step takes 32 of the contraction: the tile's rows of
// op(A) and columns of op(B) come to registers while the last step's products
// run, are split once per workgroup and stored to LDS as three bf16 planes
// [row][32], row stride 80 bytes (eight rows' 16-byte reads then touch every bank
// once).  An operand whose contraction index is contiguous in memory loads
// 16-byte vectors along it; the other kind loads eight rows of 64 consecutive
// columns.  Both put element k of the step in the same slot (slot 8 o + i holds
// k = 4 o + i % 4 + 16 (i / 4)), so any pair of layouts meets, and no operand is
// transposed in memory.  Bound by the power of the matrix cores: 4096^3 747 us =
// 184 TFLOP/s (the MFMAs busy 61% of the cycles at 1.7 GHz), against 919 us for
// the library's fp32 kernels at 98% of the fp32 matrix peak.  Two LDS buffers,
// raised priority around the MFMAs, and tiles of 128 x 64 and 64 x 64 for products
// between the two kinds (equal to the library alone, 10% slower within a layer)
// did not pay.
//
// gemm_strip: a 32 x 32 tile per workgroup, the contraction dealt to its waves in
// chunks of 16: 16 waves of two chunks in flight where the tiles number no more
// than the CUs, 4 waves of four chunks where there are more.  Operands go from
// memory straight to the wave's registers; the waves' partial tiles meet in LDS.
// One memory latency and one barrier, for products too small to fill the GPU with
// larger tiles: 128 x 768 x 256 4.8 us, where the library's best kernel takes 5.5
// us; the form of the library that a program using PyTorch has loaded takes 9 us
// there and 33 us for 128 x 256 x 256 (4.6 us here).
#include "internal.hpp"
#include "split.hpp"

#include <algorithm>
#include <type_traits>

using namespace mimir;

namespace {

constexpr int kStep = 32;       // contraction per step of gemm_tile
constexpr int kRowBytes = 80;   // LDS bytes of 32 bf16, padded
constexpr int kGemmThreads = 256;
constexpr int kXcds = 8;

struct GemmArgs {
    const float* a;
    const float* b;
    float* c;
    int64_t lda, ldb, ldc;              // row strides (floats)
    int64_t stride_a, stride_b, stride_c;
    int32_t m, n, k;
    uint32_t tiles_m, tiles_n, total;   // total = tiles_m * tiles_n * batch
    float alpha, beta;
};

struct TileAt {
    int32_t m0, n0;
    int64_t batch;
};

// Workgroup -> tile.  The hardware deals workgroups to the XCDs round-robin;
// each XCD takes a contiguous run of tiles (its operands stay in its L2), the
// tiles of a product column-fastest.
__device__ __forceinline__ bool tile_of(const GemmArgs& g, int t, TileAt* at) {
    const uint32_t per = (g.total + kXcds - 1) / kXcds;
    const uint32_t i = (blockIdx.x % kXcds) * per + blockIdx.x / kXcds;
    if (blockIdx.x / kXcds >= per || i >= g.total) return false;
    const uint32_t one = g.tiles_m * g.tiles_n;
    const uint32_t r = i % one;
    at->batch = i / one;
    at->m0 = static_cast<int32_t>(r / g.tiles_n) * t;
    at->n0 = static_cast<int32_t>(r % g.tiles_n) * t;
    return true;
}

// One operand's part of a step: R rows of op(A) (columns of op(B)) by 32.
// KC: the contraction is contiguous in memory.  VEC (KC only): 16-byte loads
// (base, stride and k multiples of four floats).
template <int R, bool KC, bool VEC>
struct Operand {
    static constexpr int kItems = R * 4 / kGemmThreads;  // slots of 8 per thread
    float x[kItems][8];
    uint32_t off[kItems];  // byte offset of the item's first element, kOutside past the last row
    uint32_t ld4;          // bytes between rows in memory
    int32_t oct[kItems];   // 4 * slot group: k = oct + i % 4 + 16 * (i / 4)
    const float* base;

    __device__ __forceinline__ void init(const float* p, int64_t ld, int64_t row0, int32_t rows) {
        ld4 = static_cast<uint32_t>(ld * 4);
        base = KC ? p + row0 * ld : p + row0;
#pragma unroll
        for (int j = 0; j < kItems; ++j) {
            const int id = threadIdx.x + j * kGemmThreads;
            const int row = KC ? id / 4 : id % R;
            oct[j] = 4 * (KC ? id % 4 : id / R);
            off[j] = row >= rows ? kOutside : KC ? row * ld4 + 4 * oct[j] : 4 * row + oct[j] * ld4;
        }
    }

    // Elements [k0, k0 + 32) of the contraction, `left` of them inside it.
    __device__ __forceinline__ void load(int64_t k0, int32_t left) {
        const __amdgpu_buffer_rsrc_t rs = buffer_of(base + (KC ? k0 : k0 * (ld4 / 4)), 0x7fffffff);
        if (left >= kStep) {
#pragma unroll
            for (int j = 0; j < kItems; ++j) fetch(rs, j, [](int) { return true; });
        } else {
#pragma unroll
            for (int j = 0; j < kItems; ++j)
                fetch(rs, j, [&](int i) { return oct[j] + (i & 3) + 16 * (i >> 2) < left; });
        }
    }
    template <class In>
    __device__ __forceinline__ void fetch(__amdgpu_buffer_rsrc_t rs, int j, In in) {
        if constexpr (KC && VEC) {
#pragma unroll
            for (int v = 0; v < 2; ++v) {
                const f4 t = buffer_f4(rs, in(4 * v) ? off[j] + 64 * v : kOutside);
#pragma unroll
                for (int e = 0; e < 4; ++e) x[j][4 * v + e] = t[e];
            }
        } else {
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const uint32_t k = (i & 3) + 16 * (i >> 2);
                // The step within the tile is uniform: it goes to the scalar offset.
                x[j][i] = __builtin_bit_cast(
                    float, __builtin_amdgcn_raw_buffer_load_b32(rs, in(i) ? off[j] : kOutside, KC ? 4 * k : k * ld4, 0));
            }
        }
    }

    // Split and store: planes h, m, l of [R][80 bytes].
    __device__ __forceinline__ void stash(char* lds) const {
#pragma unroll
        for (int j = 0; j < kItems; ++j) {
            const int id = threadIdx.x + j * kGemmThreads;
            const int row = KC ? id / 4 : id % R;
            char* p = lds + row * kRowBytes + 4 * oct[j];
            const Split8 s = split8(x[j]);
            *reinterpret_cast<u4*>(p) = s.h;
            *reinterpret_cast<u4*>(p + R * kRowBytes) = s.m;
            *reinterpret_cast<u4*>(p + 2 * R * kRowBytes) = s.l;
        }
    }
};

template <int R>
__device__ __forceinline__ Split8 operand_at(const char* lds, int row, int slot) {
    const char* p = lds + row * kRowBytes + slot * 16;
    return Split8{*reinterpret_cast<const u4*>(p), *reinterpret_cast<const u4*>(p + R * kRowBytes),
                  *reinterpret_cast<const u4*>(p + 2 * R * kRowBytes)};
}

__device__ __forceinline__ bool any_nan(const f16v& c) {
    float s = 0.0f;
#pragma unroll
    for (int r = 0; r < 16; ++r) s += c[r] - c[r];  // NaN for an infinity or a NaN
    return __any(s != s);
}

// A 32 x 32 block of the product with fp32 MFMAs, for operands that have no
// bf16 split (infinities, NaN, the largest floats): rare, unpipelined.
template <bool AK, bool BK>
__device__ __forceinline__ f16v block_f32(const GemmArgs& g, int64_t batch, int32_t m0, int32_t n0) {
    const int li = threadIdx.x % 32, hf = threadIdx.x % kWave / 32;
    const int64_t row = min(m0 + li, g.m - 1), col = min(n0 + li, g.n - 1);
    const float* a = g.a + batch * g.stride_a + (AK ? row * g.lda : row);
    const float* b = g.b + batch * g.stride_b + (BK ? col * g.ldb : col);
    f16v c = f16v{};
    for (int32_t k = hf; k < g.k + hf; k += 2) {
        const bool in = k < g.k;
        const int64_t kk = in ? k : 0;
        const float x = in ? a[AK ? kk : kk * g.lda] : 0.0f;
        const float y = in ? b[BK ? kk : kk * g.ldb] : 0.0f;
        c = __builtin_amdgcn_mfma_f32_32x32x2f32(x, y, c, 0, 0, 0);
    }
    return c;
}

// c = alpha acc + beta c for the wave's 32 x 32 block at (m0, n0).
__device__ __forceinline__ void store_block(const GemmArgs& g, int64_t batch, int32_t m0, int32_t n0, const f16v& acc) {
    const int li = threadIdx.x % 32, hf = threadIdx.x % kWave / 32;
    const int32_t col = n0 + li;
    if (col >= g.n) return;
    float* c = g.c + batch * g.stride_c + col;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        const int32_t row = m0 + 8 * (r / 4) + 4 * hf + r % 4;
        if (row >= g.m) continue;
        float* p = c + row * g.ldc;
        *p = g.beta == 0.0f ? g.alpha * acc[r] : g.alpha * acc[r] + g.beta * *p;
    }
}

template <bool AK, bool BK, bool VEC>
__global__ __launch_bounds__(kGemmThreads, 2) void gemm_tile(GemmArgs g) {
    constexpr int T = 128, kB = T / 64;  // 32 x 32 blocks per wave, each way
    __shared__ __attribute__((aligned(16))) char lds[6 * T * kRowBytes];
    char* const la = lds;
    char* const lb = lds + 3 * T * kRowBytes;
    TileAt at;
    if (!tile_of(g, T, &at)) return;
    const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
    const int li = lane % 32, hf = lane / 32;
    const int wm = wave / 2 * (T / 2), wn = wave % 2 * (T / 2);

    Operand<T, AK, VEC> oa;
    Operand<T, BK, VEC> ob;
    oa.init(g.a + at.batch * g.stride_a, g.lda, at.m0, g.m - at.m0);
    ob.init(g.b + at.batch * g.stride_b, g.ldb, at.n0, g.n - at.n0);
    f16v acc[kB][kB];
#pragma unroll
    for (int i = 0; i < kB; ++i)
#pragma unroll
        for (int j = 0; j < kB; ++j) acc[i][j] = f16v{};

    oa.load(0, g.k);
    ob.load(0, g.k);
    for (int32_t k0 = 0; k0 < g.k; k0 += kStep) {
        oa.stash(la);
        ob.stash(lb);
        __syncthreads();
        if (k0 + kStep < g.k) {
            oa.load(k0 + kStep, g.k - k0 - kStep);
            ob.load(k0 + kStep, g.k - k0 - kStep);
        }
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            Split8 a[kB], b[kB];
#pragma unroll
            for (int i = 0; i < kB; ++i) {
                a[i] = operand_at<T>(la, wm + 32 * i + li, 2 * c + hf);
                b[i] = operand_at<T>(lb, wn + 32 * i + li, 2 * c + hf);
            }
#pragma unroll
            for (int i = 0; i < kB; ++i)
#pragma unroll
                for (int j = 0; j < kB; ++j) acc[i][j] = mfma_split(a[i], b[j], acc[i][j]);
        }
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < kB; ++i)
#pragma unroll
        for (int j = 0; j < kB; ++j) {
            const int32_t m0 = at.m0 + wm + 32 * i, n0 = at.n0 + wn + 32 * j;
            if (any_nan(acc[i][j])) acc[i][j] = block_f32<AK, BK>(g, at.batch, m0, n0);
            store_block(g, at.batch, m0, n0, acc[i][j]);
        }
}

// A wave's operand for one chunk of 16 of the contraction, straight from
// memory: row (column) li of the tile, k = k0 + 8 hf + 0..7.
template <bool KC, bool VEC>
__device__ __forceinline__ void chunk_load(__amdgpu_buffer_rsrc_t rs, uint32_t row_off, uint32_t ld4, int32_t k,
                                           int32_t left, float* x) {
    if constexpr (KC && VEC) {
#pragma unroll
        for (int v = 0; v < 2; ++v) {
            const f4 t = buffer_f4(rs, 4 * v < left ? row_off + 4 * (k + 4 * v) : kOutside);
#pragma unroll
            for (int e = 0; e < 4; ++e) x[4 * v + e] = t[e];
        }
    } else {
#pragma unroll
        for (int i = 0; i < 8; ++i)
            x[i] = buffer_f1(rs, i < left ? row_off + (KC ? 4 * (k + i) : (k + i) * ld4) : kOutside);
    }
}

template <int WAVES, bool AK, bool BK, bool VEC>
__global__ __launch_bounds__(WAVES * kWave, WAVES == 16 ? 4 : 2) void gemm_strip(GemmArgs g) {
    constexpr int kWaves = WAVES;
    constexpr int kStripDepth = WAVES == 16 ? 2 : 4;  // chunks in flight per wave
    constexpr int kOwn = 16 / WAVES;                  // registers of the tile that a wave sums and stores
    __shared__ __attribute__((aligned(16))) float part[kWaves][16][kWave];
    TileAt at;
    if (!tile_of(g, 32, &at)) return;
    const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
    const int li = lane % 32, hf = lane / 32;
    const int32_t k_end = g.k;
    const uint32_t lda4 = static_cast<uint32_t>(g.lda * 4), ldb4 = static_cast<uint32_t>(g.ldb * 4);
    const __amdgpu_buffer_rsrc_t ra = buffer_of(g.a + at.batch * g.stride_a + (AK ? at.m0 * g.lda : at.m0), 0x7fffffff);
    const __amdgpu_buffer_rsrc_t rb = buffer_of(g.b + at.batch * g.stride_b + (BK ? at.n0 * g.ldb : at.n0), 0x7fffffff);
    const bool ina = at.m0 + li < g.m, inb = at.n0 + li < g.n;
    const uint32_t oa = AK ? li * lda4 : 4 * li, ob = BK ? li * ldb4 : 4 * li;

    f16v acc = f16v{};
    for (int32_t c0 = wave; 16 * c0 < k_end; c0 += kWaves * kStripDepth) {
        float x[kStripDepth][8], y[kStripDepth][8];
#pragma unroll
        for (int d = 0; d < kStripDepth; ++d) {
            const int32_t k = 16 * (c0 + kWaves * d) + 8 * hf;
            chunk_load<AK, VEC>(ra, oa, lda4, k, ina ? k_end - k : 0, x[d]);
            chunk_load<BK, VEC>(rb, ob, ldb4, k, inb ? k_end - k : 0, y[d]);
        }
#pragma unroll
        for (int d = 0; d < kStripDepth; ++d) acc = mfma_split(split8(x[d]), split8(y[d]), acc);
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) part[wave][r][lane] = acc[r];
    __syncthreads();
    // Wave w sums registers kOwn w .. of the partial tiles.
    float v[kOwn], bad = 0.0f;
#pragma unroll
    for (int e = 0; e < kOwn; ++e) {
        const int r = kOwn * wave + e;
        float t[4] = {};
#pragma unroll
        for (int w = 0; w < kWaves; ++w) t[w % 4] += part[w][r][lane];
        v[e] = (t[0] + t[1]) + (t[2] + t[3]);
        bad += v[e] - v[e];
    }
    if (__any(bad != bad)) {
        const f16v full = block_f32<AK, BK>(g, at.batch, at.m0, at.n0);
#pragma unroll
        for (int r = 0; r < 16; ++r)
            if (r / kOwn == wave) v[r % kOwn] = full[r];
    }
    const int32_t col = at.n0 + li;
    if (col >= g.n) return;
    float* c = g.c + at.batch * g.stride_c + col;
#pragma unroll
    for (int e = 0; e < kOwn; ++e) {
        const int r = kOwn * wave + e;
        const int32_t row = at.m0 + 8 * (r / 4) + 4 * hf + r % 4;
        if (row >= g.m) continue;
        float* p = c + row * g.ldc;
        *p = g.beta == 0.0f ? g.alpha * v[e] : g.alpha * v[e] + g.beta * *p;
    }
}

template <class F>
void with_layout(bool ak, bool bk, bool vec, F&& f) {
    using Y = std::true_type;
    using N = std::false_type;
    if (ak && bk) vec ? f(Y{}, Y{}, Y{}) : f(Y{}, Y{}, N{});
    else if (ak) vec ? f(Y{}, N{}, Y{}) : f(Y{}, N{}, N{});
    else if (bk) vec ? f(N{}, Y{}, Y{}) : f(N{}, Y{}, N{});
    else f(N{}, N{}, N{});  // no contiguous contraction: nothing to vectorise
}

}  // namespace

namespace mimir {

// What is taken.  Large: 1024 tiles of 128 x 128 or more.  Small: up to 256 tiles of
// 32 x 32 (one per CU) with a contraction up to 896, or up to 640 tiles and 256.  An
// operand contiguous along the contraction that cannot be read in 16-byte vectors
// (odd widths, unaligned) costs twice the time, so there the contraction is at most
// 256.  The rest goes to the library: as fast up to the large ones, and a layer's
// products run 10% faster there than with this file's tiles.  Measured on MI355X, us
// (gemm_strip or gemm_tile / library / the library in a PyTorch process): 300 x 512 x
// 512 5.5 / 6.3 / 9.0; 512^3 5.8 / 6.5 / 8.7; 100 x 1024 x 1024 7.9 / 6.9 / 8.7; 2048 x
// 768 x 256 14.1 / 10.8 / 16.7; 257 x 129 x 511, B transposed 11.6 / 5.4 / 9.1; 2048 x
// 3072 x 1024 87 / 95 / 92; 4096^3 747 / 919 / 920; 32 x 512 x 1024 x 128 35 / 45 / 45.
//
// Those limits are for the hipBLASLt that PyTorch brings (1.0), which takes 33 to 178
// us for many small products (256 x 256 x 777 117, 128 x 768 x 256 33).  From
// kGoodLibrary on (1.2, a program without PyTorch) the library is good at them, and
// the limits lie where a call here is no slower.  Calls in a row, us (here /
// library), and the kernels alone: 128 x 768 x 256 4.8 / 7.7 (5.0 / 4.9), 512^3 5.5 /
// 7.4 (5.9 / 6.8), 256 x 256 x 777, A transposed 7.5 / 7.3 (7.7 / 6.4): up to 512.  Both
// operands contiguous along the contraction (B transposed): 256 x 768 x 128 4.3 / 7.6
// (4.4 / 4.3), 512 x 512 x 768 9.1 / 7.4 (8.8 / 7.3): up to 128, and none of more than
// 256 tiles (777 x 768 x 256 8.5 / 7.4).  More than 256 tiles otherwise: 700 x 700 x 256
// kernels 6.0 / 6.4, x 128 5.8 / 5.3: only above 128.
// Fewer terms than kLeastK go to the library: six of the nine products of two
// splits leave a single product 8.7e-8 off where fp32 rounds it to 5.9e-8; from four
// terms on, the split's sum is the closer one.
constexpr int64_t kLeastK = 4;
constexpr int64_t kLargeTiles = 1024, kSmallTiles = 256, kSmallK = 896, kShortTiles = 640, kShortK = 256;
constexpr int kGoodLibrary = 100200;
constexpr int64_t kGoodLibraryK = 512, kGoodLibraryShortK = 128;

static int64_t tile_count(int64_t M, int64_t N, int64_t batch, int64_t t) {
    return (M + t - 1) / t * ((N + t - 1) / t) * batch;
}
static bool vectors(bool ak, bool bk, int64_t K, const float* A, int64_t lda, int64_t stride_a, const float* B, int64_t ldb,
                    int64_t stride_b) {
    return K % 4 == 0 && (!ak || (lda % 4 == 0 && stride_a % 4 == 0 && aligned16(A))) &&
           (!bk || (ldb % 4 == 0 && stride_b % 4 == 0 && aligned16(B)));
}
// 0: the library; 128: gemm_tile; 16, 4: gemm_strip with so many waves.
static int pick(mimir_ctx* ctx, bool ak, bool bk, bool vec, int64_t M, int64_t N, int64_t K, int64_t lda,
                int64_t ldb, int64_t batch) {
    constexpr int64_t kMost = int64_t{1} << 30;
    const int force = ctx->tune.gemm;  // one of the above, or 1 for the library
    if (force == 1 || ctx->tune.blas_lt == 0 || K < kLeastK || M > kMost || N > kMost || K > kMost) return 0;
    const auto below = [](int64_t floats) { return floats < (int64_t{1} << 29); };  // byte offsets within a tile
    if (force == 128 || (!force && tile_count(M, N, batch, 128) >= kLargeTiles))
        return below((ak ? 128 : kStep) * lda) && below((bk ? 128 : kStep) * ldb) ? 128 : 0;
    if (!below(ak ? 32 * lda + K : K * lda + 32) || !below(bk ? 32 * ldb + K : K * ldb + 32)) return 0;
    if (force) return force;
    const int64_t tiles = tile_count(M, N, batch, 32);
    if (tiles > kShortTiles) return 0;
    int64_t least = 0, most = tiles > kSmallTiles || !(vec || (!ak && !bk)) ? kShortK : kSmallK;
    if (gemm_lt_version(ctx) >= kGoodLibrary) {
        if (tiles > kSmallTiles) least = ak && bk ? most : kGoodLibraryShortK;
        else most = std::min(most, ak && bk ? kGoodLibraryShortK : kGoodLibraryK);
    }
    return K <= least || K > most ? 0 : tiles <= kSmallTiles ? 16 : 4;
}

int gemm_split(mimir_ctx* ctx, bool trans_a, bool trans_b, int64_t M, int64_t N, int64_t K, float alpha, const float* A,
               int64_t lda, int64_t stride_a, const float* B, int64_t ldb, int64_t stride_b, float beta, float* C,
               int64_t ldc, int64_t stride_c, int64_t batch, bool* taken) {
    const bool ak = !trans_a, bk = trans_b;
    const bool vec = vectors(ak, bk, K, A, lda, stride_a, B, ldb, stride_b);
    const int kind = pick(ctx, ak, bk, vec, M, N, K, lda, ldb, batch);
    const int64_t t = kind == 128 ? 128 : 32, total = tile_count(M, N, batch, t), grid = (total + kXcds - 1) / kXcds * kXcds;
    *taken = kind != 0 && dispatch_fits(grid, kind == 16 ? 1024 : kGemmThreads);
    if (!*taken) return MIMIR_OK;
    const GemmArgs g{A, B, C, lda, ldb, ldc, stride_a, stride_b, stride_c, static_cast<int32_t>(M), static_cast<int32_t>(N),
                     static_cast<int32_t>(K), static_cast<uint32_t>((M + t - 1) / t),
                     static_cast<uint32_t>((N + t - 1) / t), static_cast<uint32_t>(total), alpha, beta};
    with_layout(ak, bk, vec, [&](auto a, auto b, auto v) {
        constexpr bool kA = decltype(a)::value, kB = decltype(b)::value, kV = decltype(v)::value;
        const auto n = static_cast<unsigned>(grid);
        if (kind == 128) gemm_tile<kA, kB, kV><<<n, kGemmThreads, 0, ctx->stream>>>(g);
        else if (kind == 16) gemm_strip<16, kA, kB, kV><<<n, 16 * kWave, 0, ctx->stream>>>(g);
        else gemm_strip<4, kA, kB, kV><<<n, 4 * kWave, 0, ctx->stream>>>(g);
    });
    return launched(ctx, "gemm_split");
}

}  // namespace mimir
