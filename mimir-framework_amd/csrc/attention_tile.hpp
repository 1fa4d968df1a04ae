// attention_tile.hpp -- the streamed tiles of the attention kernels
// (attention.hip, attention_bwd.hip): 32 rows of a head on their way from
// memory to LDS as three bf16 planes (split.hpp), in one of two layouts, and
// the MFMA operands read from them; and the same products on the fp32 matrix
// cores, for rows whose split result is not finite.
#pragma once

#include "split.hpp"

namespace mimir {

constexpr int kTileRows = 32;

// What both layouts share: 4 * DP items of eight values, dealt to THREADS
// threads; where they do not fill the threads, the first threads (LAST: the
// last ones) take them.  Loads go through a descriptor that starts at the
// tile's first row and ends after the sequence's last, so rows past the end
// read as zeros; columns are clamped into the head.
template <int DP, int THREADS, bool LAST>
struct TileItems {
    static constexpr int kKind = 4 * DP;
    static constexpr int kItems = (kKind + THREADS - 1) / THREADS;
    static constexpr int kSpare = kItems * THREADS - kKind;  // threads without an item
    static __device__ __forceinline__ int item(int j) {
        return static_cast<int>(threadIdx.x) + j * THREADS - (LAST ? kSpare : 0);
    }
    // Wave-uniform: kSpare is a multiple of the wave.
    static __device__ __forceinline__ bool has(int j) {
        if constexpr (kSpare == 0) return true;
        const int start = (__builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x)) & ~(kWave - 1)) + j * THREADS;
        return LAST ? start >= kSpare : start < kKind;
    }
    static __device__ __forceinline__ __amdgpu_buffer_rsrc_t rows_of(const float* base, int tile, int64_t ld, int len,
                                                                     int head_dim) {
        const int rows = min(kTileRows, len - tile * kTileRows);
        // The last row ends with the head, not with the stride.
        return buffer_of(base + static_cast<int64_t>(tile) * kTileRows * ld,
                         static_cast<int>(((rows - 1) * ld + head_dim) * 4));
    }
};

// Rows as they are: planes [3][32 rows][DP], a row padded by 16 bytes (eight
// rows' 16-byte reads touch every bank once).  An item is eight dimensions of
// a row.  VEC: 16-byte loads (head_dim, the stride and the base pointer are
// 16-byte multiples).
template <int DP, int THREADS, bool VEC>
struct RowTile : TileItems<DP, THREADS, false> {
    using Items = TileItems<DP, THREADS, false>;
    static constexpr int kRowBytes = 2 * DP + 16;
    static constexpr int kPlane = kTileRows * kRowBytes, kBytes = 3 * kPlane;
    float x[Items::kItems][8];
    uint32_t off[Items::kItems];  // byte offset of the item's first element
    int32_t step[Items::kItems];  // VEC: bytes from its first four to its second four

    __device__ __forceinline__ void init(int64_t ld, int head_dim) {
#pragma unroll
        for (int j = 0; j < Items::kItems; ++j) {
            const int id = min(Items::item(j), Items::kKind - 1), row = id / (DP / 8), d = 8 * (id % (DP / 8));
            off[j] = static_cast<uint32_t>(row * ld * 4) + 4 * (VEC ? min(d, head_dim - 4) : d);
            step[j] = VEC ? 4 * (min(d + 4, head_dim - 4) - min(d, head_dim - 4)) : 0;
        }
    }
    __device__ __forceinline__ void load(const float* base, int tile, int64_t ld, int len, int head_dim) {
        const __amdgpu_buffer_rsrc_t rs = Items::rows_of(base, tile, ld, len, head_dim);
#pragma unroll
        for (int j = 0; j < Items::kItems; ++j) {
            if (!Items::has(j)) continue;
            if constexpr (VEC) {
                const f4 a = buffer_f4(rs, off[j]), b = buffer_f4(rs, off[j] + step[j]);
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    x[j][e] = a[e];
                    x[j][4 + e] = b[e];
                }
            } else {
                const int d = 8 * (Items::item(j) % (DP / 8));
#pragma unroll
                for (int e = 0; e < 8; ++e) x[j][e] = buffer_f1(rs, off[j] + 4 * (min(d + e, head_dim - 1) - d));
            }
        }
    }
    __device__ __forceinline__ void stash(char* lds) const {
#pragma unroll
        for (int j = 0; j < Items::kItems; ++j) {
            if (!Items::has(j)) continue;
            const int id = Items::item(j);
            char* p = lds + id / (DP / 8) * kRowBytes + id % (DP / 8) * 16;
            const Split8 s = split8(x[j]);
            *reinterpret_cast<u4*>(p) = s.h;
            *reinterpret_cast<u4*>(p + kPlane) = s.m;
            *reinterpret_cast<u4*>(p + 2 * kPlane) = s.l;
        }
    }
    // MFMA operand: dimensions 16 c + 8 hf .. + 7 of row li.
    static __device__ __forceinline__ Split8 at(const char* lds, int li, int hf, int c) {
        const char* p = lds + li * kRowBytes + 32 * c + 16 * hf;
        return Split8{*reinterpret_cast<const u4*>(p), *reinterpret_cast<const u4*>(p + kPlane),
                      *reinterpret_cast<const u4*>(p + 2 * kPlane)};
    }
};

// Columns: planes [3][DP][32 rows], a dimension's rows padded by 16 bytes, in
// the order in which a product over the rows takes them: the eight slots of
// (c, hf) hold rows 16 c + 4 hf + {0..3, 8..11}, the rows that registers
// 8 c .. 8 c + 7 of lane half hf hold of a 32 x 32 MFMA result.  An item is
// one such group of one dimension; 64 lanes read 64 dimensions of a row.
template <int DP, int THREADS>
struct ColTile : TileItems<DP, THREADS, true> {
    using Items = TileItems<DP, THREADS, true>;
    static constexpr int kDimBytes = 2 * kTileRows + 16;
    static constexpr int kPlane = DP * kDimBytes, kBytes = 3 * kPlane;
    float x[Items::kItems][8];
    uint32_t off[Items::kItems];
    uint32_t ld4;

    __device__ __forceinline__ void init(int64_t ld, int head_dim) {
        ld4 = static_cast<uint32_t>(ld * 4);
#pragma unroll
        for (int j = 0; j < Items::kItems; ++j) {
            const int id = max(Items::item(j), 0), group = id / DP;
            off[j] = 4 * min(id % DP, head_dim - 1) + (16 * (group / 2) + 4 * (group % 2)) * ld4;
        }
    }
    __device__ __forceinline__ void load(const float* base, int tile, int64_t ld, int len, int head_dim) {
        const __amdgpu_buffer_rsrc_t rs = Items::rows_of(base, tile, ld, len, head_dim);
#pragma unroll
        for (int j = 0; j < Items::kItems; ++j) {
            if (!Items::has(j)) continue;
#pragma unroll
            for (int e = 0; e < 8; ++e) x[j][e] = buffer_f1(rs, off[j] + ((e & 3) + 8 * (e >> 2)) * ld4);
        }
    }
    __device__ __forceinline__ void stash(char* lds) const {
#pragma unroll
        for (int j = 0; j < Items::kItems; ++j) {
            if (!Items::has(j)) continue;
            const int id = Items::item(j);
            char* p = lds + id % DP * kDimBytes + id / DP * 16;
            const Split8 s = split8(x[j]);
            *reinterpret_cast<u4*>(p) = s.h;
            *reinterpret_cast<u4*>(p + kPlane) = s.m;
            *reinterpret_cast<u4*>(p + 2 * kPlane) = s.l;
        }
    }
    // MFMA operand: the eight rows (c, hf) of dimension 32 db + li.
    static __device__ __forceinline__ Split8 at(const char* lds, int li, int hf, int db, int c) {
        const char* p = lds + (32 * db + li) * kDimBytes + 32 * c + 16 * hf;
        return Split8{*reinterpret_cast<const u4*>(p), *reinterpret_cast<const u4*>(p + kPlane),
                      *reinterpret_cast<const u4*>(p + 2 * kPlane)};
    }
};

// A lane's operand of one row held in registers: dimensions 16 c + 8 hf ..
// + 7 of `row`, zero past head_dim, times `scale`.
template <int DP, bool VEC>
__device__ __forceinline__ void row_operand(const float* row, int hf, int head_dim, float scale, Split8* q) {
#pragma unroll
    for (int c = 0; c < DP / 16; ++c) {
        float x[8];
#pragma unroll
        for (int v = 0; v < 2; ++v) {
            const int d = 16 * c + 8 * hf + 4 * v;
            if constexpr (VEC) {
                const f4 t = d < head_dim ? *reinterpret_cast<const f4*>(row + d) : f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int e = 0; e < 4; ++e) x[4 * v + e] = t[e] * scale;
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e) x[4 * v + e] = d + e < head_dim ? row[d + e] * scale : 0.f;
            }
        }
        q[c] = split8(x);
    }
}

// Stores a wave's 32 x 32 blocks o[DP / 32] of a transposed result (rows =
// dimensions, columns = lanes' rows): out[d] = o * scale, 16 bytes at a time
// when VEC.  Returns NaN in a lane whose values are not all finite.
template <int DP, bool VEC>
__device__ __forceinline__ float store_columns(const f16v* o, float scale, float* row, bool in, int hf, int head_dim) {
    float check = 0.f;
#pragma unroll
    for (int d = 0; d < DP / 32; ++d) {
#pragma unroll
        for (int r = 0; r < 16; r += 4) {
            const int d0 = 32 * d + 8 * (r / 4) + 4 * hf;
            const f4 val{o[d][r] * scale, o[d][r + 1] * scale, o[d][r + 2] * scale, o[d][r + 3] * scale};
#pragma unroll
            for (int e = 0; e < 4; ++e) check += val[e] - val[e];
            if (!in) continue;
            if constexpr (VEC) {
                if (d0 < head_dim) *reinterpret_cast<f4*>(row + d0) = val;
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (d0 + e < head_dim) row[d0 + e] = val[e];
            }
        }
    }
    return check;
}

// The rows (lane % 32) of a wave that a check found not finite.
__device__ __forceinline__ uint32_t bad_rows(float check, bool in) {
    const uint64_t b = __ballot(check != check && in);
    return static_cast<uint32_t>(b | b >> 32);
}

// ---------------------------------------------------------------------------
// Blocks without a split.  A wave whose split result for its 32 rows holds a NaN
// or an infinity computes them again with v_mfma_f32_32x32x2_f32, which gives what
// fp32 arithmetic gives.  Operands come straight from memory, few at a time, and
// kRedoBlocks x 32 dimensions of the result per pass (the scores again for each),
// so that the kernels around it keep their registers.
// ---------------------------------------------------------------------------
template <int DP>
constexpr int kRedoBlocks = DP >= 64 ? 2 : 1;

// D[row0 + 8 (r / 4) + 4 hf + r % 4][lane's row] in register r: the products of
// 32 rows of a matrix with one row per lane (li; both halves the same), times
// `scale`.  Rows at and past len: the last one's, for the caller to mask.  Few
// registers, so that the kernels around it keep theirs.
__device__ __forceinline__ f16v f32_scores(const float* base, int64_t ld, int row0, int len, int head_dim, const float* mine,
                                           float scale) {
    const int li = threadIdx.x % 32, hf = threadIdx.x % kWave / 32;
    const float* row = base + min(row0 + li, len - 1) * ld;
    f16v s = f16v{};
#pragma unroll 1
    for (int j = hf; j < head_dim + hf; j += 16) {  // the halves take turns: dimensions 2 i + hf
        float x[8], y[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int d = min(j + 2 * i, head_dim - 1);
            x[i] = row[d];
            y[i] = mine[d];
        }
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const bool in = j + 2 * i < head_dim;
            s = __builtin_amdgcn_mfma_f32_32x32x2f32(in ? x[i] : 0.f, in ? y[i] * scale : 0.f, s, 0, 0, 0);
        }
    }
    return s;
}

// acc += rows^T w for 32 NB dimensions: rows row0 .. row0 + 31 of a matrix, w as
// f32_scores lays it out (zero for rows a lane does not see), acc as store_columns
// takes it.  A lane sees rows lo .. hi - 1; where some lane does not see a row that
// others see, the row's values, which may not be finite, reach only those that do.
// head_dim: dimensions from `base` on.
template <int NB>
__device__ __forceinline__ void f32_accumulate(const float* base, int64_t ld, int row0, int len, int head_dim, const f16v& w,
                                               int lo, int hi, f16v* acc) {
    const int li = threadIdx.x % 32, hf = threadIdx.x % kWave / 32;
    const int end = min(row0 + kTileRows, len);
    if (__all(lo <= row0 && hi >= end)) {
        int first = row0 + 4 * hf;
        asm volatile("" : "+v"(first));
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int row = first + 8 * (r / 4) + r % 4;
            const float* p = base + min(row, len - 1) * ld;
#pragma unroll
            for (int d = 0; d < NB; ++d) {
                const float v = p[min(32 * d + li, head_dim - 1)];
                acc[d] = __builtin_amdgcn_mfma_f32_32x32x2f32(row < len && 32 * d + li < head_dim ? v : 0.f, w[r], acc[d], 0, 0, 0);
            }
            if (r % 4 == 3) __builtin_amdgcn_sched_barrier(0);  // no more than four rows in flight
        }
        return;
    }
#pragma unroll 1
    for (int row = row0; row < end; ++row) {
        const int at = row - row0;
        float own = 0.f;  // this row's weight, in one of the lane halves
#pragma unroll
        for (int r = 0; r < 16; ++r) own = r == at % 4 + 4 * (at / 8) ? w[r] : own;
        const float weight = __shfl(own, li + 32 * (at / 4 % 2));
        const bool sees = lo <= row && row < hi;
        const float* p = base + row * ld;
        int last = head_dim - 1;
        asm volatile("" : "+v"(last));  // the offsets are computed where they are used, not kept for the loop
#pragma unroll
        for (int d = 0; d < NB; ++d) {
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const float v = p[min(32 * d + 8 * (r / 4) + 4 * hf + r % 4, last)];
                acc[d][r] = sees ? acc[d][r] + weight * v : acc[d][r];
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    }
}

}  // namespace mimir
