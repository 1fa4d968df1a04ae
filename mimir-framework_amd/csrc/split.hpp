// split.hpp -- fp32 products on the bf16 matrix cores.
//
// After Henry, Tang and Heinecke, "Leveraging the bfloat16 Artificial Intelligence
// Datatype For Higher-Precision Computations" (ARITH 2019), which describes the
// three-term split and how many of its nine products to take.
//
// gfx950 multiplies fp32 operands at 157 TFLOP/s dense and bf16 operands at
// 16 times that.  An fp32 value is the exact sum of three bf16 values
// x = h + m + l (each the round-to-nearest bf16 of what the ones before it
// leave: 3 x 8 significant bits hold the 24 of fp32, and bf16 has fp32's
// exponent range), so a product is
//   x y = h h' + (h m' + m h') + (m m' + h l' + l h') + terms below 2^-24 |x y|,
// six bf16 products accumulated in fp32 by v_mfma_f32_32x32x16_bf16: 6/16 of
// the fp32 matrix time for the same 24-bit operands.  bf16 products are
// exact in fp32, and one MFMA rounds once per 16 products where
// v_mfma_f32_32x32x2_f32 rounds once per 2.  Measured on MI355X against
// float64, relative error of dot products of N(0,1) values, this form / the
// fp32 MFMA chain: length 32 0.69e-7 / 1.03e-7, 128 1.6e-7 / 2.0e-7, 1024
// 4.9e-7 / 5.7e-7.  The builtin rounds to nearest even and keeps subnormal
// inputs and results (checked on the same GPU).  Contractions of one or two terms
// have nothing to gain there: a single product is up to 8.7e-8 off, one fp32
// rounding 5.9e-8 (gemm_split.hip leaves fewer than four terms to the library;
// the attention core's results are no further off down to heads of 1, where the
// errors of the weights are larger).
//
// A value that is infinite, NaN, or so near the largest float that its bf16
// rounds to infinity has no such split: its residues are NaN, so every
// result it reaches is NaN.  The kernels redo the results that come out NaN
// with fp32 products, which gives them the values (infinite, NaN or finite)
// that fp32 arithmetic gives.  Values below 2^-110 lose their last bits to
// bf16's smallest subnormal, 2^-133 (mimir_hip.h says so).
#pragma once

#include "common.hpp"

namespace mimir {

typedef __bf16 b8 __attribute__((ext_vector_type(8)));
typedef __bf16 b2 __attribute__((ext_vector_type(2)));
typedef float f16v __attribute__((ext_vector_type(16)));
typedef float f2 __attribute__((ext_vector_type(2)));
typedef uint32_t u2 __attribute__((ext_vector_type(2)));

// One 16-byte operand per plane: eight values' h, m and l terms.
struct Split8 {
    u4 h, m, l;
};

// Two roundings in one instruction.  The empty asm keeps the compiler from
// converting again to get at one half.
__device__ __forceinline__ uint32_t pack_bf16(float a, float b) {
    uint32_t r = __builtin_bit_cast(uint32_t, b2{static_cast<__bf16>(a), static_cast<__bf16>(b)});
    asm("" : "+v"(r));
    return r;
}

// The three terms of a pair, packed; a in the low half.
__device__ __forceinline__ void split2(float a, float b, uint32_t& h, uint32_t& m, uint32_t& l) {
    h = pack_bf16(a, b);
    a -= __builtin_bit_cast(float, h << 16);
    b -= __builtin_bit_cast(float, h & 0xffff0000u);
    m = pack_bf16(a, b);
    a -= __builtin_bit_cast(float, m << 16);
    b -= __builtin_bit_cast(float, m & 0xffff0000u);
    l = pack_bf16(a, b);
}

__device__ __forceinline__ Split8 split8(const float* x) {
    Split8 s;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        uint32_t h, m, l;
        split2(x[2 * i], x[2 * i + 1], h, m, l);
        s.h[i] = h;
        s.m[i] = m;
        s.l[i] = l;
    }
    return s;
}

__device__ __forceinline__ f16v mfma_bf16(u4 a, u4 b, f16v c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(b8, a), __builtin_bit_cast(b8, b), c, 0, 0, 0);
}

// c += a b for 32x32x16 operands held as splits: the small terms first.
// Lane l supplies row (column) l % 32 of a (b), k slots 8 (l / 32) + 0..7, and
// receives D[8 (r / 4) + 4 (l / 32) + r % 4][l % 32] in register r.
__device__ __forceinline__ f16v mfma_split(const Split8& a, const Split8& b, f16v c) {
    c = mfma_bf16(a.l, b.h, c);
    c = mfma_bf16(a.h, b.l, c);
    c = mfma_bf16(a.m, b.m, c);
    c = mfma_bf16(a.m, b.h, c);
    c = mfma_bf16(a.h, b.m, c);
    return mfma_bf16(a.h, b.h, c);
}

// The same products in the order that mfma_split(b, a, c) takes them, so that the
// transposed result has the same bits.
__device__ __forceinline__ f16v mfma_split_mirror(const Split8& a, const Split8& b, f16v c) {
    c = mfma_bf16(a.h, b.l, c);
    c = mfma_bf16(a.l, b.h, c);
    c = mfma_bf16(a.m, b.m, c);
    c = mfma_bf16(a.h, b.m, c);
    c = mfma_bf16(a.m, b.h, c);
    return mfma_bf16(a.h, b.h, c);
}

// Word 3 of a raw (stride 0) buffer descriptor on gfx9-family GPUs: 32-bit
// data format, no swizzle; out-of-range offsets return zeros.
constexpr int kBufferWord3 = 0x00020000;
// A byte offset past every range the kernels use: the load returns zero.
constexpr uint32_t kOutside = 0x80000000u;

__device__ __forceinline__ __amdgpu_buffer_rsrc_t buffer_of(const float* p, int bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(p), 0, bytes, kBufferWord3);
}
__device__ __forceinline__ f4 buffer_f4(__amdgpu_buffer_rsrc_t r, uint32_t off) {
    return __builtin_bit_cast(f4, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0));
}
__device__ __forceinline__ float buffer_f1(__amdgpu_buffer_rsrc_t r, uint32_t off) {
    return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, off, 0, 0));
}

}  // namespace mimir
