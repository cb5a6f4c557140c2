// Matrix products on 16-byte pieces of rows, for any of the element types: 16-bit ones on the 32x32x16 instruction of
// their type, fp32 on v_mfma_f32_32x32x2_f32.
#pragma once
#include "br_common.h"

typedef float br_f32x16v __attribute__((ext_vector_type(16)));
typedef __bf16 br_bf16x8v __attribute__((ext_vector_type(8)));
typedef _Float16 br_f16x8v __attribute__((ext_vector_type(8)));

__device__ inline br_f32x16v br_zero16() {
    br_f32x16v z;
#pragma unroll
    for (int i = 0; i < 16; ++i) z[i] = 0.f;
    return z;
}
__device__ inline br_f32x16v br_mma2(float a, float b, br_f32x16v c) { return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0); }

// One 16-byte piece of a row per lane (lane = row or column lane % 32, half lane / 32 of the step's dims) as operand of
// a product over STEP dims.  Which dim goes to which k index of the instruction does not matter as long as both
// operands agree.
template <typename T> struct BrPiece;
template <> struct BrPiece<__bf16> {
    static constexpr int STEP = 16, N = 8;
    static __device__ inline br_f32x16v mma(uint4 a, uint4 b, br_f32x16v c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(br_bf16x8v, a), __builtin_bit_cast(br_bf16x8v, b), c, 0, 0, 0);
    }
};
template <> struct BrPiece<_Float16> {
    static constexpr int STEP = 16, N = 8;
    static __device__ inline br_f32x16v mma(uint4 a, uint4 b, br_f32x16v c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(br_f16x8v, a), __builtin_bit_cast(br_f16x8v, b), c, 0, 0, 0);
    }
};
template <> struct BrPiece<float> {
    static constexpr int STEP = 8, N = 4;
    static __device__ inline br_f32x16v mma(uint4 a, uint4 b, br_f32x16v c) {
        c = br_mma2(__uint_as_float(a.x), __uint_as_float(b.x), c);
        c = br_mma2(__uint_as_float(a.y), __uint_as_float(b.y), c);
        c = br_mma2(__uint_as_float(a.z), __uint_as_float(b.z), c);
        return br_mma2(__uint_as_float(a.w), __uint_as_float(b.w), c);
    }
};
