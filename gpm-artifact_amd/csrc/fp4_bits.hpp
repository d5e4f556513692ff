// Products of 0/1 matrices held as bit rows, on the FP4 matrix cores of gfx950:
// 32 bits of a row become 32 FP4 values in four registers, 128 positions of 16
// by 16 rows are one instruction, and sums of whole numbers are exact in its
// FP32 accumulators up to 2^24.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace gpm {

typedef int intx4 __attribute__((ext_vector_type(4)));
typedef uint32_t uintx4 __attribute__((ext_vector_type(4)));
typedef int intx8 __attribute__((ext_vector_type(8)));
typedef float floatx4 __attribute__((ext_vector_type(4)));

// 32 bits -> 32 FP4 (E2M1) values, eight to a register, register r holding bits
// r, r + 4, ...: a set bit becomes the value whose code it already is in place
// (0b0001 = 0.5, 0b0010 = 1, 0b0100 = 2; the bit at the sign's place moves down,
// 2) on the one side of a product, and the reciprocal on the other, so that two
// set bits make 1.  The side that is expanded more often takes the in-place codes.
__device__ __forceinline__ intx4 fp4_in_place(uint32_t w) {
  return intx4{(int)(w & 0x11111111u), (int)(w & 0x22222222u), (int)(w & 0x44444444u),
               (int)((w >> 1) & 0x44444444u)};
}
__device__ __forceinline__ intx4 fp4_reciprocal(uint32_t w) {
  return intx4{(int)((w << 2) & 0x44444444u), (int)(w & 0x22222222u),
               (int)((w >> 2) & 0x11111111u), (int)((w >> 3) & 0x11111111u)};
}

// c + A B^T over 128 positions: A, B = 16 rows of FP4 values, lane l holding
// 32 positions (4 of the 128-position chunk's 32-bit words: word l / 16) of row
// l % 16.
__device__ __forceinline__ floatx4 mfma_fp4(intx4 a, intx4 b, floatx4 c) {
  constexpr int kFp4 = 4, kOne = 127;  // operand format; block scale 2^0
  const intx8 a8 = __builtin_shufflevector(a, a, 0, 1, 2, 3, -1, -1, -1, -1);
  const intx8 b8 = __builtin_shufflevector(b, b, 0, 1, 2, 3, -1, -1, -1, -1);
  return __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(a8, b8, c, kFp4, kFp4, 0, kOne, 0, kOne);
}

}  // namespace gpm
