// bnn_mfma_f4.h - device helpers of the binary layers on the FP4 matrix cores
// (bnn_bconv_mfma.hip says how bits become operands and sums become rules).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace bnn {
namespace {

typedef int i32x4v __attribute__((ext_vector_type(4)));
typedef int i32x8v __attribute__((ext_vector_type(8)));
typedef float f32x4v __attribute__((ext_vector_type(4)));

__device__ __forceinline__ f32x4v mfma_f4(const i32x4v& a, const i32x4v& b, const f32x4v& c) {
  const i32x8v A = {a[0], a[1], a[2], a[3], 0, 0, 0, 0}, B = {b[0], b[1], b[2], b[3], 0, 0, 0, 0};
  // cbsz = blgp = 4: FP4 operands (four registers each); both scales 1
  return __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(A, B, c, 4, 4, 0, 0, 0, 0);
}
__device__ __forceinline__ i32x4v bits_f4(uint32_t w) {
  return i32x4v{(int)(w & 0x11111111u), (int)(w & 0x22222222u), (int)(w & 0x44444444u), (int)((w >> 3) & 0x11111111u)};
}
// rows of 16 lanes: from a and b, rows 0, 1 hold a's row pairs (0 | 2, 1 | 3)
// and rows 2, 3 b's
__device__ __forceinline__ uint32_t or_halves(uint32_t a, uint32_t b) {
  const auto s = __builtin_amdgcn_permlane32_swap(a, b, false, false);
  return s[0] | s[1];
}
// rows {a0 | a1, b0 | b1, a2 | a3, b2 | b3}
__device__ __forceinline__ uint32_t or_rows(uint32_t a, uint32_t b) {
  const auto s = __builtin_amdgcn_permlane16_swap(a, b, false, false);
  return s[0] | s[1];
}
// shift the sign bit of d into v
__device__ __forceinline__ uint32_t push_sign(uint32_t v, float d) {
  return __builtin_amdgcn_alignbit(v, __builtin_bit_cast(uint32_t, d), 31);
}
// (one instruction; fmaxf would first quiet each operand)
__device__ __forceinline__ float max2(float x, float y) { return __builtin_elementwise_maximum(x, y); }
// x of lane l ^ 1
__device__ __forceinline__ float swap_pair(float x) {
  return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, x), 0xB1, 0xF, 0xF, true));  // [1, 0, 3, 2]
}

}  // namespace
}  // namespace bnn
