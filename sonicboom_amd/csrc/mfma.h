// Matrix-core (MFMA) building blocks for gfx950, wave of 64 lanes.
//
// v_mfma_f32_16x16x32_bf16: D[16x16] += A[16x32] * B[32x16].  Lane l holds
//   A[row = l % 16][k = 8 * (l / 16) + 0..7]   (8 bf16 = 16 bytes)
//   B[k = 8 * (l / 16) + 0..7][col = l % 16]
//   D[row = 4 * (l / 16) + i][col = l % 16], i = 0..3
// A and B take their k elements by the same rule, so a kernel that feeds both
// operands from memory with one address formula computes the full dot product
// whatever that rule is; only the D layout shapes the epilogues.
#pragma once

#include "common.h"

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float floatx4_t __attribute__((ext_vector_type(4)));
typedef float floatx16_t __attribute__((ext_vector_type(16)));

__device__ __forceinline__ bf16x8_t as_bf16x8(uint4 v) { return __builtin_bit_cast(bf16x8_t, v); }

__device__ __forceinline__ floatx4_t mfma16(bf16x8_t a, bf16x8_t b, floatx4_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ floatx16_t mfma32(bf16x8_t a, bf16x8_t b, floatx16_t c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

// 16 bytes from global memory, or zeros when the guard fails.
__device__ __forceinline__ uint4 ld16(const void *p, bool ok) {
  return ok ? *reinterpret_cast<const uint4 *>(p) : make_uint4(0u, 0u, 0u, 0u);
}

// The cache policy of loads of what a launch reads once, as buffer loads take it (non-temporal): the weights of a product of
// few rows, which no other block wants and no cache holds until the next step.  Measured, replayed graphs, weights cold, without
// and with it (us): gated 18,944 x 3,584 of 8 rows 53.8 -> 48.7, 3,584 x 18,944 26.5 -> 25.2, gated 11,008 x 2,048 of 2 rows
// 20.8 -> 19.6, gated 4,864 x 896 of one row 7.6 -> 7.2, 1,536 x 8,960 of 48 rows 11.0 -> 10.7; a plain read of 272 MB in the same
// order of addresses 46.8 -> 41.9.  Weights that stay in a cache from one step to the next lose by it, 8.7 MB read again and again by one
// product 3.1 -> 4.5.  Whole decode steps, us, at 1, 8 and 24 rows: models of 42 MB 198 -> 190, 217 -> 208, 281 -> 283; 84 MB 337 -> 332, 367 ->
// 372, 468 -> 481; 176 MB 353 -> 358, 380 -> 389, 495 -> 507; 251 MB 460 -> 447, 509 -> 497, 674 -> 649; 459 MB 736 -> 657, 772 -> 718, 1,033 ->
// 991; 988 MB 832 -> 748, 883 -> 840, 1,126 -> 1,133.  What loses is not told by a matrix (those of 176 and 251 MB are the same, in other
// numbers), so the policy is one for all.
constexpr int kReadOnce = 2;

// Two floats to two bf16 packed in 32 bits (low half first), round to nearest even: one
// v_cvt_pk_bf16_f32.
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint32_t pack_bf16(float lo, float hi) {
  const bf16x2_t v = {(__bf16)lo, (__bf16)hi};
  return __builtin_bit_cast(uint32_t, v);
}

// The maximum over the four lanes l % 16, l % 16 + 16, + 32, + 48 (the four lane groups that hold
// one column of an MFMA result), in every one of them.  Two lane swaps inside the vector unit
// (v_permlane32_swap, v_permlane16_swap: halves of the wave, then odd against even rows of 16)
// where a shuffle would go through LDS and make the wave wait for everything it has asked of it.
// Both operands of a swap are the same value, and the halves it returns are taken apart into
// variables first: written as max(p[0], p[1]) the compiler drops the maximum.
__device__ __forceinline__ float max_over_lane_groups(float v) {
  const uint32_t u = __builtin_bit_cast(uint32_t, v);
  const auto p = __builtin_amdgcn_permlane32_swap(u, u, false, false);
  const uint32_t p0 = p[0], p1 = p[1];
  const float a = fmaxf(__builtin_bit_cast(float, p0), __builtin_bit_cast(float, p1));
  const uint32_t ua = __builtin_bit_cast(uint32_t, a);
  const auto q = __builtin_amdgcn_permlane16_swap(ua, ua, false, false);
  const uint32_t q0 = q[0], q1 = q[1];
  return fmaxf(__builtin_bit_cast(float, q0), __builtin_bit_cast(float, q1));
}
