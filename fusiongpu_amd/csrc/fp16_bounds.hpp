// fp16_bounds.hpp -- fp16 operands with a stated rounding, for the kernels that
// bound distances on v_mfma_f32_32x32x16_f16 (screen.hip, assign.hip, knn.hip).
#pragma once

#include <cmath>

#include "common.hpp"

namespace fgpu {

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));

// ---- fp16 with stated rounding, normal values and zero only ----------------------
// Every operand and constant a bound kernel gives the MFMA is 0 or a normal fp16:
// magnitudes below 2^-14 are flushed by these helpers (in the stated
// direction), and the error norms are measured against the stored values, so
// nothing depends on how the MFMA treats subnormal inputs.
constexpr float kHMin = 0x1p-14f;            // smallest normal fp16
constexpr uint16_t kHOne = 0x3C00u;          // 1.0
constexpr uint16_t kHBig = 0x7BFFu;          // 65504, the largest finite fp16
constexpr uint32_t kOneOne = 0x3C003C00u;    // two fp16 1.0
__device__ __forceinline__ double h_val(uint16_t b) { return (double)(float)__builtin_bit_cast(_Float16, b); }
__device__ __forceinline__ float h_float(uint16_t b) { return (float)__builtin_bit_cast(_Float16, b); }
// Nearest (f finite, |f| < 65504), magnitudes below 2^-14 to zero.
__device__ __forceinline__ uint16_t h_rn(float f) {
  return fabsf(f) < kHMin ? (uint16_t)0 : __builtin_bit_cast(uint16_t, (_Float16)f);
}
// The neighbours of b among {0, normal fp16}.
__device__ __forceinline__ uint16_t h_next_down(uint16_t b) {
  const uint16_t mag = b & 0x7FFFu;
  if (mag == 0) return 0x8400u;                                     // 0 -> -2^-14
  if (b & 0x8000u) return (uint16_t)(b + 1u);                       // larger magnitude
  return mag == 0x0400u ? (uint16_t)0 : (uint16_t)(b - 1u);         // 2^-14 -> 0
}
__device__ __forceinline__ uint16_t h_next_up(uint16_t b) {
  const uint16_t mag = b & 0x7FFFu;
  if (mag == 0) return 0x0400u;                                     // 0 -> 2^-14
  if (b & 0x8000u) return mag == 0x0400u ? (uint16_t)0 : (uint16_t)(b - 1u);
  return (uint16_t)(b + 1u);
}
// A value of {0, normal fp16} <= v, and one >= v (|v| < 65504): the nearest,
// moved one step when it lies on the wrong side.
__device__ __forceinline__ uint16_t h_down(double v) {
  uint16_t b = h_rn((float)v);
  while (h_val(b) > v) b = h_next_down(b);
  return b;
}
__device__ __forceinline__ uint16_t h_up(double v) {
  uint16_t b = h_rn((float)v);
  while (h_val(b) < v) b = h_next_up(b);
  return b;
}
// The largest float <= v and the smallest float >= v (v finite).
__device__ __forceinline__ float f_step_down(float f) {
  if (f == 0.0f) return -0x1p-149f;
  const uint32_t u = __float_as_uint(f);
  return __uint_as_float(f > 0.0f ? u - 1u : u + 1u);
}
__device__ __forceinline__ float f_step_up(float f) {
  if (f == 0.0f) return 0x1p-149f;
  const uint32_t u = __float_as_uint(f);
  return __uint_as_float(f > 0.0f ? u + 1u : u - 1u);
}
__device__ __forceinline__ float f_below(double v) {
  const float f = (float)v;
  return (double)f > v ? f_step_down(f) : f;
}
__device__ __forceinline__ float f_above(double v) {
  const float f = (float)v;
  return (double)f < v ? f_step_up(f) : f;
}
// Three fp16 whose sum is <= v (UP false) or >= v (UP true), within about
// 2^-34 |v| + 2^-13 (|v| < 65504).  The first two parts are nearest roundings,
// so each remainder is exact in double; the last is rounded in the stated
// direction.
template <bool UP>
__device__ __forceinline__ void split3(double v, uint16_t& b1, uint16_t& b2, uint16_t& b3) {
  b1 = h_rn((float)v);
  const double r1 = v - h_val(b1);
  b2 = h_rn((float)r1);
  const double r2 = r1 - h_val(b2);
  b3 = UP ? h_up(r2) : h_down(r2);
}
__device__ __forceinline__ uint32_t pack2(uint16_t lo, uint16_t hi) { return (uint32_t)lo | ((uint32_t)hi << 16); }

// ---- scales of rows and columns (assign.hip, knn.hip) -----------------------------
// The margins take the exact fp32 chain as within a relative gamma(130) of the
// distance.  Near the subnormal range its roundings are absolute, 130 of at most
// 2^-150: below 2^-142.  Scaled (by at most 2^13 / M, M = max(||x||^2, ||c||^2))
// that stays below 2^-38 for M >= kNormMin, nothing against the margins' absolute
// 2^-13; the fp32 norms and rounding errors, whose squares may each have lost
// 2^-150, keep their bounds too.  Smaller data takes every exact distance: without
// the limit, of 32768 Gaussian rows of 128 dims 1 lost its nearest of 200 columns
// at coordinates of 2^-72 and 2542 at 2^-74.
constexpr float kNormMin = 0x1p-90f;
constexpr float kNormMax = 0x1p100f;
// Whether a row of squared norm n2 against columns of at most cn_max has scales.
__device__ __forceinline__ bool norms_in_range(float n2, float cn_max) {
  return n2 < kNormMax && cn_max < kNormMax && fmaxf(n2, cn_max) >= kNormMin;
}
// n2 < 2^norm_exp(n2), the least such power.
__device__ __forceinline__ int norm_exp(float n2) {
  int e = 0;
  (void)frexpf(n2, &e);
  return e;
}
// sc: sqrt(cn_max) 2^sc <= 64.
__device__ __forceinline__ int column_scale(float cn_max) {
  const int s = 6 - ((norm_exp(cn_max) + 1) >> 1);
  return s > 100 ? 100 : s < -100 ? -100 : s;
}

}  // namespace fgpu
