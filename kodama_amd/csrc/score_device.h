// Device helpers of the FP16 score operands (knn_stream.hip has the layout and
// the error bound's use), shared by the kNN and the k-means assignment.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace kodama_hip {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));  // a 16-byte operand piece

__device__ __forceinline__ f16x8 as_f16x8(u32x4 v) { return __builtin_bit_cast(f16x8, v); }

__device__ __forceinline__ uint32_t order_key(float v) {
  const uint32_t b = __float_as_uint(v);
  return (b & 0x80000000u) ? ~b : (b | 0x80000000u);
}
__device__ __forceinline__ float key_value(uint32_t k) {
  return __uint_as_float((k & 0x80000000u) ? (k & 0x7FFFFFFFu) : ~k);
}

// Power-of-two scale: the largest norm lands in (2^13, 2^14].
__device__ __forceinline__ float operand_scale(const float* __restrict__ norm2_max) {
  const float m = fmaxf(norm2_max[0], norm2_max[1]);
  if (!(m > 0.0f)) return 1.0f;
  int e;
  (void)frexpf(sqrtf(m), &e);  // sqrt(m) <= 2^e
  return ldexpf(1.0f, min(max(14 - e, -126), 126));
}

// Norm maxima outside this range (distances may overflow, or squares
// underflow) are not served: every query is flagged.
__device__ __forceinline__ bool norms_usable(const float* __restrict__ norm2_max) {
  const float m = fmaxf(norm2_max[0], norm2_max[1]);
  return m < 1e37f && norm2_max[2] < 1e37f && (m == 0.0f || m > 1e-30f);
}

// Bound of |s - exact score| in scaled units, for a query of scaled norm q and
// train rows of scaled norm <= t (u = 2^-11, FP16's unit roundoff; operands
// below 2^-14 may be flushed):
//   rounding of the operands  parts 1: (2u + u^2) q t; parts 3: 3.1 u^2 q t,
//   flushed operands          2.1 2^-14 sqrt(p) (q + t) + 1,
//   FP32 accumulation         K 2^-23 (q t + t^2 / 2), any order,
//   the norm column           2^-22 t^2 / 2, and its FP32 sum (p + 2) 2^-25 t^2,
//   the reference's own FP32 value  ref 2^-24 values2, values2 the sum of the
//   squared (scaled) norms that this value is computed from.
__device__ __forceinline__ float pair_error(float q, float t, int p, int parts, int width, float values2, float ref) {
  const float u = 0x1p-11f;
  const float c1 = (parts == 1 ? 2.0f * u + u * u : 3.1f * u * u) + width * 0x1.04p-23f;
  const float c2 = 0x1p-23f + (p + 2) * 0x1p-25f + width * 0x1p-24f;
  const float c3 = 2.1f * 0x1p-14f * sqrtf(static_cast<float>(p));
  return 1.05f * (c1 * q * t + c2 * (q * q + t * t) + ref * 0x1p-24f * values2 + c3 * (q + t) + 1.0f);
}

// Wave maximum / minimum by DPP (gfx9 row shifts and row broadcasts), uniform.
__device__ __forceinline__ uint32_t wave_max(uint32_t v) {
#define KODAMA_DPP_MAX(ctrl, rows) \
  v = max(v, static_cast<uint32_t>(__builtin_amdgcn_update_dpp(static_cast<int>(v), static_cast<int>(v), ctrl, rows, 0xf, false)))
  KODAMA_DPP_MAX(0x111, 0xf);
  KODAMA_DPP_MAX(0x112, 0xf);
  KODAMA_DPP_MAX(0x114, 0xf);
  KODAMA_DPP_MAX(0x118, 0xf);
  KODAMA_DPP_MAX(0x142, 0xa);
  KODAMA_DPP_MAX(0x143, 0xc);
#undef KODAMA_DPP_MAX
  return static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(v), 63));
}

// T - 2E with room for its own rounding.
__device__ __forceinline__ float drop_bound(float t, float err2) { return t - err2 - fabsf(t) * 0x1p-22f; }

}  // namespace kodama_hip
