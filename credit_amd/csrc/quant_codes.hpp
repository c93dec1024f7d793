// The codes of the row-wise int8 quantisation (quant.hip's formulas).
#pragma once

#include "common.hpp"

namespace credit {

__device__ __forceinline__ float absmax4(f32x4 v) {
  return fmax_nan(fmax_nan(__builtin_fabsf(v.x), __builtin_fabsf(v.y)),
                  fmax_nan(__builtin_fabsf(v.z), __builtin_fabsf(v.w)));
}

__device__ __forceinline__ uint32_t quant1(float x, float inv) {
  float q = __builtin_rintf(x * inv);
  q = __builtin_fminf(127.0f, __builtin_fmaxf(-127.0f, q));
  return static_cast<uint32_t>(static_cast<int32_t>(q)) & 0xFFu;
}

// Four int8 codes packed little-endian (element 0 in the low byte).
__device__ __forceinline__ uint32_t quant4(f32x4 v, float inv) {
  return quant1(v.x, inv) | (quant1(v.y, inv) << 8) | (quant1(v.z, inv) << 16) |
         (quant1(v.w, inv) << 24);
}

// inv as the reference's torch function computes it.
__device__ __forceinline__ float inv_scale(float max_abs) {
  return max_abs > 0.0f ? (1.0f / max_abs) * 127.0f : 0.0f;
}

// The four codes of a vector, at any address.
__device__ __forceinline__ void store_codes(int8_t* q, uint32_t codes) {
  __builtin_memcpy(q, &codes, 4);
}
__device__ __forceinline__ int8_t code1(float x, float inv) {
  return static_cast<int8_t>(static_cast<int32_t>(quant1(x, inv) << 24) >> 24);
}

}  // namespace credit
