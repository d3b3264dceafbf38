// FP8 (OCP E4M3) row quantisation shared by the KV append kernel
// (append_kv.hip), the fused RoPE append (rope_append.hip) and the decode
// step's append carried by the split reduce kernel (paged_decode.hip), so
// that all write the same codes and scales. The append kernels hold a (token,
// head) row in a wave, lane l elements 4l .. 4l + 3 (head_dim <= 256); the
// RoPE append in an aligned group of lanes. The row maximum gives the scale
// e4m3_row_scale(amax); the codes are e4m3(x / scale) clamped to +-448,
// rounded to nearest even by v_cvt_pk_fp8_f32.
#pragma once

#include "ikl_common.h"

namespace ikl {

template <typename Tag>
__device__ inline void load4(const char *p, float *x);
template <>
__device__ inline void load4<bf16_tag>(const char *p, float *x) {
  const uint2 w = *reinterpret_cast<const uint2 *>(p);
  x[0] = elem<bf16_tag>::lo(w.x);
  x[1] = elem<bf16_tag>::hi(w.x);
  x[2] = elem<bf16_tag>::lo(w.y);
  x[3] = elem<bf16_tag>::hi(w.y);
}
template <>
__device__ inline void load4<f16_tag>(const char *p, float *x) {
  const uint2 w = *reinterpret_cast<const uint2 *>(p);
  x[0] = elem<f16_tag>::lo(w.x);
  x[1] = elem<f16_tag>::hi(w.x);
  x[2] = elem<f16_tag>::lo(w.y);
  x[3] = elem<f16_tag>::hi(w.y);
}
template <>
__device__ inline void load4<f32_tag>(const char *p, float *x) {
  const float4 w = *reinterpret_cast<const float4 *>(p);
  x[0] = w.x;
  x[1] = w.y;
  x[2] = w.z;
  x[3] = w.w;
}

// Maximum over aligned groups of N contiguous lanes; every lane of the wave
// calls it and receives its group's.
template <int N>
__device__ inline float group_max(float v) {
  if constexpr (N >= 2) v = fmaxf(v, dpp_mov<DPP_QUAD_XOR1>(v));
  if constexpr (N >= 4) v = fmaxf(v, dpp_mov<DPP_QUAD_XOR2>(v));
  if constexpr (N >= 8) v = fmaxf(v, dpp_mov<DPP_ROW_HALF_MIRROR>(v));
  if constexpr (N >= 16) v = fmaxf(v, dpp_mov<DPP_ROW_MIRROR>(v));
  if constexpr (N >= 32) v = max_xor16(v);
  if constexpr (N >= 64) v = max_xor32(v);
  return v;
}

// The codes of four elements at a row scale.
__device__ inline int fp8x4(const float *v, float s) {
  float y[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) y[i] = fminf(fmaxf(v[i] / s, -448.0f), 448.0f);
  const int w = __builtin_amdgcn_cvt_pk_fp8_f32(y[0], y[1], 0, false);
  return __builtin_amdgcn_cvt_pk_fp8_f32(y[2], y[3], w, true);
}

// Quantises one row (every lane of the wave calls it; lanes with on == false
// hold no elements) and stores its codes at row + 4 lane and its scale at
// *scale (lane 0).
__device__ inline void store_fp8_row(char *row, float *scale, int lane, bool on, const float *x) {
  float v[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) v[i] = on ? x[i] : 0.f;
  const float amax = group_max<64>(fmaxf(fmaxf(fabsf(v[0]), fabsf(v[1])), fmaxf(fabsf(v[2]), fabsf(v[3]))));
  const float s = e4m3_row_scale(amax);
  if (on) *reinterpret_cast<int *>(row + 4 * lane) = fp8x4(v, s);
  if (lane == 0) *scale = s;
}

}  // namespace ikl
