// Float32-arithmetic tile pieces shared by the chunk-parallel scan kernels
// (chunk_scan_par.hip, chunk_bwd_f32.hip): float32 MFMA over 16-deep steps whose
// operands come from LDS rows (16 bytes) or columns (four single elements), and
// element-wise global access for any width and alignment.
#pragma once

#include <stdint.h>

#include "grm_hip_common.h"

namespace grmhip {

__device__ __forceinline__ f32x4 mfma4(f32x4 a, f32x4 b, f32x4 acc) {
#pragma unroll
  for (int s = 0; s < 4; ++s) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a[s], b[s], acc, 0, 0, 0);
  return acc;
}

// Four consecutive elements of an LDS row (reduction slots 4g + s of a 16-deep step).
template <class E>
__device__ __forceinline__ f32x4 lds_row4(const typename ET<E>::raw* p) {
  f32x4 r;
  if constexpr (sizeof(typename ET<E>::raw) == 2) {
    const uint2 u = *reinterpret_cast<const uint2*>(p);
    r[0] = ET<E>::to_f(static_cast<uint16_t>(u.x & 0xffffu));
    r[1] = ET<E>::to_f(static_cast<uint16_t>(u.x >> 16));
    r[2] = ET<E>::to_f(static_cast<uint16_t>(u.y & 0xffffu));
    r[3] = ET<E>::to_f(static_cast<uint16_t>(u.y >> 16));
  } else {
    const float4 u = *reinterpret_cast<const float4*>(p);
    r[0] = u.x; r[1] = u.y; r[2] = u.z; r[3] = u.w;
  }
  return r;
}

// Four elements of an LDS column, rows p, p + stride, ...
template <class E>
__device__ __forceinline__ f32x4 lds_col4(const typename ET<E>::raw* p, int stride) {
  f32x4 r;
#pragma unroll
  for (int s = 0; s < 4; ++s) r[s] = ET<E>::to_f(p[s * stride]);
  return r;
}

// Four consecutive output elements at element `el` (`left` of them inside the row).
template <class E>
__device__ __forceinline__ void out4(__amdgpu_buffer_rsrc_t r, int el, int left, bool vec, f32x4 v) {
  constexpr int ES = static_cast<int>(sizeof(typename ET<E>::raw));
  if (vec) {
    buf_store4<E>(r, left > 0 ? el * ES : kBufOOB, v);
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i) buf_store1<E>(r, i < left ? (el + i) * ES : kBufOOB, v[i]);
  }
}

__device__ __forceinline__ float ld_mem(__amdgpu_buffer_rsrc_t r, int el, bool f32, bool ok, F32) {
  (void)f32;
  return buf_load1<F32>(r, ok ? el * 4 : kBufOOB);
}
template <class E>
__device__ __forceinline__ float ld_mem(__amdgpu_buffer_rsrc_t r, int el, bool f32, bool ok, E) {
  return f32 ? buf_load1<F32>(r, ok ? el * 4 : kBufOOB) : ET<E>::to_f(buf_load1<E>(r, ok ? el * 2 : kBufOOB));
}

template <class E>
__device__ __forceinline__ float ld_state(const void* p, int64_t i, bool f32) {
  return f32 ? static_cast<const float*>(p)[i] : ET<E>::to_f(static_cast<const typename ET<E>::raw*>(p)[i]);
}

template <class E>
__device__ __forceinline__ void st_state(void* p, int64_t i, bool f32, float x) {
  if (f32) static_cast<float*>(p)[i] = x;
  else static_cast<typename ET<E>::raw*>(p)[i] = ET<E>::from_f(x);
}

}  // namespace grmhip
