// A row of bf16 to e4m3 with one scale: what its kernels and the norms that
// write bytes share.
#pragma once
#include "common.h"

namespace helix {

// The greatest of what the workgroup's threads have; red has room for a word of
// each wave, and nothing else uses it.
template <int NT>
__device__ __forceinline__ uint32_t block_reduce_top(uint32_t top,
                                                     uint32_t* red) {
#pragma unroll
  for (int off = WAVE / 2; off > 0; off >>= 1)
    top = max(top, (uint32_t)__shfl_xor((int)top, off, WAVE));
  if (threadIdx.x % WAVE == 0) red[threadIdx.x / WAVE] = top;
  __syncthreads();
#pragma unroll
  for (int w = 0; w < NT / WAVE; ++w) top = max(top, red[w]);
  return top;
}

// top: the greatest bf16 of a row by its bits without the sign, which order
// like magnitudes, and NaN after all. 1 / 448 multiplies it, and a maximum that
// is not a number stays one.
__device__ __forceinline__ float fp8_scale(uint32_t top) {
  float amax = bf16_to_f32((uint16_t)top);
  if (amax < 1e-8f) amax = 1e-8f;
  return amax * (1.f / 448.f);
}

// Four bf16 over their scale, each quotient rounded once; to nearest even.
__device__ __forceinline__ uint32_t fp8x4(u16x4 v, float scale) {
  int a = __builtin_amdgcn_cvt_pk_fp8_f32(bf16_to_f32(v[0]) / scale,
                                          bf16_to_f32(v[1]) / scale, 0, false);
  return (uint32_t)__builtin_amdgcn_cvt_pk_fp8_f32(
      bf16_to_f32(v[2]) / scale, bf16_to_f32(v[3]) / scale, a, true);
}

__device__ __forceinline__ uint32_t top_of(u16x4 v) {
  uint32_t top = 0;
#pragma unroll
  for (int i = 0; i < 4; ++i) top = max(top, (uint32_t)(v[i] & 0x7fff));
  return top;
}

}  // namespace helix
