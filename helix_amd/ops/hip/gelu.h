// GELU (tanh form) and SiLU of the products' epilogues.
#pragma once
#include "common.h"

namespace helix {

__device__ __forceinline__ float gelu_tanh_f32(float v) {
  // v (1 + tanh u) / 2 = v / (1 + 2^-(2 u log2 e)), u = sqrt(2 / pi)
  // (v + 0.044715 v^3)
  constexpr float C = -2.f * 0.7978845608028654f * 1.4426950408889634f;
  const float e = v * fmaf(v * v, C * 0.044715f, C);
  return v * __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(e));
}

// v / (1 + e^-v). A tile's epilogue has nothing to hide behind, so the division
// is a reciprocal and one correction of its quotient: as exact as a division (over
// 16 million normal values, times another factor, 4.77e-8 from 64 bits; without the
// correction 5.34e-8) in fewer instructions (us divided and now: 8192 rows of 2 x
// 14336 x 4096 1256 and 1249, 4096 of 2 x 4096 x 1024 52.9 and 51.4; without the
// correction 1230 and 49.2). Both sides are a quarter, so that the reciprocal stays
// above the subnormal numbers that the instruction gives as 0; beyond 88 there is
// nothing to correct, or the correction would be inf - inf.
__device__ __forceinline__ float silu_f32(float v) {
  const float n = 0.25f * v;
  const float d = fmaf(
      __builtin_amdgcn_exp2f(v * -1.4426950408889634f), 0.25f, 0.25f);
  const float r = __builtin_amdgcn_rcpf(d), q = n * r;
  return fabsf(v) < 88.f ? fmaf(fmaf(-d, q, n), r, q) : q;
}

}  // namespace helix
