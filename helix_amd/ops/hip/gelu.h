// GELU (tanh form) of the products' epilogues.
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

}  // namespace helix
