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

// v / (1 + e^-v). A tile's epilogue has nothing to hide behind, and the ten
// instructions of an exact division were a third of a gated one's: 8192 rows of
// 2 x 14336 x 4096 1272 us -> 1246, 4096 of 2 x 4096 x 1024 57 -> 52. Times another
// factor and rounded to bf16 the error against 64 bits is the same (0.00165734 of
// 16 million normal values; before the rounding 5.3e-8 for 4.7e-8).
__device__ __forceinline__ float silu_f32(float v) {
  return v * __builtin_amdgcn_rcpf(
                 1.f + __builtin_amdgcn_exp2f(v * -1.4426950408889634f));
}

}  // namespace helix
