// Stretches of a product's inner dimension, joined.
#pragma once
#include "gelu.h"
#include "hybrid/tile.h"

namespace helix {
namespace {

// The sums of all stretches, in order; then bias and GELU.
__global__ __launch_bounds__(256) void gemm_join_kernel(
    uint16_t* __restrict__ out, const float* __restrict__ sums,
    const uint16_t* __restrict__ bias, int64_t MN, int N, int stretches,
    bool gelu) {
  const int64_t i = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4;
  if (i >= MN) return;
  float v[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
  for (int s = 0; s < stretches; ++s) {
    const f32x4 p = *reinterpret_cast<const f32x4*>(sums + s * MN + i);
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] += p[j];
  }
  if (bias != nullptr)
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] += bf16_to_f32(bias[i % N + j]);
  if (gelu)
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] = gelu_tanh_f32(v[j]);
  if ((uintptr_t)out % 8 == 0) {
    st_bf16x4(out + i, v);
  } else {
#pragma unroll
    for (int j = 0; j < 4; ++j) out[i + j] = f32_to_bf16(v[j]);
  }
}

}  // namespace
}  // namespace helix
