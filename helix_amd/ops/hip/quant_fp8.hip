// Rows of bf16 to e4m3 with a scale each: scale = max |x| / 448 (of at least
// 1e-8 / 448), bytes = x / scale, to nearest even.
//
// The activations of 8-bit projections. A launch, bound by its latency at a
// few rows; as library calls it was eight launches of 4 to 8 us each. Bytes
// and scales are those of the calls: 1 / 448 multiplies the maximum, the
// quotient is rounded once, and a maximum that is not a number stays one.
#include "common.h"
#include <torch/extension.h>
#include <ATen/hip/HIPContext.h>

using namespace helix;

namespace {

constexpr int NT = 256;

__global__ __launch_bounds__(NT) void quantize_rows_kernel(
    uint8_t* __restrict__ out, float* __restrict__ scales,
    const uint16_t* __restrict__ x, int K) {
  __shared__ uint32_t red[NT / WAVE];
  const int64_t t = blockIdx.x;
  const uint16_t* row = x + t * K;
  // magnitudes order like their bits, and NaN after all
  uint32_t top = 0;
  for (int c = threadIdx.x * 8; c < K; c += NT * 8) {
    const u16x8 v = *reinterpret_cast<const u16x8*>(row + c);
#pragma unroll
    for (int i = 0; i < 8; ++i) top = max(top, (uint32_t)(v[i] & 0x7fff));
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1)
    top = max(top, (uint32_t)__shfl_xor((int)top, off, WAVE));
  if (threadIdx.x % WAVE == 0) red[threadIdx.x / WAVE] = top;
  __syncthreads();
#pragma unroll
  for (int w = 0; w < NT / WAVE; ++w) top = max(top, red[w]);
  float amax = bf16_to_f32((uint16_t)top);
  if (amax < 1e-8f) amax = 1e-8f;
  const float scale = amax * (1.f / 448.f);
  if (threadIdx.x == 0) scales[t] = scale;
  for (int c = threadIdx.x * 8; c < K; c += NT * 8) {
    float v[8];
    load_bf16x8(row + c, v);
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = v[i] / scale;
    int a = __builtin_amdgcn_cvt_pk_fp8_f32(v[0], v[1], 0, false);
    a = __builtin_amdgcn_cvt_pk_fp8_f32(v[2], v[3], a, true);
    int b = __builtin_amdgcn_cvt_pk_fp8_f32(v[4], v[5], 0, false);
    b = __builtin_amdgcn_cvt_pk_fp8_f32(v[6], v[7], b, true);
    *reinterpret_cast<u32x2*>(out + t * K + c) =
        u32x2{(uint32_t)a, (uint32_t)b};
  }
}

}  // namespace

void quantize_rows(torch::Tensor out, torch::Tensor scales, torch::Tensor x) {
  TORCH_CHECK(x.dim() == 2 && x.is_contiguous() &&
              x.scalar_type() == torch::kBFloat16 && x.size(1) % 8 == 0 &&
              (uintptr_t)x.data_ptr() % 16 == 0);
  TORCH_CHECK(out.is_contiguous() && out.scalar_type() == torch::kUInt8 &&
              out.sizes() == x.sizes() &&
              (uintptr_t)out.data_ptr() % 8 == 0);
  TORCH_CHECK(scales.is_contiguous() &&
              scales.scalar_type() == torch::kFloat32 &&
              scales.numel() == x.size(0));
  if (x.numel() == 0) return;
  hipLaunchKernelGGL(quantize_rows_kernel, dim3(x.size(0)), dim3(NT), 0,
                     at::hip::getCurrentHIPStream(),
                     (uint8_t*)out.data_ptr(), scales.data_ptr<float>(),
                     (const uint16_t*)x.data_ptr(), (int)x.size(1));
}
