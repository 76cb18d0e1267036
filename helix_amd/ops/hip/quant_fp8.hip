// Rows of bf16 to e4m3 with a scale each: scale = max |x| / 448 (of at least
// 1e-8 / 448), bytes = x / scale, to nearest even.
//
// The activations of 8-bit projections that no norm has written as bytes
// (add_sums_rms_norm_fp8). Bytes and scales are those of torch's eight launches
// of 4 to 8 us each. Bound by latency at a few rows, where a row that stays in
// registers meets memory once instead of once a turn of two loops: us by the
// loop and in registers, after the launch that writes the rows, 1 row of 14336
// 5.4 and 3.2, 32 6.3 and 3.7, of 8192 4.3 and 2.9, of 4096 2.4 and 2.0, 512 of
// 4096 3.3 and 2.9, of 14336 9.6 and 8.6; by memory at many: 8192 rows of 14336
// 87 and 65 (5.4 TB/s), but of 4096 19.2 and 20.1, whose second read comes from
// cache, and 1000 of 2048 2.6 and 3.2.
#include "quant.h"
#include <torch/extension.h>
#include <ATen/hip/HIPContext.h>

using namespace helix;

namespace {

// Pieces of 8 columns, V of a thread where the row stays in registers (8 V NT
// columns or fewer), else (V 0) any number of them.
template <int NT, int V>
__global__ __launch_bounds__(NT) void quantize_rows_kernel(
    uint8_t* __restrict__ out, float* __restrict__ scales,
    const uint16_t* __restrict__ x, int K) {
  __shared__ uint32_t red[NT / WAVE];
  const int64_t t = blockIdx.x;
  const uint16_t* row = x + t * K;
  uint8_t* to = out + t * K;
  auto at = [&](int c) { return *reinterpret_cast<const u16x8*>(row + c); };
  auto low = [](u16x8 v) { return u16x4{v[0], v[1], v[2], v[3]}; };
  auto high = [](u16x8 v) { return u16x4{v[4], v[5], v[6], v[7]}; };
  uint32_t top = 0;
  auto see = [&](u16x8 v) { top = max(top, max(top_of(low(v)), top_of(high(v)))); };
  auto put = [&](int c, u16x8 v, float scale) {
    *reinterpret_cast<u32x2*>(to + c) =
        u32x2{fp8x4(low(v), scale), fp8x4(high(v), scale)};
  };
  u16x8 v[V > 0 ? V : 1];
  if constexpr (V > 0) {
#pragma unroll
    for (int i = 0; i < V; ++i)               // past the end: the last piece
      v[i] = at(min((i * NT + (int)threadIdx.x) * 8, K - 8));
#pragma unroll
    for (int i = 0; i < V; ++i) see(v[i]);
  } else {
    for (int c = threadIdx.x * 8; c < K; c += NT * 8) see(at(c));
  }
  const float scale = fp8_scale(block_reduce_top<NT>(top, red));
  if (threadIdx.x == 0) scales[t] = scale;
  if constexpr (V > 0) {
#pragma unroll
    for (int i = 0; i < V; ++i) {
      const int c = (i * NT + threadIdx.x) * 8;
      if (c < K) put(c, v[i], scale);
    }
  } else {
    for (int c = threadIdx.x * 8; c < K; c += NT * 8) put(c, at(c), scale);
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
#define HELIX_QR(NT, V)                                                      \
  hipLaunchKernelGGL((quantize_rows_kernel<NT, V>), dim3(x.size(0)),         \
                     dim3(NT), 0, at::hip::getCurrentHIPStream(),            \
                     (uint8_t*)out.data_ptr(), scales.data_ptr<float>(),     \
                     (const uint16_t*)x.data_ptr(), (int)K)
  const int64_t K = x.size(1);
  if (K > 16384 && K <= 32768) HELIX_QR(1024, 4);
  else if (K > 4096 && K <= 16384) HELIX_QR(512, 4);
  else if (K > 2048 && K <= 4096 && x.size(0) <= 512) HELIX_QR(256, 2);
  else HELIX_QR(256, 0);
#undef HELIX_QR
}
