// RMSNorm kernels (CDNA4 / gfx950).
//
// Memory-bound: fully vectorized bf16x8 loads/stores (guide G13), fp32
// accumulation, one workgroup per token row.
//
// Replaces the RMSNorm and the residual addition that the reference delegates
// to vLLM's containers.
#include "quant.h"
#include <torch/extension.h>
#include <ATen/hip/HIPContext.h>

using namespace helix;

namespace {

constexpr int WIDE = 1024;     // threads to a row that stays in registers

// Whether a row stays in registers. A CU has room for two such rows, and for
// four of the loop's, whose loads then cover each other: up to one row for each
// of the 256 CUs registers are never slower, up to two where at least three
// quarters of the threads have columns. us by the loop and in registers, 4
// stretches: 256 rows of 256 columns 3.6 and 3.5, 1024 3.8 and 3.6, 4096 6.1
// and 6.0; 257 of 256 3.6 and 3.9, 300 of 2048 5.2 and 5.3, of 3072 6.1 and
// 6.0; 512 of 1024 4.8 and 5.0, of 3072 7.7 and 7.6, of 4096 9.2 and 9.1; 513
// of 4096 9.5 and 10.9, 1024 of 512 4.8 and 7.4. (8 stretches of 257 to 300 rows
// lose up to 0.9 us by it and gain up to 0.9 from 400 rows on.)
bool stays_in_registers(int64_t rows, int64_t columns) {
  return columns <= WIDE * 4 &&
         (rows <= 256 || (rows <= 512 && columns >= WIDE * 3));
}

// out[t, :] = x[t, :] / rms(x[t, :]) * w
// H must be a multiple of 8. One block per token.
template <int BLOCK>
__global__ void rms_norm_kernel(uint16_t* __restrict__ out,
                                const uint16_t* __restrict__ x,
                                const uint16_t* __restrict__ w, float eps,
                                int H) {
  __shared__ float red[BLOCK / WAVE];
  const int t = blockIdx.x;
  const uint16_t* row = x + (int64_t)t * H;
  uint16_t* orow = out + (int64_t)t * H;

  float ss = 0.f;
  const int nvec = H / 8;
  for (int v = threadIdx.x; v < nvec; v += BLOCK) {
    float e[8];
    load_bf16x8(row + v * 8, e);
#pragma unroll
    for (int i = 0; i < 8; ++i) ss += e[i] * e[i];
  }
  ss = block_reduce_sum(ss, red);
  const float inv = rsqrtf(ss / H + eps);

  for (int v = threadIdx.x; v < nvec; v += BLOCK) {
    float e[8], ww[8];
    load_bf16x8(row + v * 8, e);
    load_bf16x8(w + v * 8, ww);
#pragma unroll
    for (int i = 0; i < 8; ++i) e[i] = e[i] * inv * ww[i];
    store_bf16x8(orow + v * 8, e);
  }
}

// residual' = x + residual ; x' = rmsnorm(residual') * w    (both in-place)
template <int BLOCK>
__global__ void fused_add_rms_norm_kernel(uint16_t* __restrict__ x,
                                          uint16_t* __restrict__ residual,
                                          const uint16_t* __restrict__ w,
                                          float eps, int H) {
  __shared__ float red[BLOCK / WAVE];
  const int t = blockIdx.x;
  uint16_t* xrow = x + (int64_t)t * H;
  uint16_t* rrow = residual + (int64_t)t * H;

  float ss = 0.f;
  const int nvec = H / 8;
  for (int v = threadIdx.x; v < nvec; v += BLOCK) {
    float a[8], b[8];
    load_bf16x8(xrow + v * 8, a);
    load_bf16x8(rrow + v * 8, b);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      a[i] += b[i];
      ss += a[i] * a[i];
    }
    store_bf16x8(rrow + v * 8, a);  // new residual
  }
  ss = block_reduce_sum(ss, red);
  const float inv = rsqrtf(ss / H + eps);

  for (int v = threadIdx.x; v < nvec; v += BLOCK) {
    float e[8], ww[8];
    load_bf16x8(rrow + v * 8, e);
    load_bf16x8(w + v * 8, ww);
#pragma unroll
    for (int i = 0; i < 8; ++i) e[i] = e[i] * inv * ww[i];
    store_bf16x8(xrow + v * 8, e);
  }
}

// residual' = sum of x's stretches + residual ; h = rmsnorm(residual') * w
// x is a product whose inner dimension was cut (fp32 [stretches, T, H]); its
// sum is taken here, in order, instead of in a launch of its own (2.5 to 3 us)
// and is not rounded before it meets the residual. FP8: the row leaves as e4m3 and a
// scale, bit by bit what quantize_rows makes of h, for 8-bit projections. That
// launch is bound by its start and its latency: us of both and of one, 4
// stretches: 32 rows of 4096 6.4 and 4.9, of 8192 (the loop) 9.7 and 8.6.
template <int BLOCK, bool FP8>
__global__ __launch_bounds__(BLOCK) void add_sums_rms_norm_kernel(
    void* __restrict__ h, float* __restrict__ scales,
    const float* __restrict__ x, uint16_t* __restrict__ residual,
    const uint16_t* __restrict__ w, float eps, int H, int stretches) {
  __shared__ float red[BLOCK / WAVE];
  const int t = blockIdx.x;
  const int64_t all = (int64_t)gridDim.x * H;
  const float* xrow = x + (int64_t)t * H;
  uint16_t* rrow = residual + (int64_t)t * H;

  float ss = 0.f;
  const int nvec = H / 8;
  for (int v = threadIdx.x; v < nvec; v += BLOCK) {
    float a[8] = {0, 0, 0, 0, 0, 0, 0, 0}, b[8];
    load_bf16x8(rrow + v * 8, b);
#pragma unroll 8
    for (int s = 0; s < stretches; ++s) {
      const f32x4* p = reinterpret_cast<const f32x4*>(xrow + s * all + v * 8);
      const f32x4 u = p[0], z = p[1];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        a[i] += u[i];
        a[4 + i] += z[i];
      }
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      a[i] += b[i];
      ss += a[i] * a[i];
    }
    store_bf16x8(rrow + v * 8, a);  // new residual
  }
  ss = block_reduce_sum(ss, red);
  const float inv = rsqrtf(ss / H + eps);

  auto normed = [&](int v, float (&e)[8]) {
    float ww[8];
    load_bf16x8(rrow + v * 8, e);
    load_bf16x8(w + v * 8, ww);
#pragma unroll
    for (int i = 0; i < 8; ++i) e[i] = e[i] * inv * ww[i];
  };
  if constexpr (FP8) {
    __shared__ uint32_t tops[BLOCK / WAVE];
    auto half = [](const float* e) {
      return u16x4{f32_to_bf16(e[0]), f32_to_bf16(e[1]), f32_to_bf16(e[2]),
                   f32_to_bf16(e[3])};
    };
    uint32_t top = 0;
    for (int v = threadIdx.x; v < nvec; v += BLOCK) {
      float e[8];
      normed(v, e);
      top = max(top, max(top_of(half(e)), top_of(half(e + 4))));
    }
    const float scale = fp8_scale(block_reduce_top<BLOCK>(top, tops));
    if (threadIdx.x == 0) scales[t] = scale;
    for (int v = threadIdx.x; v < nvec; v += BLOCK) {
      float e[8];
      normed(v, e);
      reinterpret_cast<u32x2*>((uint8_t*)h + (int64_t)t * H)[v] =
          u32x2{fp8x4(half(e), scale), fp8x4(half(e + 4), scale)};
    }
  } else {
    for (int v = threadIdx.x; v < nvec; v += BLOCK) {
      float e[8];
      normed(v, e);
      store_bf16x8((uint16_t*)h + (int64_t)t * H + v * 8, e);
    }
  }
}

// The same where a row is at most 4 columns a thread: it stays in registers,
// and all it takes is loaded at once. Bound by the latency of memory, met once
// instead of three times (sums, the row again, weights): after the product that
// writes the stretches, us before -> now 1 row of 8 stretches of 4096 4.9 -> 3.4,
// 16 rows 5.3 -> 3.8. With 8 columns a thread 300 rows of 8192 took 9.3 us
// instead of 7.7, so longer rows keep the loop. stays_in_registers says which
// others do.
template <bool FP8>
__global__ __launch_bounds__(WIDE) void add_sums_rms_norm_wide_kernel(
    void* __restrict__ h, float* __restrict__ scales,
    const float* __restrict__ x, uint16_t* __restrict__ residual,
    const uint16_t* __restrict__ w, float eps, int H, int stretches) {
  __shared__ float red[WIDE / WAVE];
  const int64_t row = (int64_t)blockIdx.x * H, all = (int64_t)gridDim.x * H;
  const bool mine = (int)threadIdx.x * 4 < H;
  const int c = mine ? threadIdx.x * 4 : H - 4;
  u16x4 b = *reinterpret_cast<const u16x4*>(residual + row + c);
  const u16x4 wc = *reinterpret_cast<const u16x4*>(w + c);
  f32x4 a = {0, 0, 0, 0};
#pragma unroll 8
  for (int s = 0; s < stretches; ++s)
    a += *reinterpret_cast<const f32x4*>(x + s * all + row + c);
  float ss = 0.f;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    a[i] += bf16_to_f32(b[i]);
    ss += a[i] * a[i];
    b[i] = f32_to_bf16(a[i]);
  }
  if (mine) *reinterpret_cast<u16x4*>(residual + row + c) = b;
  ss = block_reduce_sum(mine ? ss : 0.f, red);
  const float inv = rsqrtf(ss / H + eps);
  u16x4 o;
#pragma unroll
  for (int i = 0; i < 4; ++i)
    o[i] = f32_to_bf16(bf16_to_f32(b[i]) * inv * bf16_to_f32(wc[i]));
  if constexpr (FP8) {
    __shared__ uint32_t tops[WIDE / WAVE];
    const float scale =
        fp8_scale(block_reduce_top<WIDE>(mine ? top_of(o) : 0, tops));
    if (threadIdx.x == 0) scales[blockIdx.x] = scale;
    if (mine)
      *reinterpret_cast<uint32_t*>((uint8_t*)h + row + c) = fp8x4(o, scale);
  } else if (mine) {
    *reinterpret_cast<u16x4*>((uint16_t*)h + row + c) = o;
  }
}

// LayerNorm (for encoder / bge-class models): out = (x - mu)/sigma * w + b
template <int BLOCK>
__global__ void layer_norm_kernel(uint16_t* __restrict__ out,
                                  const uint16_t* __restrict__ x,
                                  const uint16_t* __restrict__ w,
                                  const uint16_t* __restrict__ b, float eps,
                                  int H) {
  __shared__ float red[BLOCK / WAVE];
  const int t = blockIdx.x;
  const uint16_t* row = x + (int64_t)t * H;
  uint16_t* orow = out + (int64_t)t * H;

  float s = 0.f;
  const int nvec = H / 8;
  for (int v = threadIdx.x; v < nvec; v += BLOCK) {
    float e[8];
    load_bf16x8(row + v * 8, e);
#pragma unroll
    for (int i = 0; i < 8; ++i) s += e[i];
  }
  const float mu = block_reduce_sum(s, red) / H;
  float ss = 0.f;
  for (int v = threadIdx.x; v < nvec; v += BLOCK) {
    float e[8];
    load_bf16x8(row + v * 8, e);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      float d = e[i] - mu;
      ss += d * d;
    }
  }
  ss = block_reduce_sum(ss, red);
  const float inv = rsqrtf(ss / H + eps);
  for (int v = threadIdx.x; v < nvec; v += BLOCK) {
    float e[8], ww[8], bb[8];
    load_bf16x8(row + v * 8, e);
    load_bf16x8(w + v * 8, ww);
    load_bf16x8(b + v * 8, bb);
#pragma unroll
    for (int i = 0; i < 8; ++i) e[i] = (e[i] - mu) * inv * ww[i] + bb[i];
    store_bf16x8(orow + v * 8, e);
  }
}

}  // namespace

void rms_norm(torch::Tensor out, torch::Tensor x, torch::Tensor w,
              double eps) {
  const int T = x.numel() / x.size(-1);
  const int H = x.size(-1);
  TORCH_CHECK(H % 8 == 0, "H must be a multiple of 8");
  TORCH_CHECK(x.scalar_type() == torch::kBFloat16);
  auto stream = at::hip::getCurrentHIPStream();
  hipLaunchKernelGGL((rms_norm_kernel<256>), dim3(T), dim3(256), 0, stream,
                     (uint16_t*)out.data_ptr(), (const uint16_t*)x.data_ptr(),
                     (const uint16_t*)w.data_ptr(), (float)eps, H);
}

void fused_add_rms_norm(torch::Tensor x, torch::Tensor residual,
                        torch::Tensor w, double eps) {
  const int T = x.numel() / x.size(-1);
  const int H = x.size(-1);
  TORCH_CHECK(H % 8 == 0, "H must be a multiple of 8");
  auto stream = at::hip::getCurrentHIPStream();
  hipLaunchKernelGGL((fused_add_rms_norm_kernel<256>), dim3(T), dim3(256), 0,
                     stream, (uint16_t*)x.data_ptr(),
                     (uint16_t*)residual.data_ptr(),
                     (const uint16_t*)w.data_ptr(), (float)eps, H);
}

namespace {

// h: rows of bf16, or with scales of e4m3 bytes
template <bool FP8>
void add_sums(const torch::Tensor& h, float* scales, const torch::Tensor& x,
              const torch::Tensor& residual, const torch::Tensor& w,
              double eps) {
  TORCH_CHECK(x.dim() == 3 && x.is_contiguous() &&
              x.scalar_type() == torch::kFloat32 && h.is_contiguous() &&
              residual.is_contiguous() && residual.dim() == 2 &&
              residual.size(0) == x.size(1) && residual.size(1) == x.size(2) &&
              h.sizes() == residual.sizes());
  for (const auto& t : {h, residual, w})
    TORCH_CHECK(t.device() == x.device() && t.is_contiguous() &&
                t.scalar_type() == (FP8 && t.is_same(h) ? torch::kUInt8
                                                        : torch::kBFloat16),
                "packed bf16 beside the stretches");
  TORCH_CHECK(w.numel() == x.size(2) && x.is_cuda(), "weights of a row");
  const int T = x.size(1);
  const int H = x.size(2);
  TORCH_CHECK(H % 8 == 0, "H must be a multiple of 8");
  if (T == 0 || H == 0) return;               // no row, or no column of one
  auto stream = at::hip::getCurrentHIPStream();
  if (stays_in_registers(T, H)) {
    hipLaunchKernelGGL(add_sums_rms_norm_wide_kernel<FP8>, dim3(T), dim3(WIDE),
                       0, stream, h.data_ptr(), scales, x.data_ptr<float>(),
                       (uint16_t*)residual.data_ptr(),
                       (const uint16_t*)w.data_ptr(), (float)eps, H,
                       (int)x.size(0));
    return;
  }
  hipLaunchKernelGGL((add_sums_rms_norm_kernel<512, FP8>), dim3(T), dim3(512),
                     0, stream, h.data_ptr(), scales, x.data_ptr<float>(),
                     (uint16_t*)residual.data_ptr(),
                     (const uint16_t*)w.data_ptr(), (float)eps, H,
                     (int)x.size(0));
}

}  // namespace

void add_sums_rms_norm(torch::Tensor h, torch::Tensor x,
                       torch::Tensor residual, torch::Tensor w, double eps) {
  add_sums<false>(h, nullptr, x, residual, w, eps);
}

void add_sums_rms_norm_fp8(torch::Tensor h, torch::Tensor scales,
                           torch::Tensor x, torch::Tensor residual,
                           torch::Tensor w, double eps) {
  TORCH_CHECK(scales.is_contiguous() && scales.device() == x.device() &&
              scales.scalar_type() == torch::kFloat32 && x.dim() == 3 &&
              scales.numel() == x.size(1));
  add_sums<true>(h, scales.data_ptr<float>(), x, residual, w, eps);
}

bool norm_in_registers(int64_t rows, int64_t columns) {
  return stays_in_registers(rows, columns);
}

void layer_norm(torch::Tensor out, torch::Tensor x, torch::Tensor w,
                torch::Tensor b, double eps) {
  const int T = x.numel() / x.size(-1);
  const int H = x.size(-1);
  TORCH_CHECK(H % 8 == 0, "H must be a multiple of 8");
  auto stream = at::hip::getCurrentHIPStream();
  hipLaunchKernelGGL((layer_norm_kernel<256>), dim3(T), dim3(256), 0, stream,
                     (uint16_t*)out.data_ptr(), (const uint16_t*)x.data_ptr(),
                     (const uint16_t*)w.data_ptr(),
                     (const uint16_t*)b.data_ptr(), (float)eps, H);
}
