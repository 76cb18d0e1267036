// What stands between the projections of an encoder or an image block (bf16).
//
//   norm:  s = x (+ y, or + gate * y);  out = norm(s) * a + b
//   add:   x + gate * y
//
// y may be the stretches of a product (fp32), which are added up here, with its
// bias, instead of in a launch of their own that rounds them.
//
// norm is a layer norm; a and b are its weights, or belong to the image a row
// is part of (a = 1 + scale). Everything inside is fp32, s is rounded only
// where it is kept. Bound by memory: a wave has a row and keeps it in
// registers, so each value is read once and written once. As separate launches
// this was a cast of either operand, an add, a cast back, a norm and for the
// image model four more: 16600 rows of 768 took 74 us a sum and norm (17 now),
// 2304 rows of 1024 46 us a gated sum, norm and modulation (6 now).
#include "common.h"
#include <torch/extension.h>
#include <ATen/hip/HIPContext.h>

using namespace helix;
using OptT = c10::optional<torch::Tensor>;

namespace {

constexpr int NT = 256;

struct Rows {
  const uint16_t *x, *y, *gate, *a, *b;       // y, gate may be null
  const float* sums;           // in the place of y: [stretches][T][H]
  const uint16_t* bias;        // of sums
  int stretches;
  uint16_t *sum, *out;                        // sum may be null
  int64_t gate_stride, mod_stride;      // of an image's row in gate; in a and b
  int T, H, L;                 // rows of an image; 0: a and b are weights
  float eps;
};

// NV: vectors of 8 that a lane has. SUMS: y is m.sums.
template <int NV, bool SUMS>
__global__ __launch_bounds__(NT) void add_norm_kernel(Rows m) {
  const int64_t t = (int64_t)blockIdx.x * (NT / WAVE) + threadIdx.x / WAVE;
  if (t >= m.T) return;
  const int lane = threadIdx.x & (WAVE - 1), nvec = m.H / 8;
  const int64_t of = m.L > 0 ? t / m.L : 0, img = of * m.mod_stride;
  float v[NV][8], total = 0.f;
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int c = (i * WAVE + lane) * 8;
    if (i * WAVE + lane < nvec) {
      load_bf16x8(m.x + t * m.H + c, v[i]);
      if (SUMS || m.y != nullptr) {
        float y[8];
        if constexpr (SUMS) {
          const float* p = m.sums + t * m.H + c;
#pragma unroll
          for (int j = 0; j < 8; ++j) y[j] = 0.f;
#pragma unroll 4
          for (int s = 0; s < m.stretches; ++s, p += (int64_t)m.T * m.H) {
            const f32x4 u = *reinterpret_cast<const f32x4*>(p);
            const f32x4 w = *reinterpret_cast<const f32x4*>(p + 4);
#pragma unroll
            for (int j = 0; j < 4; ++j) {
              y[j] += u[j];
              y[4 + j] += w[j];
            }
          }
          float bias[8];
          load_bf16x8(m.bias + c, bias);
#pragma unroll
          for (int j = 0; j < 8; ++j) y[j] += bias[j];
        } else {
          load_bf16x8(m.y + t * m.H + c, y);
        }
        if (m.gate != nullptr) {
          float g[8];
          load_bf16x8(m.gate + of * m.gate_stride + c, g);
#pragma unroll
          for (int j = 0; j < 8; ++j) y[j] *= g[j];
        }
#pragma unroll
        for (int j = 0; j < 8; ++j) v[i][j] += y[j];
        if (m.sum != nullptr) store_bf16x8(m.sum + t * m.H + c, v[i]);
      }
    } else {
#pragma unroll
      for (int j = 0; j < 8; ++j) v[i][j] = 0.f;
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) total += v[i][j];
  }
  const float mean = wave_reduce_sum(total) / m.H;
  float square = 0.f;
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    if (i * WAVE + lane >= nvec) continue;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      v[i][j] -= mean;
      square += v[i][j] * v[i][j];
    }
  }
  const float inv = rsqrtf(wave_reduce_sum(square) / m.H + m.eps);
  const float one = m.L > 0 ? 1.f : 0.f;
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int c = (i * WAVE + lane) * 8;
    if (i * WAVE + lane >= nvec) continue;
    float a[8], b[8];
    load_bf16x8(m.a + img + c, a);
    load_bf16x8(m.b + img + c, b);
#pragma unroll
    for (int j = 0; j < 8; ++j) b[j] += v[i][j] * inv * (one + a[j]);
    store_bf16x8(m.out + t * m.H + c, b);
  }
}

__global__ __launch_bounds__(NT) void gated_add_kernel(Rows m, int64_t total) {
  const int64_t i = ((int64_t)blockIdx.x * NT + threadIdx.x) * 8;
  if (i >= total) return;
  const int64_t t = i / m.H;
  float x[8], y[8], g[8];
  load_bf16x8(m.x + i, x);
  load_bf16x8(m.y + i, y);
  load_bf16x8(m.gate + t / m.L * m.gate_stride + i % m.H, g);
#pragma unroll
  for (int j = 0; j < 8; ++j) x[j] += g[j] * y[j];
  store_bf16x8(m.out + i, x);
}

// Whether these are values as the kernels read them: bf16 on x's device, on
// 16-byte boundaries.
bool reads(const torch::Tensor& t, const torch::Tensor& x) {
  return t.scalar_type() == torch::kBFloat16 && t.device() == x.device() &&
         (uintptr_t)t.data_ptr() % 16 == 0;
}
// Packed rows like x.
bool like(const torch::Tensor& t, const torch::Tensor& x) {
  return reads(t, x) && t.is_contiguous() && t.sizes() == x.sizes();
}
// A row for every L of x, each `stride` from the next (-1: not known yet).
bool of_image(const torch::Tensor& t, const torch::Tensor& x, const Rows& m,
              int64_t& stride, const uint16_t** at) {
  if (!reads(t, x) || t.dim() != 2 || t.size(1) != m.H || t.stride(1) != 1 ||
      t.stride(0) % 8 != 0 || m.L <= 0 || t.size(0) * m.L < m.T ||
      (stride >= 0 && stride != t.stride(0)))
    return false;
  stride = t.stride(0);
  *at = (const uint16_t*)t.data_ptr();
  return true;
}

bool rows_of(const torch::Tensor& x, const torch::Tensor& out, int64_t L,
             Rows& m) {
  if (!x.is_cuda() || x.dim() != 2 || x.size(1) % 8 != 0 || x.size(1) > 4096 ||
      !like(x, x) || !like(out, x))
    return false;
  m.T = x.size(0);
  m.H = x.size(1);
  m.L = L;
  m.gate_stride = m.mod_stride = -1;
  m.x = (const uint16_t*)x.data_ptr();
  m.out = (uint16_t*)out.data_ptr();
  return true;
}

}  // namespace

// L = 0: out = norm(x + y) a + b with weights a, b; else rows of images of L
// tokens each: sum = x + gate y, out = norm(sum) (1 + a) + b. False, and nothing
// done, for other forms of operands than the kernel reads. y may be the stretches
// [n, T, H] (fp32) of a product whose bias is y_bias.
bool add_norm(OptT sum, torch::Tensor out, torch::Tensor x, OptT y, OptT gate,
              torch::Tensor a, torch::Tensor b, int64_t L, double eps,
              OptT y_bias) {
  Rows m{};
  if (!rows_of(x, out, L, m)) return false;
  m.eps = (float)eps;
  if (y_bias.has_value()) {
    if (!y.has_value() || y->dim() != 3 || y->size(0) < 1 ||
        y->size(1) != m.T || y->size(2) != m.H || !y->is_contiguous() ||
        y->scalar_type() != torch::kFloat32 || y->device() != x.device() ||
        (uintptr_t)y->data_ptr() % 16 != 0 || !reads(*y_bias, x) ||
        !y_bias->is_contiguous() || y_bias->numel() != m.H)
      return false;
    m.sums = y->data_ptr<float>();
    m.bias = (const uint16_t*)y_bias->data_ptr();
    m.stretches = y->size(0);
  } else if (y.has_value()) {
    if (!like(*y, x)) return false;
    m.y = (const uint16_t*)y->data_ptr();
  }
  if (sum.has_value()) {
    if (!like(*sum, x)) return false;
    m.sum = (uint16_t*)sum->data_ptr();
  }
  if (L > 0) {
    if (!of_image(a, x, m, m.mod_stride, &m.a) ||
        !of_image(b, x, m, m.mod_stride, &m.b) ||
        (gate.has_value() &&
         !of_image(*gate, x, m, m.gate_stride, &m.gate)))
      return false;
  } else {
    for (const auto& t : {a, b})
      TORCH_CHECK(t.scalar_type() == torch::kBFloat16 && t.is_contiguous() &&
                  t.dim() == 1 && t.numel() == m.H, "weights of H values");
    if (!reads(a, x) || !reads(b, x) || gate.has_value()) return false;
    m.a = (const uint16_t*)a.data_ptr();
    m.b = (const uint16_t*)b.data_ptr();
  }
  if (m.T == 0) return true;
  const dim3 grid(cdiv(m.T, NT / WAVE));
  auto stream = at::hip::getCurrentHIPStream();
#define HELIX_AN(NV)                                                         \
  do {                                                                       \
    if (m.sums != nullptr)                                                   \
      hipLaunchKernelGGL((add_norm_kernel<NV, true>), grid, dim3(NT), 0,     \
                         stream, m);                                         \
    else                                                                     \
      hipLaunchKernelGGL((add_norm_kernel<NV, false>), grid, dim3(NT), 0,    \
                         stream, m);                                         \
  } while (0)
  if (m.H <= 512) HELIX_AN(1);
  else if (m.H <= 1024) HELIX_AN(2);
  else if (m.H <= 2048) HELIX_AN(4);
  else HELIX_AN(8);
#undef HELIX_AN
  return true;
}

// out = x + gate y; false as above.
bool gated_add(torch::Tensor out, torch::Tensor x, torch::Tensor y,
               torch::Tensor gate, int64_t L) {
  Rows m{};
  if (!rows_of(x, out, L, m) || !like(y, x) ||
      !of_image(gate, x, m, m.gate_stride, &m.gate))
    return false;
  m.y = (const uint16_t*)y.data_ptr();
  const int64_t total = (int64_t)m.T * m.H;
  if (total == 0) return true;
  hipLaunchKernelGGL(gated_add_kernel, dim3((total / 8 + NT - 1) / NT),
                     dim3(NT), 0, at::hip::getCurrentHIPStream(), m, total);
  return true;
}
