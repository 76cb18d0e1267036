// Fused QKV epilogue: one pass over the fused qkv projection output.
//
// Reads qkv [T, (Hq+2*Hkv)*D] (row stride = the projection's output
// width, so no .contiguous() splits) or its stretches (fp32, summed here in
// order), applies rotate-half rope to Q and K, writes compact roped Q for the
// attention kernels, scatters roped K and V straight into the paged cache, and
// optionally emits compact K/V for the fresh-prefill attention path.
//
// Replaces 5 kernels (3 split copies + rope + reshape_and_cache) with 1. A
// thread has 8 pairs of a head or 8 values, and a token's threads are spread
// over workgroups of 128: with one workgroup of 256 a token, a pair a thread
// at a time, a row took 7.8 us and 16k rows 115.
//
// A few rows are bound by a launch and the latency of memory: both halves of a
// head and its angles are under way together, and a page is found by a shift.
// us before -> now: 1 row of 4 stretches of 6144 2.85 -> 2.6, 8 of 5 3.1 -> 2.75,
// 61 of 2 3.1 -> 2.7; rows in bf16 512 4.15 -> 3.8, 1540 7.7 -> 7.35, 16000 74.5
// -> 74.1.
#include "common.h"
#include <torch/extension.h>
#include <ATen/hip/HIPContext.h>

using namespace helix;

namespace {

constexpr int NT = 128;

struct Epilogue {
  const int64_t* positions;
  const int64_t* slots;
  const void* qkv;
  int64_t stride, all;         // of a row; of a stretch
  uint16_t *q, *k, *v;         // compact; k and v may be null
  void *kc, *vc;
  const float* cs;
  int Hq, Hkv, D, bs, shift, stretches;      // bs is 1 << shift, or shift -1
};

// P times N values of a row from column c on, apart columns from each other.
template <int N, int P, bool SUMS>
__device__ __forceinline__ void read(const Epilogue& m, int64_t t, int c,
                                     int apart, float (*o)[N]) {
  if constexpr (SUMS) {
    const float* p = (const float*)m.qkv + t * m.stride + c;
#pragma unroll
    for (int k = 0; k < P; ++k)
#pragma unroll
      for (int i = 0; i < N; ++i) o[k][i] = 0.f;
#pragma unroll 4
    for (int s = 0; s < m.stretches; ++s, p += m.all)
#pragma unroll
      for (int k = 0; k < P; ++k) {
        const float* from = p + k * apart;
        if constexpr (N == 8) {
          const f32x4 a = *reinterpret_cast<const f32x4*>(from);
          const f32x4 b = *reinterpret_cast<const f32x4*>(from + 4);
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            o[k][i] += a[i];
            o[k][4 + i] += b[i];
          }
        } else {
          o[k][0] += *from;
        }
      }
  } else {
    const uint16_t* p = (const uint16_t*)m.qkv + t * m.stride + c;
#pragma unroll
    for (int k = 0; k < P; ++k)
      if constexpr (N == 8) load_bf16x8(p + k * apart, o[k]);
      else o[k][0] = bf16_to_f32(p[k * apart]);
  }
}
template <int N>
__device__ __forceinline__ void write(uint16_t* p, const float* v) {
  if constexpr (N == 8) store_bf16x8(p, v);
  else *p = f32_to_bf16(*v);
}
template <int N, bool F8>
__device__ __forceinline__ void write_cache(void* c, int64_t at,
                                            const float* v) {
  if constexpr (!F8) {
    write<N>((uint16_t*)c + at, v);
  } else if constexpr (N == 8) {       // OCP e4m3 cache
    u8x8 q;
#pragma unroll
    for (int i = 0; i < 8; ++i) q[i] = f32_to_fp8(v[i]);
    *reinterpret_cast<u8x8*>((uint8_t*)c + at) = q;
  } else {
    ((uint8_t*)c)[at] = f32_to_fp8(*v);
  }
}

template <int N, bool SUMS, bool F8>
__global__ __launch_bounds__(NT) void rope_qkv_cache_kernel(Epilogue m) {
  const int64_t t = blockIdx.x;
  const int half = m.D / 2, per = half / N;
  const int turned = (m.Hq + m.Hkv) * per;    // then the values
  int i = blockIdx.y * NT + threadIdx.x;
  if (i >= turned + m.Hkv * m.D / N) return;
  const int64_t position = m.positions[t];
  const int64_t slot = m.slots != nullptr ? m.slots[t] : -1;
  auto place = [&](int h) {
    const int64_t page = m.shift >= 0 ? slot >> m.shift : slot / m.bs;
    return ((page * m.Hkv + h) * m.bs + (slot - page * m.bs)) * m.D;
  };
  if (i >= turned) {
    i = (i - turned) * N;
    float v[1][N];
    read<N, 1, SUMS>(m, t, (m.Hq + m.Hkv) * m.D + i, 0, v);
    if (m.v != nullptr) write<N>(m.v + t * m.Hkv * m.D + i, v[0]);
    if (slot >= 0) write_cache<N, F8>(m.vc, place(i / m.D) + i % m.D, v[0]);
    return;
  }
  const int h = i / per, d = i % per * N;
  const float* cs = m.cs + position * m.D + d;
  // before the row, so that they are under way with it
  float cosine[N], sine[N], xy[2][N];
#pragma unroll
  for (int j = 0; j < N; ++j) {
    cosine[j] = cs[j];
    sine[j] = cs[half + j];
  }
  read<N, 2, SUMS>(m, t, h * m.D + d, half, xy);
  float *x = xy[0], *y = xy[1];
#pragma unroll
  for (int j = 0; j < N; ++j) {
    const float a = x[j], b = y[j], c = cosine[j], s = sine[j];
    x[j] = a * c - b * s;
    y[j] = b * c + a * s;
  }
  if (h < m.Hq) {
    uint16_t* o = m.q + (t * m.Hq + h) * m.D + d;
    write<N>(o, x);
    write<N>(o + half, y);
    return;
  }
  const int g = h - m.Hq;
  if (m.k != nullptr) {
    uint16_t* o = m.k + (t * m.Hkv + g) * m.D + d;
    write<N>(o, x);
    write<N>(o + half, y);
  }
  if (slot >= 0) {
    write_cache<N, F8>(m.kc, place(g) + d, x);
    write_cache<N, F8>(m.kc, place(g) + half + d, y);
  }
}

}  // namespace

// qkv: [T, C] or [T, heads, head_dim] bf16, or [stretches, T, C] fp32
void rope_qkv_cache(torch::Tensor positions, torch::Tensor qkv,
                    torch::Tensor q_out,
                    c10::optional<torch::Tensor> k_cache,
                    c10::optional<torch::Tensor> v_cache,
                    c10::optional<torch::Tensor> slot_mapping,
                    c10::optional<torch::Tensor> k_out,
                    c10::optional<torch::Tensor> v_out,
                    torch::Tensor cos_sin, int64_t num_q_heads,
                    int64_t num_kv_heads, int64_t head_dim) {
  const int T = positions.size(0);
  if (T == 0) return;
  const bool sums = qkv.dim() == 3 && qkv.scalar_type() == torch::kFloat32;
  TORCH_CHECK(positions.scalar_type() == torch::kInt64);
  TORCH_CHECK(cos_sin.scalar_type() == torch::kFloat32);
  TORCH_CHECK(qkv.stride(-1) == 1, "qkv innermost must be contiguous");
  TORCH_CHECK(sums || qkv.scalar_type() == torch::kBFloat16);
  TORCH_CHECK(head_dim % 8 == 0);
  Epilogue m{};
  m.positions = positions.data_ptr<int64_t>();
  m.qkv = qkv.data_ptr();
  m.stride = qkv.stride(sums ? 1 : 0);
  m.all = sums ? qkv.stride(0) : 0;
  m.stretches = sums ? qkv.size(0) : 1;
  m.q = (uint16_t*)q_out.data_ptr();
  m.k = k_out.has_value() ? (uint16_t*)k_out->data_ptr() : nullptr;
  m.v = v_out.has_value() ? (uint16_t*)v_out->data_ptr() : nullptr;
  m.cs = cos_sin.data_ptr<float>();
  m.Hq = num_q_heads;
  m.Hkv = num_kv_heads;
  m.D = head_dim;
  m.bs = 1;
  m.shift = 0;
  bool f8 = false;
  if (k_cache.has_value()) {
    f8 = k_cache->scalar_type() == torch::kUInt8;
    TORCH_CHECK(v_cache.has_value() && slot_mapping.has_value());
    TORCH_CHECK(slot_mapping->scalar_type() == torch::kInt64);
    m.bs = k_cache->size(2);
    m.shift = (m.bs & (m.bs - 1)) == 0 ? __builtin_ctz(m.bs) : -1;
    m.kc = k_cache->data_ptr();
    m.vc = v_cache->data_ptr();
    m.slots = slot_mapping->data_ptr<int64_t>();
  }
  // 8 values at a time where halves of a head and rows begin on 16 bytes
  const bool vec = head_dim % 16 == 0 && m.stride % 8 == 0 &&
                   (uintptr_t)m.qkv % 16 == 0;
  const int items = ((m.Hq + m.Hkv) * m.D / 2 + m.Hkv * m.D) / (vec ? 8 : 1);
  const dim3 grid(T, cdiv(items, NT));
  auto stream = at::hip::getCurrentHIPStream();
#define LAUNCH(N, S, F)                                                      \
  hipLaunchKernelGGL((rope_qkv_cache_kernel<N, S, F>), grid, dim3(NT), 0,    \
                     stream, m)
#define KIND(N)                                                              \
  do {                                                                       \
    if (sums) {                                                              \
      if (f8) LAUNCH(N, true, true); else LAUNCH(N, true, false);            \
    } else {                                                                 \
      if (f8) LAUNCH(N, false, true); else LAUNCH(N, false, false);          \
    }                                                                        \
  } while (0)
  if (vec) KIND(8); else KIND(1);
#undef KIND
#undef LAUNCH
}
