// bf16 MFMA GEMM for gfx950: out[M,N] = act(x[M,K] @ w[N,K]^T + bias).
//
// The encoder's and the image model's projections; act: none or GELU (tanh).
// Bound by the matrix cores from a few hundred rows on. Tiles of both operands
// go straight to double-buffered LDS, 64 of the inner dimension at a time,
// with one barrier a step; their 16-byte pieces lie crosswise (piece p of row
// r at p ^ r % 8), so operands leave LDS without bank conflicts. Tiles that
// share rows of x run on one XCD.
//
// Before, 128 x 128 tiles of all sizes, one buffer, rows as in memory (8 lanes
// on a bank). us before -> now (tile; TFLOP/s), M x N x K:
//   16600 x 2304 x 768   131 -> 104  (256; 565)   2304 x 3072 x 1024  33 -> 23
//   16600 x 768 x 768     54 -> 33   (256; 586)   2304 x 1024 x 1024  28 -> 12
//   16600 x 3072 x 768   203 -> 128  (256; 611)   2304 x 4096 x 1024  68 -> 39
//   16600 x 768 x 3072   149 -> 86   (256; 915)   2304 x 1024 x 4096  86 -> 40
//   300 x 768 x 3072      66 -> 18   (64)         8 x 6144 x 1024     21 -> 6
// 192 tiles of 256 against those of 128: 16600 x 768 x 3072 86 and 98; 108
// of them: 2304 x 3072 x 1024 35 and 23. 144 tiles of 128 against those of 64:
// 2304 x 1024 x 1024 13.4 and 12.4. Steps of 32 and scheduling hints for the
// reads from LDS gave nothing.
#include "hybrid/tile.h"
#include <torch/extension.h>
#include <ATen/hip/HIPContext.h>

using namespace helix;

namespace {

constexpr int BK = 64;

struct Gemm {
  const uint16_t* bias;
  int M, N, K, m_tiles, n_tiles, gelu;
};

// Neighbouring numbers on one XCD.
__device__ __forceinline__ int xcd_chunk(int orig, int nwg) {
  const int q = nwg / 8, r = nwg % 8;
  const int xcd = orig % 8, pos = orig / 8;
  return (xcd < r ? xcd * (q + 1) : r * (q + 1) + (xcd - r) * q) + pos;
}

__device__ __forceinline__ float finish(float v, float b, int gelu) {
  v += b;
  if (!gelu) return v;
  const float u = 0.7978845608028654f * (v + 0.044715f * v * v * v);
  // v (1 + tanh u) / 2
  return v * __builtin_amdgcn_rcpf(1.f + __expf(-2.f * u));
}

// WM x WN waves
template <int BM, int BN, int WM, int WN>
__global__ __launch_bounds__(WM* WN* WAVE) void gemm_bf16_kernel(
    uint16_t* __restrict__ out, const uint16_t* __restrict__ x,
    const uint16_t* __restrict__ w, Gemm m) {
  constexpr int TH = WM * WN * WAVE;
  constexpr int MI = BM / WM / 16, NI = BN / WN / 16;
  constexpr int XT = BM * BK / (TH * 8), WT = BN * BK / (TH * 8);
  constexpr int HALF = (BM + BN) * BK;
  extern __shared__ __attribute__((aligned(16))) uint16_t lds[];
  const int lin = xcd_chunk(blockIdx.x, gridDim.x);
  const int m0 = lin / m.n_tiles * BM, n0 = lin % m.n_tiles * BN;
  const int tid = threadIdx.x, wid = tid / WAVE, lane = tid & (WAVE - 1);
  const int lo = lane & 15, hi = lane >> 4;
  const int wr = wid / WN, wc = wid % WN;

  // this thread's 16-byte pieces of either tile; rows past the end repeat
  // the last one and are not stored
  const uint16_t *xp[XT], *wp[WT];
  constexpr int PR = BK / 8;
  const int row0 = tid / PR, p0 = tid % PR;
#pragma unroll
  for (int i = 0; i < XT; ++i) {
    const int r = i * (TH / PR) + row0;
    xp[i] = x + (int64_t)min(m0 + r, m.M - 1) * m.K + (p0 ^ (r & 7)) * 8;
  }
#pragma unroll
  for (int i = 0; i < WT; ++i) {
    const int r = i * (TH / PR) + row0;
    wp[i] = w + (int64_t)min(n0 + r, m.N - 1) * m.K + (p0 ^ (r & 7)) * 8;
  }
  auto load = [&](int k0, uint16_t* dst) {
#pragma unroll
    for (int i = 0; i < XT; ++i)
      __builtin_amdgcn_global_load_lds(
          (const __attribute__((address_space(1))) uint32_t*)(xp[i] + k0),
          (__attribute__((address_space(3))) uint32_t*)(
              dst + (i * TH + wid * WAVE) * 8),
          16, 0, 0);
#pragma unroll
    for (int i = 0; i < WT; ++i)
      __builtin_amdgcn_global_load_lds(
          (const __attribute__((address_space(1))) uint32_t*)(wp[i] + k0),
          (__attribute__((address_space(3))) uint32_t*)(
              dst + BM * BK + (i * TH + wid * WAVE) * 8),
          16, 0, 0);
  };
  floatx4 acc[NI][MI];
#pragma unroll
  for (int j = 0; j < NI; ++j)
#pragma unroll
    for (int i = 0; i < MI; ++i) acc[j][i] = floatx4{0, 0, 0, 0};

  load(0, lds);
  for (int k0 = 0, cur = 0; k0 < m.K; k0 += BK, cur ^= 1) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (k0 + BK < m.K) load(k0 + BK, lds + (cur ^ 1) * HALF);
    const uint16_t* xl = lds + cur * HALF + (wr * MI * 16 + lo) * BK;
    const uint16_t* wl = lds + cur * HALF + (BM + wc * NI * 16 + lo) * BK;
#pragma unroll
    for (int kk = 0; kk < BK / 32; ++kk) {
      const int piece = ((kk * 4 + hi) ^ (lo & 7)) * 8;
      u16x8 xf[MI], wf[NI];
#pragma unroll
      for (int i = 0; i < MI; ++i) xf[i] = ld_u16x8(xl + i * 16 * BK + piece);
#pragma unroll
      for (int j = 0; j < NI; ++j) wf[j] = ld_u16x8(wl + j * 16 * BK + piece);
#pragma unroll
      for (int j = 0; j < NI; ++j)
#pragma unroll
        for (int i = 0; i < MI; ++i)
          acc[j][i] = mfma16(wf[j], xf[i], acc[j][i]);
    }
  }
  // lane: columns 4 hi + q of row lo
#pragma unroll
  for (int j = 0; j < NI; ++j) {
    const int c = n0 + (wc * NI + j) * 16 + hi * 4;
    float b[4];
#pragma unroll
    for (int q = 0; q < 4; ++q)
      b[q] = m.bias != nullptr && c + q < m.N ? bf16_to_f32(m.bias[c + q])
                                              : 0.f;
#pragma unroll
    for (int i = 0; i < MI; ++i) {
      const int r = m0 + (wr * MI + i) * 16 + lo;
      if (r >= m.M) continue;
      uint16_t* o = out + (int64_t)r * m.N + c;
      float v[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) v[q] = finish(acc[j][i][q], b[q], m.gelu);
      if (m.N % 4 == 0) {
        if (c < m.N) st_bf16x4(o, v);
      } else {
#pragma unroll
        for (int q = 0; q < 4; ++q)
          if (c + q < m.N) o[q] = f32_to_bf16(v[q]);
      }
    }
  }
}

template <int BM, int BN, int WM, int WN>
void launch(uint16_t* out, const uint16_t* x, const uint16_t* w, Gemm m) {
  static const hipError_t big = hipFuncSetAttribute(
      (const void*)gemm_bf16_kernel<BM, BN, WM, WN>,
      hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
  TORCH_CHECK(big == hipSuccess, "LDS size refused");
  m.n_tiles = cdiv(m.N, BN);
  hipLaunchKernelGGL((gemm_bf16_kernel<BM, BN, WM, WN>),
                     dim3(cdiv(m.M, BM) * m.n_tiles), dim3(WM * WN * WAVE),
                     2 * (BM + BN) * BK * 2, at::hip::getCurrentHIPStream(),
                     out, x, w, m);
}

}  // namespace

void gemm_bf16(torch::Tensor out, torch::Tensor x, torch::Tensor w,
               c10::optional<torch::Tensor> bias, int64_t act) {
  Gemm m{};
  m.M = x.size(0);
  m.K = x.size(1);
  m.N = w.size(0);
  m.gelu = act == 1;
  TORCH_CHECK(w.size(1) == m.K);
  TORCH_CHECK(m.K % BK == 0, "K must be a multiple of 64");
  TORCH_CHECK(x.is_contiguous() && w.is_contiguous());
  if (m.M == 0 || m.N == 0) return;
  if (bias.has_value()) m.bias = (const uint16_t*)bias->data_ptr();
  uint16_t* o = (uint16_t*)out.data_ptr();
  const uint16_t* xp = (const uint16_t*)x.data_ptr();
  const uint16_t* wp = (const uint16_t*)w.data_ptr();
  // The largest tile of which there are enough for the 256 CUs: operands are
  // read least often, and a CU without work costs more than that.
  auto tiles = [&](int bm, int bn) {
    return (int64_t)cdiv(m.M, bm) * cdiv(m.N, bn);
  };
  if (tiles(256, 256) >= 192) launch<256, 256, 2, 4>(o, xp, wp, m);
  else if (tiles(128, 128) >= 256) launch<128, 128, 2, 4>(o, xp, wp, m);
  else if (m.M > 64) launch<64, 64, 2, 2>(o, xp, wp, m);
  else launch<32, 64, 2, 2>(o, xp, wp, m);
}
