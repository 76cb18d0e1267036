// bf16 MFMA GEMM for gfx950: out[M,N] = act(x[M,K] @ w[N,K]^T + bias).
//
// The encoder's and the image model's projections (act: none or GELU, tanh) of
// more than a few rows, and Llama's deep ones at a few hundred rows, whose inner
// dimension is cut into stretches that a later reader adds up (fp32
// [stretch][M][N]).
//
// Bound by the matrix cores and by LDS reads, which take about as long. Tiles
// of both operands go straight to LDS; their 16-byte pieces lie crosswise, so
// that the 16 rows of an operand meet every bank once. Workgroups that follow
// each other on an XCD share rows of x and, GROUP at a time, columns of w.
//
//  - 256 x 256 by two halves of 4 waves, a phase apart: while one reads its
//    operands (and orders the tiles of three steps later) the other multiplies,
//    on the same SIMDs. Four tiles of 32 of the inner dimension are in LDS.
//  - smaller tiles with two buffers of 64 and one barrier a step; several
//    workgroups on a CU fill each other's gaps.
//  - 128 x 128 tiles in stretches where tiles leave CUs idle (cut).
//
// Before, 128 x 128 tiles of all sizes, one buffer, rows as in memory (8 lanes
// on a bank). us before -> now with weights in the caches (tile, or stretches of
// 128; TFLOP/s), M x N x K:
//   16600 x 2304 x 768   131 -> 105  (128; 562)   2304 x 3072 x 1024  33 -> 24
//   16600 x 768 x 768     54 -> 35   (128; 557)   2304 x 1024 x 1024  28 -> 13
//   16600 x 3072 x 768   203 -> 123  (128; 639)   2304 x 4096 x 1024  68 -> 36
//   16600 x 768 x 3072   149 -> 83   (256; 950)   2304 x 1024 x 4096  86 -> 36
//   300 x 768 x 3072      66 -> 14   (6 stretches; the one above: 3)
// Products of few rows stream their weights instead (gemm_rows.hip): 8 x 6144 x
// 1024 takes 6.4 from the caches, 7.6 from memory, by tiles 14.1.
// 8192^3 runs at 1248 TFLOP/s. 256 x 256 as 128 is, with two buffers, takes 10%
// longer; three buffers, steps of 32 for the smaller tiles, 256 x 128 and
// scheduling hints for the reads from LDS gave nothing. Tile counts: 108 of
// 256 against 432 of 128 (2304 x 3072 x 1024) 34 and 23; 144 of 128 against
// 576 of 64 (2304 x 1024 x 1024) 14.8 and 12.9.
#include "gemm_join.h"
#include "hybrid/tile.h"
#include <torch/extension.h>
#include <ATen/hip/HIPContext.h>
#include <c10/core/DeviceGuard.h>

using namespace helix;

namespace {

constexpr int GROUP = 4;                      // tiles of rows

struct Gemm {
  const uint16_t* bias;
  float* sums;                 // null: out
  int M, N, K, m_tiles, n_tiles, stretch, gelu;
};

__device__ __forceinline__ float finish(float v, float b, int gelu) {
  v += b;
  return gelu ? gelu_tanh_f32(v) : v;
}

// What a workgroup does: its tile and its part of the inner dimension.
struct Place {
  int m0, n0, split, k0, k1;
};
__device__ __forceinline__ Place place(const Gemm& m, int BM, int BN) {
  const int all = xcd_chunk(blockIdx.x, gridDim.x);
  const int tiles = m.m_tiles * m.n_tiles, at = all % tiles;
  const int first = at / (GROUP * m.n_tiles) * GROUP;
  const int rows = min(GROUP, m.m_tiles - first);
  const int in = at % (GROUP * m.n_tiles);
  Place p;
  p.split = all / tiles;
  p.m0 = (first + in % rows) * BM;
  p.n0 = in / rows * BN;
  p.k0 = p.split * m.stretch;
  p.k1 = min(m.K, p.k0 + m.stretch);
  return p;
}

// Piece p of a row of BK elements lies at p ^ cross(row).
template <int BK>
__device__ __forceinline__ int cross(int r) {
  return BK == 64 ? r >> 1 & 7 : r >> 2 & 3;
}

// This thread's 16-byte pieces of a tile; rows past the end repeat the last
// one and are not stored.
template <int ROWS, int TH, int BK>
struct Pieces {
  static constexpr int PR = BK / 8, N = ROWS * PR / TH;
  const uint16_t* from[N];
  __device__ __forceinline__ Pieces(const uint16_t* a, int row0, int rows,
                                    int K) {
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const int e = i * TH + threadIdx.x, r = e / PR;
      from[i] = a + (int64_t)min(row0 + r, rows - 1) * K +
                (e % PR ^ cross<BK>(r)) * 8;
    }
  }
  __device__ __forceinline__ void load(int k, uint16_t* lds) const {
    const int wave = threadIdx.x / WAVE * WAVE;
#pragma unroll
    for (int i = 0; i < N; ++i)
      __builtin_amdgcn_global_load_lds(
          (const __attribute__((address_space(1))) uint32_t*)(from[i] + k),
          (__attribute__((address_space(3))) uint32_t*)(
              lds + (i * TH + wave) * 8),
          16, 0, 0);
  }
};

// lane: columns c + 4 hi + q (tiles of 16 apart) of rows r + lo
template <int MI, int NI>
__device__ __forceinline__ void store(const Gemm& m, uint16_t* out, int split,
                                      int row0, int col0,
                                      const floatx4 (*acc)[MI]) {
  const int lane = threadIdx.x & (WAVE - 1), lo = lane & 15, hi = lane >> 4;
#pragma unroll
  for (int j = 0; j < NI; ++j) {
    const int c = col0 + j * 16 + hi * 4;
    float b[4];
#pragma unroll
    for (int q = 0; q < 4; ++q)
      b[q] = m.bias != nullptr && c + q < m.N ? bf16_to_f32(m.bias[c + q])
                                              : 0.f;
#pragma unroll
    for (int i = 0; i < MI; ++i) {
      const int r = row0 + i * 16 + lo;
      if (r >= m.M) continue;
      if (m.sums != nullptr) {                // N % 4 == 0
        if (c < m.N)
          *reinterpret_cast<floatx4*>(
              m.sums + ((int64_t)split * m.M + r) * m.N + c) = acc[j][i];
        continue;
      }
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

// WM x WN waves, two buffers.
template <int BM, int BN, int WM, int WN>
__global__ __launch_bounds__(WM* WN* WAVE) void gemm_tiles_kernel(
    uint16_t* __restrict__ out, const uint16_t* __restrict__ x,
    const uint16_t* __restrict__ w, Gemm m) {
  constexpr int BK = 64, TH = WM * WN * WAVE;
  constexpr int MI = BM / WM / 16, NI = BN / WN / 16, HALF = (BM + BN) * BK;
  extern __shared__ __attribute__((aligned(16))) uint16_t lds[];
  const Place p = place(m, BM, BN);
  const int wid = threadIdx.x / WAVE, lane = threadIdx.x & (WAVE - 1);
  const int lo = lane & 15, hi = lane >> 4;
  const int wr = wid / WN, wc = wid % WN;
  const Pieces<BM, TH, BK> xs(x, p.m0, m.M, m.K);
  const Pieces<BN, TH, BK> ws(w, p.n0, m.N, m.K);
  floatx4 acc[NI][MI];
#pragma unroll
  for (int j = 0; j < NI; ++j)
#pragma unroll
    for (int i = 0; i < MI; ++i) acc[j][i] = floatx4{0, 0, 0, 0};

  xs.load(p.k0, lds);
  ws.load(p.k0, lds + BM * BK);
  for (int k = p.k0, cur = 0; k < p.k1; k += BK, cur ^= 1) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (k + BK < p.k1) {
      xs.load(k + BK, lds + (cur ^ 1) * HALF);
      ws.load(k + BK, lds + (cur ^ 1) * HALF + BM * BK);
    }
    const uint16_t* xl = lds + cur * HALF + (wr * MI * 16 + lo) * BK;
    const uint16_t* wl = lds + cur * HALF + (BM + wc * NI * 16 + lo) * BK;
#pragma unroll
    for (int kk = 0; kk < BK / 32; ++kk) {
      const int piece = ((kk * 4 + hi) ^ cross<BK>(lo)) * 8;
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
  store<MI, NI>(m, out, p.split, p.m0 + wr * MI * 16, p.n0 + wc * NI * 16,
                acc);
}

// 256 x 256, 2 x 4 waves, the second row of waves a phase behind the first. A
// step of 32 has two phases, with a barrier after each: operands from LDS,
// products. What a half orders in step t lands in the buffer that both have
// read in step t - 1; before the barrier that ends its reading of step t a
// half waits for its own part of step t + 1, so that the other half, which is
// a phase ahead or behind, finds all of it there.
constexpr int PAIR = 256;

__global__ __launch_bounds__(512, 2) void gemm_pair_kernel(
    uint16_t* __restrict__ out, const uint16_t* __restrict__ x,
    const uint16_t* __restrict__ w, Gemm m) {
  constexpr int BK = 32, TH = 512, MI = 8, NI = 4, BUF = 2 * PAIR * BK;
  extern __shared__ __attribute__((aligned(16))) uint16_t lds[];
  const Place p = place(m, PAIR, PAIR);
  const int wid = threadIdx.x / WAVE, lane = threadIdx.x & (WAVE - 1);
  const int lo = lane & 15, hi = lane >> 4;
  const int wr = wid / 4, wc = wid % 4;
  const Pieces<PAIR, TH, BK> xs(x, p.m0, m.M, m.K);
  const Pieces<PAIR, TH, BK> ws(w, p.n0, m.N, m.K);
  floatx4 acc[NI][MI];
#pragma unroll
  for (int j = 0; j < NI; ++j)
#pragma unroll
    for (int i = 0; i < MI; ++i) acc[j][i] = floatx4{0, 0, 0, 0};
  auto load = [&](int step) {
    uint16_t* to = lds + (step & 3) * BUF;
    xs.load(p.k0 + step * BK, to);
    ws.load(p.k0 + step * BK, to + PAIR * BK);
  };
  const int steps = (p.k1 - p.k0) / BK;
#pragma unroll
  for (int i = 0; i < 3; ++i)
    if (i < steps) load(i);
  asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
  if (wr == 1) asm volatile("s_barrier" ::: "memory");
  const int piece = (hi ^ cross<BK>(lo)) * 8;
  for (int t = 0; t < steps; ++t) {
    const uint16_t* at = lds + (t & 3) * BUF + lo * BK + piece;
    u16x8 xf[MI], wf[NI];
#pragma unroll
    for (int i = 0; i < MI; ++i)
      xf[i] = ld_u16x8(at + (wr * MI + i) * 16 * BK);
#pragma unroll
    for (int j = 0; j < NI; ++j)
      wf[j] = ld_u16x8(at + (PAIR + (wc * NI + j) * 16) * BK);
    if (t + 3 < steps) {
      load(t + 3);                            // 4 pieces of this thread
      asm volatile("s_waitcnt vmcnt(8) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    } else {
      asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    }
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int j = 0; j < NI; ++j)
#pragma unroll
      for (int i = 0; i < MI; ++i)
        acc[j][i] = mfma16(wf[j], xf[i], acc[j][i]);
    __builtin_amdgcn_s_setprio(0);
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_barrier" ::: "memory");
  }
  if (wr == 0) asm volatile("s_barrier" ::: "memory");
  store<MI, NI>(m, out, p.split, p.m0 + wr * MI * 16, p.n0 + wc * NI * 16,
                acc);
}

void start(const void* kernel, int threads, int bytes, Gemm& m, int bm, int bn,
           int stretches, uint16_t* out, const uint16_t* x,
           const uint16_t* w) {
  m.m_tiles = cdiv(m.M, bm);
  m.n_tiles = cdiv(m.N, bn);
  void* args[] = {&out, &x, &w, &m};
  const hipError_t err = hipLaunchKernel(
      kernel, dim3(m.m_tiles * m.n_tiles * stretches), dim3(threads), args,
      bytes, at::hip::getCurrentHIPStream());
  TORCH_CHECK(err == hipSuccess, hipGetErrorString(err));
}

void allow(const void* kernel) {
  TORCH_CHECK(hipFuncSetAttribute(
                  kernel, hipFuncAttributeMaxDynamicSharedMemorySize,
                  160 * 1024) == hipSuccess, "LDS size refused");
}

template <int BM, int BN, int WM, int WN>
void run_tiles(Gemm m, uint16_t* out, const uint16_t* x, const uint16_t* w,
               int stretches = 1) {
  const void* k = (const void*)gemm_tiles_kernel<BM, BN, WM, WN>;
  static const bool once = (allow(k), true);
  (void)once;
  start(k, WM * WN * WAVE, 2 * (BM + BN) * 64 * 2, m, BM, BN, stretches, out,
        x, w);
}

void run_pair(Gemm m, uint16_t* out, const uint16_t* x, const uint16_t* w,
              int stretches = 1) {
  const void* k = (const void*)gemm_pair_kernel;
  static const bool once = (allow(k), true);
  (void)once;
  start(k, 512, 4 * 2 * PAIR * 32 * 2, m, PAIR, PAIR, stretches, out, x, w);
}

// Stretches of 128 x 128 tiles for a product whose tiles leave CUs idle, joined
// by a launch; 1 where whole tiles take no longer. Both are estimated in us:
//   whole:      0.6 a step of 64, times rounds of 256 tiles
//   stretches:  6, 0.6 a step or 0.37 for each 256 workgroups, and their sums
//               written and read at 4.5 TB/s; 4 more, as the launch that joins
//               them costs a host that is behind
// from 693 sizes (66 to 4500 rows of 256 to 4096 columns, 512 to 14336 deep,
// weights from memory) timed whole and in 2, 3, 4, 6 and 8 stretches. What is
// taken is within 2.2% of the best of these, at worst 48%; whole tiles alone
// take 1.54 times as long. Some, whole and as taken: 2304 x 1024 x 4096 48.1
// and 36.3, 300 of its rows 44.0 and 18.5, 700 x 768 x 3072 25.5 and 19.0, 200
// x 2048 x 2048 21.1 and 16.0; as taken and in two: 1000 x 768 x 1024 11.3 and
// 15.1, 1500 x 4096 x 4096 64.9 and 75.3.
int cut(Gemm& m) {
  const int tiles = cdiv(m.M, 128) * cdiv(m.N, 128), steps = m.K / 64;
  if (m.M <= 64 || m.N % 4 != 0) return 1;
  float best = 0.6f * steps * std::max(1.f, tiles / 256.f);
  int n = 1;
  for (int i = 2; i <= std::min(steps, 8); ++i) {
    const float us = 10 + cdiv(steps, i) * std::max(0.6f, 0.37f * tiles * i / 256)
                     + 8.f * i * m.M * m.N / 4.5e6f;
    if (us < best) best = us, n = i;
  }
  m.stretch = cdiv(steps, n) * 64;
  return cdiv(m.K, m.stretch);
}

}  // namespace

void gemm_bf16(torch::Tensor out, torch::Tensor x, torch::Tensor w,
               c10::optional<torch::Tensor> bias, int64_t act) {
  TORCH_CHECK(x.dim() == 2 && w.dim() == 2, "x and w are matrices");
  Gemm m{};
  m.M = x.size(0);
  m.K = x.size(1);
  m.N = w.size(0);
  m.gelu = act == 1;
  TORCH_CHECK(w.size(1) == m.K);
  TORCH_CHECK(m.K % 64 == 0, "K must be a multiple of 64");
  TORCH_CHECK(x.is_contiguous() && w.is_contiguous());
  for (const auto& t : {x, w, out})
    TORCH_CHECK(t.scalar_type() == torch::kBFloat16 &&
                t.device() == x.device(), "bf16 on one device");
  TORCH_CHECK(out.is_contiguous() && out.dim() == 2 && out.size(0) == m.M &&
              out.size(1) == m.N, "out is [M, N]");
  if (bias.has_value()) {
    TORCH_CHECK(bias->scalar_type() == torch::kBFloat16 &&
                bias->numel() == m.N && bias->device() == x.device(),
                "a bias of N values in bf16");
    bias = bias->contiguous();
    m.bias = (const uint16_t*)bias->data_ptr();
  }
  if (m.M == 0 || m.N == 0) return;
  if (m.K == 0) {              // no operands to load: act(bias)
    const torch::Tensor b = bias.has_value() ? bias->reshape({1, m.N})
                                             : at::zeros_like(out);
    out.copy_(m.gelu ? at::gelu(b.to(torch::kFloat32), "tanh") : b);
    return;
  }
  TORCH_CHECK(x.is_cuda(), "operands on the GPU");
  // tiles are loaded 16 bytes at a time
  if ((uintptr_t)x.data_ptr() % 16 != 0) x = x.clone();
  if ((uintptr_t)w.data_ptr() % 16 != 0) w = w.clone();
  uint16_t* o = (uint16_t*)out.data_ptr();
  const uint16_t* xp = (const uint16_t*)x.data_ptr();
  const uint16_t* wp = (const uint16_t*)w.data_ptr();
  m.stretch = m.K;
  // The largest tile of which there are enough for the 256 CUs: operands are
  // read least often, and a CU without work costs more than that. The two
  // halves of 256 x 256 need a long inner dimension, as nothing runs beside
  // their first loads and their stores (768: 16600 x 2304 105 us, 104 with
  // 128; 3072: 16600 x 768 82, 100 with 128).
  auto tiles = [&](int bm, int bn) {
    return (int64_t)cdiv(m.M, bm) * cdiv(m.N, bn);
  };
  if (m.K >= 2048 && tiles(PAIR, PAIR) >= 192) run_pair(m, o, xp, wp);
  else if (const int n = cut(m); n > 1) {
    torch::Tensor sums =
        torch::empty({n, m.M, m.N}, x.options().dtype(torch::kFloat32));
    const uint16_t* b = m.bias;
    const int64_t MN = (int64_t)m.M * m.N;
    m.sums = sums.data_ptr<float>();
    run_tiles<128, 128, 2, 4>(m, nullptr, xp, wp, n);
    hipLaunchKernelGGL(gemm_join_kernel, dim3((MN + 1023) / 1024), dim3(256),
                       0, at::hip::getCurrentHIPStream(), o,
                       sums.data_ptr<float>(), b, MN, m.N, n, m.gelu != 0);
  }
  else if (tiles(128, 128) >= 256) run_tiles<128, 128, 2, 4>(m, o, xp, wp);
  else if (m.M > 64) run_tiles<64, 64, 2, 2>(m, o, xp, wp);
  else run_tiles<32, 64, 2, 2>(m, o, xp, wp);
}

// Sums [stretches, M, N] of as many stretches as there are workgroups for: up
// to 256 of 256 x 256 or 512 of 128 x 128, at most 8.
torch::Tensor gemm_bf16_sums(torch::Tensor x, torch::Tensor w, int64_t tile) {
  const c10::DeviceGuard on(x.device());
  Gemm m{};
  m.M = x.size(0);
  m.K = x.size(1);
  m.N = w.size(0);
  for (const auto& t : {x, w})
    TORCH_CHECK(t.dim() == 2 && t.is_contiguous() && t.is_cuda() &&
                t.device() == x.device() &&
                t.scalar_type() == torch::kBFloat16 &&
                (uintptr_t)t.data_ptr() % 16 == 0);
  TORCH_CHECK(w.size(1) == m.K && m.K > 0 && m.K % 64 == 0 && m.M >= 1 &&
              m.N >= 4 && m.N % 4 == 0 && (tile == PAIR || tile == 128));
  const int tiles = cdiv(m.M, (int)tile) * cdiv(m.N, (int)tile);
  const int most = (tile == PAIR ? 256 : 512) / tiles;
  const int steps = m.K / 64;
  m.stretch = cdiv(steps, std::max(1, std::min({most, steps, 8}))) * 64;
  const int n = cdiv(m.K, m.stretch);
  torch::Tensor sums =
      torch::empty({n, m.M, m.N}, x.options().dtype(torch::kFloat32));
  m.sums = sums.data_ptr<float>();
  const uint16_t* xp = (const uint16_t*)x.data_ptr();
  const uint16_t* wp = (const uint16_t*)w.data_ptr();
  if (tile == PAIR) run_pair(m, nullptr, xp, wp, n);
  else run_tiles<128, 128, 2, 4>(m, nullptr, xp, wp, n);
  return sums;
}
