// Product of a few rows with a large matrix: x[M,K] @ w[N,K]^T, bf16 with fp32
// sums, M <= 64.
//
// Bound by reading w once. A wave streams its columns of w straight into MFMA
// operands, a chunk of 256 of the inner dimension ahead; x goes to LDS by
// direct loads, once for the columns of all waves. 16-byte piece p of row r
// lies at p ^ r % 16, so operands leave LDS without bank conflicts.
//
// Narrow matrices leave CUs idle, so the inner dimension is cut into stretches
// until there are about WANT workgroups. Their sums (fp32, [stretch][M][N])
// are added by whatever reads the result (norm, rotation), in order, or by a
// launch of their own; nothing is added with atomics.
//
// Gated feed-forward: a wave has 16 columns of the gate and the same 16 of the
// other half and writes silu(gate) * up; neither half goes to memory.
//
// us for N x K = 6144x4096, 4096x4096, 28672x4096, 4096x14336 (the sums left
// to the reader), library kernel in brackets:
//   M  1   11.7 (14.4)   8.6 (15.5)   44.5 (63.4)   23.2 (26.6)
//   M 16   12.4 (15.7)   8.9 (15.6)   45.4 (65.1)   25.2 (27.3)
//   M 32   15.2 (16.3)  10.4 (13.9)   51.8 (54.2)   27.8 (33.8)
//   M 64   17.6 (18.0)  12.2 (15.2)   55.4 (52.3)   31.9 (41.9)
// Adding them up in a launch takes 2.5 to 3 us more. The gated product
// replaces a launch of 4.5 us as well. Reading 28672 x 4096 at 44.5 us is 5.3
// TB/s. Eight waves a workgroup, chunks of 128 or 512, 32 columns a wave and
// 256 or 768 workgroups were each slower on most of these.
#include "hybrid/tile.h"
#include <torch/extension.h>
#include <ATen/hip/HIPContext.h>

using namespace helix;

namespace {

constexpr int KC = 256;                       // inner dimension of a chunk
constexpr int WANT = 512;                     // workgroups, 2 on each CU

struct Product {
  const uint16_t* bias;
  int M, N, K, n_tiles, per;   // per: chunks of a stretch
};

// 16 MI rows, NW waves. GLU: columns n and N + n are a pair of a wave.
template <int MI, int NW, bool GLU>
__global__ __launch_bounds__(NW* WAVE, 2) void gemm_rows_kernel(
    uint16_t* __restrict__ out, float* __restrict__ sums,
    const uint16_t* __restrict__ x, const uint16_t* __restrict__ w,
    Product m) {
  constexpr int NI = GLU ? 2 : 1;
  constexpr int TH = NW * WAVE, BM = MI * 16;
  constexpr int PR = KC / 8, XL = BM * PR / TH, U = KC / 32;
  static_assert(BM * PR % TH == 0, "x tile");
  __shared__ __attribute__((aligned(16))) uint16_t xl[2][BM * KC];
  const int stretch = blockIdx.x / m.n_tiles;
  const int tid = threadIdx.x, wid = tid / WAVE, lane = tid & (WAVE - 1);
  const int lo = lane & 15, hi = lane >> 4;
  const int n0 = (blockIdx.x % m.n_tiles * NW + wid) * 16;
  const int c0 = stretch * m.per, c1 = min(m.K / KC, c0 + m.per);
  const uint16_t* wp[NI];
#pragma unroll
  for (int j = 0; j < NI; ++j)
    wp[j] = w + ((int64_t)j * m.N + min(n0 + lo, m.N - 1)) * m.K + hi * 8;
  const uint16_t* xp[XL];
#pragma unroll
  for (int i = 0; i < XL; ++i) {
    const int e = i * TH + tid, r = e / PR, p = e % PR ^ (r & 15);
    xp[i] = x + (int64_t)min(r, m.M - 1) * m.K + p * 8;
  }
  auto load_x = [&](int c, int b) {
#pragma unroll
    for (int i = 0; i < XL; ++i)
      __builtin_amdgcn_global_load_lds(
          (const __attribute__((address_space(1))) uint32_t*)(xp[i] + c * KC),
          (__attribute__((address_space(3))) uint32_t*)(
              xl[b] + (i * TH + wid * WAVE) * 8),
          16, 0, 0);
  };
  u16x8 wr[2][U][NI];
  auto load_w = [&](int c, int b) {
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int j = 0; j < NI; ++j)
        wr[b][u][j] = ld_u16x8(wp[j] + c * KC + u * 32);
  };
  floatx4 acc[NI][MI];
#pragma unroll
  for (int j = 0; j < NI; ++j)
#pragma unroll
    for (int i = 0; i < MI; ++i) acc[j][i] = floatx4{0, 0, 0, 0};
  auto step = [&](int c, int b) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (c + 1 < c1) {
      load_x(c + 1, b ^ 1);
      load_w(c + 1, b ^ 1);
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int i = 0; i < MI; ++i) {
        const u16x8 xf =
            ld_u16x8(xl[b] + (i * 16 + lo) * KC + ((u * 4 + hi) ^ lo) * 8);
#pragma unroll
        for (int j = 0; j < NI; ++j)
          acc[j][i] = mfma16(wr[b][u][j], xf, acc[j][i]);
      }
  };
  if (c0 < c1) {
    load_x(c0, 0);
    load_w(c0, 0);
  }
  for (int c = c0; c < c1; c += 2) {
    step(c, 0);
    if (c + 1 < c1) step(c + 1, 1);
  }
  // lane: columns 4 hi + q of row lo
  const int n = n0 + hi * 4;
  if (n >= m.N) return;
#pragma unroll
  for (int i = 0; i < MI; ++i) {
    const int r = i * 16 + lo;
    if (r >= m.M) continue;
    float v[4];
    if constexpr (GLU) {
#pragma unroll
      for (int q = 0; q < 4; ++q)
        v[q] = acc[0][i][q] / (1.f + __expf(-acc[0][i][q])) * acc[1][i][q];
    } else {
      if (sums != nullptr) {
        *reinterpret_cast<floatx4*>(
            sums + ((int64_t)stretch * m.M + r) * m.N + n) = acc[0][i];
        continue;
      }
#pragma unroll
      for (int q = 0; q < 4; ++q)
        v[q] = acc[0][i][q] +
               (m.bias != nullptr ? bf16_to_f32(m.bias[n + q]) : 0.f);
    }
    st_bf16x4(out + (int64_t)r * m.N + n, v);
  }
}

// The sums of all stretches, in order.
__global__ __launch_bounds__(256) void gemm_join_kernel(
    uint16_t* __restrict__ out, const float* __restrict__ sums,
    const uint16_t* __restrict__ bias, int64_t MN, int N, int stretches) {
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
  st_bf16x4(out + i, v);
}

Product product_of(const torch::Tensor& x, const torch::Tensor& w, int64_t N,
                   int columns) {
  for (const auto& t : {x, w})
    TORCH_CHECK(t.dim() == 2 && t.is_contiguous() && t.is_cuda() &&
                t.scalar_type() == torch::kBFloat16 &&
                (uintptr_t)t.data_ptr() % 16 == 0);
  Product m{};
  m.M = x.size(0);
  m.K = x.size(1);
  m.N = N;
  TORCH_CHECK(w.size(1) == m.K && m.M >= 1 && m.M <= 64);
  TORCH_CHECK(m.N >= 4 && m.N % 4 == 0 && m.K >= KC && m.K % KC == 0);
  m.n_tiles = cdiv(m.N, columns);
  m.per = m.K / KC;
  return m;
}

// Stretches of the inner dimension: about WANT workgroups in all.
int cut(Product& m) {
  const int chunks = m.K / KC;
  m.per = cdiv(chunks, std::max(1, std::min(WANT / m.n_tiles, chunks)));
  return cdiv(chunks, m.per);
}

template <int NW, bool GLU>
void run(uint16_t* out, float* sums, const torch::Tensor& x,
         const torch::Tensor& w, const Product& m, int stretches) {
#define HELIX_GR(MI)                                                         \
  hipLaunchKernelGGL((gemm_rows_kernel<MI, NW, GLU>),                        \
                     dim3(m.n_tiles * stretches), dim3(NW * WAVE), 0,        \
                     at::hip::getCurrentHIPStream(), out, sums,              \
                     (const uint16_t*)x.data_ptr(),                          \
                     (const uint16_t*)w.data_ptr(), m)
  if (m.M <= 16) HELIX_GR(1);
  else if (m.M <= 32) HELIX_GR(2);
  else if (m.M <= 48) HELIX_GR(3);
  else HELIX_GR(4);
#undef HELIX_GR
}

}  // namespace

// Sums [stretches, M, N] for a reader that adds them up.
torch::Tensor gemm_rows_sums(torch::Tensor x, torch::Tensor w) {
  Product m = product_of(x, w, w.size(0), 64);
  const int stretches = cut(m);
  torch::Tensor sums = torch::empty({stretches, m.M, m.N},
                                    x.options().dtype(torch::kFloat32));
  run<4, false>(nullptr, sums.data_ptr<float>(), x, w, m, stretches);
  return sums;
}

void gemm_rows(torch::Tensor out, torch::Tensor x, torch::Tensor w,
               c10::optional<torch::Tensor> bias) {
  Product m = product_of(x, w, w.size(0), 64);
  TORCH_CHECK(out.is_contiguous() && out.scalar_type() == x.scalar_type() &&
              out.size(0) == m.M && out.size(1) == m.N &&
              (uintptr_t)out.data_ptr() % 8 == 0);
  if (bias.has_value()) {
    TORCH_CHECK(bias->scalar_type() == torch::kBFloat16 &&
                bias->is_contiguous() && bias->numel() == m.N);
    m.bias = (const uint16_t*)bias->data_ptr();
  }
  const int stretches = cut(m);
  uint16_t* o = (uint16_t*)out.data_ptr();
  if (stretches == 1) {
    run<4, false>(o, nullptr, x, w, m, 1);
    return;
  }
  torch::Tensor sums = torch::empty({stretches, m.M, m.N},
                                    x.options().dtype(torch::kFloat32));
  run<4, false>(nullptr, sums.data_ptr<float>(), x, w, m, stretches);
  const int64_t MN = (int64_t)m.M * m.N;
  hipLaunchKernelGGL(gemm_join_kernel, dim3((MN + 1023) / 1024), dim3(256), 0,
                     at::hip::getCurrentHIPStream(), o,
                     sums.data_ptr<float>(), m.bias, MN, m.N, stretches);
}

// out[M,N] = silu(x w[:N]^T) * (x w[N:]^T)
void gemm_rows_glu(torch::Tensor out, torch::Tensor x, torch::Tensor w) {
  TORCH_CHECK(w.size(0) % 2 == 0);
  Product m = product_of(x, w, w.size(0) / 2, 32);
  TORCH_CHECK(out.is_contiguous() && out.scalar_type() == x.scalar_type() &&
              out.size(0) == m.M && out.size(1) == m.N &&
              (uintptr_t)out.data_ptr() % 8 == 0);
  run<2, true>((uint16_t*)out.data_ptr(), nullptr, x, w, m, 1);
}
