// Product of a few rows with a large matrix: x[M,K] @ w[N,K]^T, bf16 or e4m3
// with fp32 sums, M <= 128.
//
// Bound by reading w once. A wave streams its columns of w straight into MFMA
// operands, a chunk of 512 bytes of the inner dimension ahead; x goes to LDS
// by direct loads, once for the columns of all waves, and only the rows there
// are. 16-byte piece p of row r lies at p ^ r % 16, so operands leave LDS without
// bank conflicts.
//
// Where the inner dimension is not cut, groups of columns begin at different
// chunks and go round: rows of w that are a power of two apart lie on the same
// channels, and workgroups that started together would all read those (us at 1
// row of 28672 x 4096 gated 44.9 -> 42.2, of 32000 x 4096 52.1 -> 46.0, of 128256 x
// 4096 180 -> 172; e4m3 gated 26.1 -> 22.6). Stretches have few chunks, and where
// to begin takes longer than it saves (6144 x 4096 11.4 -> 11.7).
//
// Narrow matrices leave CUs idle, so the inner dimension is cut into stretches
// until there are about as many workgroups as Shape wants (cut). Their sums
// (fp32, [stretch][M][N]) are added by whatever reads the result (norm,
// rotation), in order, or by a launch of their own; nothing is added with
// atomics.
//
// Gated feed-forward: a wave has 16 columns of the gate and the same 16 of the
// other half and writes silu(gate) * up; neither half goes to memory.
//
// us for N x K = 6144x4096, 4096x4096, 28672x4096, 4096x14336 (the sums left
// to the reader), library kernel in brackets:
//   M  1   11.2 (14.4)   8.0 (15.5)   42.2 (63.4)   22.1 (26.6)
//   M 16   12.7 (15.7)   8.6 (15.6)   42.7 (65.1)   23.6 (27.3)
//   M 32   14.4 (16.3)   9.3 (13.9)   46.8 (54.2)   24.9 (33.8)
//   M 64   17.6 (18.0)  12.2 (15.2)   54.0 (52.3)   31.9 (41.9)
// A language model's layers of up to 16 rows have kernels of their own
// (layer_rows.hip). Tiles (gemm_ring.h) have taken over bf16 from 17 rows on, but for the stretches
// of small products and of deep ones with few columns, up to 48 rows of wide
// matrices and up to 64 of vocabularies whose rows are 4 or 8 KB (_streams_pay in
// ops/__init__.py). From 65 rows on a wave has 32 columns, so that x is read from
// LDS half as often, chunks are half as long and 256 workgroups are enough:
//   M 128  20.0 (24.6)  15.5 (24.7)                   34.6 (73.9)
// Adding them up in a launch, with bias and GELU, takes 2.5 to 3 us more; up to
// 64 rows of small deep matrices of the encoder and the image model do so (8 of
// 768 x 3072 7.9, by tiles 8.9). The gated product replaces a launch of 4.5 us as
// well. Reading 28672 x 4096 at 42.2 us is 5.6 TB/s. Eight waves a workgroup,
// chunks half or twice as long, and for up to 64 rows 32 columns a wave and 256
// or 768 workgroups were each slower on most of these.
//
// e4m3 (weights with a scale per column, x with one per row) runs the scaled
// 16x16x128 instruction with unity scales; the scales meet the fp32 sums of
// every stretch. us at 32 rows of the four matrices, the tiles of gemm_fp8.hip
// in brackets: 9.4 (49.5), 7.4 (51.6), 27.4 (53.9), 16.0 (158).
#include "gemm_join.h"
#include "hybrid/tile.h"
#include <torch/extension.h>
#include <ATen/hip/HIPContext.h>
#include <c10/core/DeviceGuard.h>
#include <numeric>
#include <type_traits>

using namespace helix;

namespace {

// Up to 64 rows, and up to 128: bytes of a chunk's row, columns of a workgroup
// and the workgroups that stretches are cut for.
struct Shape {
  int chunk, columns, want;
};
constexpr Shape FEW{512, 64, 512}, MORE{256, 128, 256};
constexpr int UNITY = 0x7F7F7F7F;             // e8m0 2^0 in all four bytes

typedef int v8i __attribute__((ext_vector_type(8)));

struct Product {
  const uint16_t* bias;
  const float *xs, *ws;        // e4m3: scales of rows and columns
  int64_t row;                 // bytes of a row of x and w
  int M, N, n_tiles, chunks, per, want;       // per: chunks of a stretch
};

// Matrices of one width that the same rows are multiplied by, all in one launch
// (gemm_rows_many). ld: of the product that a matrix is a part of.
struct One {};
struct Many {
  static constexpr int MOST = 48;
  struct {
    const uint16_t *w, *bias;
    uint16_t* out;
    int64_t ld;
  } at[MOST];
};

__device__ __forceinline__ v8i join(u32x4 a, u32x4 b) {
  return v8i{(int)a[0], (int)a[1], (int)a[2], (int)a[3],
             (int)b[0], (int)b[1], (int)b[2], (int)b[3]};
}

// 16 MI rows, NW waves of 16 NI columns each, chunks of CB bytes. GLU (NI 2):
// columns n and N + n are a pair of a wave. TURN: one stretch, whose groups of
// columns begin apart.
template <int MI, int NI, int NW, int CB, bool GLU, bool F8, bool TURN,
          typename T>
__global__ __launch_bounds__(NW* WAVE, 2) void gemm_rows_kernel(
    uint16_t* __restrict__ out, float* __restrict__ sums,
    const char* __restrict__ x, const char* __restrict__ w, Product m, T many) {
  constexpr int CN = GLU ? 1 : NI;            // 16-column tiles of the output
  constexpr int TH = NW * WAVE, BM = MI * 16;
  constexpr int PR = CB / 16, XL = BM * PR / TH, U = CB / 64;
  static_assert(BM * PR % TH == 0, "x tile");
  __shared__ __attribute__((aligned(16))) char xl[2][BM * CB];
  const int stretch = blockIdx.x / m.n_tiles;
  int64_t ld = m.N;
  if constexpr (std::is_same_v<T, Many>) {
    const auto& one = many.at[stretch];
    w = (const char*)one.w;
    m.bias = one.bias;
    out = one.out;
    ld = one.ld;
  }
  const int tid = threadIdx.x, wid = tid / WAVE, lane = tid & (WAVE - 1);
  const int lo = lane & 15, hi = lane >> 4;
  const int n0 = (blockIdx.x % m.n_tiles * NW + wid) * 16 * CN;
  // Products in one stretch go by these bounds as well: with 0 and all chunks
  // written out the loop takes longer (8 rows of 28672 x 4096 gated 41.5 us in a
  // step, then 46.8).
  const bool many_of = std::is_same_v<T, Many>;
  const int c0 = many_of ? 0 : stretch * m.per;
  const int c1 = many_of ? m.chunks : min(m.chunks, c0 + m.per);
  // a lane's 16 bytes u of a chunk's row: bf16 has four lane groups to 64
  // bytes, e4m3 two pieces side by side to 128
  auto piece = [&](int u) {
    return F8 ? (u >> 1) * 8 + hi * 2 + (u & 1) : u * 4 + hi;
  };
  const char* wp[NI];
#pragma unroll
  for (int j = 0; j < NI; ++j)
    wp[j] = w + (GLU ? (int64_t)j * m.N + min(n0 + lo, m.N - 1)
                     : (int64_t)min(n0 + j * 16 + lo, m.N - 1)) * m.row;
  const char* xp[XL];
#pragma unroll
  for (int i = 0; i < XL; ++i) {
    const int e = i * TH + tid, r = e / PR, p = e % PR ^ (r & 15);
    xp[i] = x + min(r, m.M - 1) * m.row + p * 16;
  }
  const int from = TURN ? (int)(blockIdx.x % m.chunks) : 0;
  auto place = [&](int c) {
    if (TURN) c = c + from < m.chunks ? c + from : c + from - m.chunks;
    return c;
  };
  // rows past the last one stay as LDS was: no row's sums see another's
  auto load_x = [&](int at, int b) {
    const int c = place(at);
#pragma unroll
    for (int i = 0; i < XL; ++i)
      if ((i * TH + tid) / PR < m.M)
        __builtin_amdgcn_global_load_lds(
            (const __attribute__((address_space(1))) uint32_t*)(xp[i] + c * CB),
            (__attribute__((address_space(3))) uint32_t*)(
                xl[b] + (i * TH + wid * WAVE) * 16),
            16, 0, 0);
  };
  u32x4 wr[2][U][NI];
  auto load_w = [&](int at, int b) {
    const int c = place(at);
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int j = 0; j < NI; ++j)
        wr[b][u][j] = *reinterpret_cast<const u32x4*>(wp[j] + c * CB +
                                                      piece(u) * 16);
  };
  floatx4 acc[NI][MI];
#pragma unroll
  for (int j = 0; j < NI; ++j)
#pragma unroll
    for (int i = 0; i < MI; ++i) acc[j][i] = floatx4{0, 0, 0, 0};
  auto x_at = [&](int b, int i, int u) {
    return *reinterpret_cast<const u32x4*>(xl[b] + (i * 16 + lo) * CB +
                                           (piece(u) ^ lo) * 16);
  };
  auto step = [&](int c, int b) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (c + 1 < c1) {
      load_x(c + 1, b ^ 1);
      load_w(c + 1, b ^ 1);
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < U; u += F8 ? 2 : 1)
#pragma unroll
      for (int i = 0; i < MI; ++i) {
        if constexpr (F8) {
          const v8i xf = join(x_at(b, i, u), x_at(b, i, u + 1));
#pragma unroll
          for (int j = 0; j < NI; ++j)
            acc[j][i] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(
                join(wr[b][u][j], wr[b][u + 1][j]), xf, acc[j][i], 0, 0, 0,
                UNITY, 0, UNITY);
        } else {
          const u16x8 xf = __builtin_bit_cast(u16x8, x_at(b, i, u));
#pragma unroll
          for (int j = 0; j < NI; ++j)
            acc[j][i] = mfma16(__builtin_bit_cast(u16x8, wr[b][u][j]), xf,
                               acc[j][i]);
        }
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
#pragma unroll
  for (int i = 0; i < MI; ++i) {
    const int r = i * 16 + lo;
    if (r >= m.M) continue;
#pragma unroll
    for (int j = 0; j < CN; ++j) {
      const int n = n0 + j * 16 + hi * 4;
      if (n >= m.N) continue;
      if constexpr (F8) {
        const float xs = m.xs[r];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          acc[j][i][q] = acc[j][i][q] * xs * m.ws[n + q];
          if constexpr (GLU)
            acc[1][i][q] = acc[1][i][q] * xs * m.ws[m.N + n + q];
        }
      }
      float v[4];
      if constexpr (GLU) {
#pragma unroll
        for (int q = 0; q < 4; ++q)
          v[q] = acc[0][i][q] / (1.f + __expf(-acc[0][i][q])) * acc[1][i][q];
      } else {
        if (sums != nullptr) {
          *reinterpret_cast<floatx4*>(
              sums + ((int64_t)stretch * m.M + r) * m.N + n) = acc[j][i];
          continue;
        }
#pragma unroll
        for (int q = 0; q < 4; ++q)
          v[q] = acc[j][i][q] +
                 (m.bias != nullptr ? bf16_to_f32(m.bias[n + q]) : 0.f);
      }
      st_bf16x4(out + r * ld + n, v);
    }
  }
}

using OptT = c10::optional<torch::Tensor>;

// x_scale, w_scale: both (e4m3 bytes) or neither (bf16).
Product product_of(const torch::Tensor& x, const torch::Tensor& w,
                   const OptT& x_scale, const OptT& w_scale) {
  const bool f8 = x_scale.has_value();
  for (const auto& t : {x, w})
    TORCH_CHECK(t.dim() == 2 && t.is_contiguous() && t.is_cuda() &&
                t.device() == x.device() &&
                t.scalar_type() == (f8 ? torch::kUInt8 : torch::kBFloat16) &&
                (uintptr_t)t.data_ptr() % 16 == 0);
  Product m{};
  m.M = x.size(0);
  m.N = w.size(0);
  m.row = x.size(1) * (f8 ? 1 : 2);
  TORCH_CHECK(w.size(1) == x.size(1) && m.M >= 1 && m.M <= 128);
  const Shape s = m.M <= 64 ? FEW : MORE;
  TORCH_CHECK(m.N >= 4 && m.N % 4 == 0 && m.row > 0 && m.row % s.chunk == 0);
  TORCH_CHECK(w_scale.has_value() == f8);
  if (f8) {
    for (const auto& t : {*x_scale, *w_scale})
      TORCH_CHECK(t.is_contiguous() && t.scalar_type() == torch::kFloat32 &&
                  t.device() == x.device());
    TORCH_CHECK(x_scale->numel() == m.M && w_scale->numel() == w.size(0));
    m.xs = x_scale->data_ptr<float>();
    m.ws = w_scale->data_ptr<float>();
  }
  m.n_tiles = cdiv(m.N, s.columns);
  m.chunks = m.per = m.row / s.chunk;
  m.want = s.want;
  return m;
}

// Stretches of the inner dimension: about m.want workgroups in all, and at most
// 16, as the reader has to go through them (16 rows of 256 x 8192 with a norm:
// 32 stretches 16.6 us, 16 12.8, the library 11.9). Where a launch joins them,
// it takes a third chunk to pay for it (16 rows of 512 x 512, 2 chunks: 5.4 us
// in two stretches, 4.5 in one, the library 4.1).
int cut(Product& m, bool join) {
  const int most = join && m.chunks <= 2
                       ? 1 : std::min({m.want / m.n_tiles, m.chunks, 16});
  m.per = cdiv(m.chunks, std::max(1, most));
  return cdiv(m.chunks, m.per);
}

template <bool GLU, bool F8, bool TURN, typename T = One>
void run_as(uint16_t* out, float* sums, const torch::Tensor& x,
            const void* w, const Product& m, int stretches, T many = T{}) {
#define HELIX_GR(MI, NI, NW, CB)                                             \
  hipLaunchKernelGGL((gemm_rows_kernel<MI, NI, NW, CB, GLU, F8, TURN, T>),   \
                     dim3(m.n_tiles * stretches), dim3(NW * WAVE), 0,        \
                     at::hip::getCurrentHIPStream(), out, sums,              \
                     (const char*)x.data_ptr(), (const char*)w, m, many)
  constexpr int NI = GLU ? 2 : 1, NW = GLU ? 2 : 4;
  if (m.M <= 16) HELIX_GR(1, NI, NW, 512);
  else if (m.M <= 32) HELIX_GR(2, NI, NW, 512);
  else if (m.M <= 48) HELIX_GR(3, NI, NW, 512);
  else if (m.M <= 64) HELIX_GR(4, NI, NW, 512);
  else if constexpr (!GLU && std::is_same_v<T, One>) {
    if (m.M <= 96) HELIX_GR(6, 2, 4, 256);
    else HELIX_GR(8, 2, 4, 256);
  }
#undef HELIX_GR
}

template <bool GLU>
void run(uint16_t* out, float* sums, const torch::Tensor& x,
         const torch::Tensor& w, const Product& m, int stretches) {
#define HELIX_AS(F8)                                                         \
  if (GLU || stretches == 1)                                                 \
    return run_as<GLU, F8, true>(out, sums, x, w.data_ptr(), m, stretches);  \
  if constexpr (!GLU)                                                        \
    run_as<GLU, F8, false>(out, sums, x, w.data_ptr(), m, stretches)
  if (m.xs != nullptr) {
    HELIX_AS(true);
  } else {
    HELIX_AS(false);
  }
#undef HELIX_AS
}

torch::Tensor sums_for(const torch::Tensor& x, const Product& m,
                       int stretches) {
  return torch::empty({stretches, m.M, m.N},
                      x.options().dtype(torch::kFloat32));
}

void check_out(const torch::Tensor& out, const torch::Tensor& x,
               const Product& m) {
  TORCH_CHECK(out.is_contiguous() && out.dim() == 2 &&
              out.device() == x.device() &&
              out.scalar_type() == torch::kBFloat16 && out.size(0) == m.M &&
              out.size(1) == m.N && (uintptr_t)out.data_ptr() % 8 == 0);
}

}  // namespace

// Sums [stretches, M, N] for a reader that adds them up.
torch::Tensor gemm_rows_sums(torch::Tensor x, torch::Tensor w, OptT x_scale,
                             OptT w_scale) {
  const c10::DeviceGuard on(x.device());
  Product m = product_of(x, w, x_scale, w_scale);
  const int stretches = cut(m, false);
  torch::Tensor sums = sums_for(x, m, stretches);
  run<false>(nullptr, sums.data_ptr<float>(), x, w, m, stretches);
  return sums;
}

void gemm_rows(torch::Tensor out, torch::Tensor x, torch::Tensor w, OptT bias,
               OptT x_scale, OptT w_scale, bool gelu) {
  const c10::DeviceGuard on(x.device());
  Product m = product_of(x, w, x_scale, w_scale);
  check_out(out, x, m);
  if (bias.has_value()) {
    TORCH_CHECK(bias->scalar_type() == torch::kBFloat16 &&
                bias->is_contiguous() && bias->numel() == m.N &&
                bias->device() == x.device());
    m.bias = (const uint16_t*)bias->data_ptr();
  }
  const int stretches = cut(m, !gelu);
  uint16_t* o = (uint16_t*)out.data_ptr();
  if (stretches == 1 && !gelu) {
    run<false>(o, nullptr, x, w, m, 1);
    return;
  }
  torch::Tensor sums = sums_for(x, m, stretches);
  run<false>(nullptr, sums.data_ptr<float>(), x, w, m, stretches);
  const int64_t MN = (int64_t)m.M * m.N;
  hipLaunchKernelGGL(gemm_join_kernel, dim3((MN + 1023) / 1024), dim3(256), 0,
                     at::hip::getCurrentHIPStream(), o,
                     sums.data_ptr<float>(), m.bias, MN, m.N, stretches,
                     gelu);
}

// out[M,N] = silu(x w[:N]^T) * (x w[N:]^T)
void gemm_rows_glu(torch::Tensor out, torch::Tensor x, torch::Tensor w,
                   OptT x_scale, OptT w_scale) {
  const c10::DeviceGuard on(x.device());
  Product m = product_of(x, w, x_scale, w_scale);
  TORCH_CHECK(m.M <= 64 && m.N % 8 == 0);
  m.N /= 2;                                   // 32 columns of a workgroup
  m.n_tiles = cdiv(m.N, 32);
  check_out(out, x, m);
  run<true>((uint16_t*)out.data_ptr(), nullptr, x, w, m, 1);
}

// x w^T + bias for every w, in launches of up to Many::MOST matrices: cut to the
// largest width that divides all of theirs. Empty, and nothing done, for other
// forms of operands than the kernel reads. Bound by reading the matrices, where
// one launch each is bound by its start: 8 rows of 12 x 6144 x 1024 and 2048 x 1024
// 91 us -> 31.
std::vector<torch::Tensor> gemm_rows_many(torch::Tensor x,
                                          std::vector<torch::Tensor> ws,
                                          std::vector<OptT> biases) {
  std::vector<torch::Tensor> outs;
  auto reads = [&](const torch::Tensor& t, int64_t to) {
    return t.scalar_type() == torch::kBFloat16 && t.device() == x.device() &&
           t.is_contiguous() && (uintptr_t)t.data_ptr() % to == 0;
  };
  if (!x.is_cuda() || x.dim() != 2 || !reads(x, 16) || x.size(0) < 1 ||
      x.size(0) > 64 || x.size(1) < 1 || x.size(1) * 2 % FEW.chunk != 0 ||
      ws.size() != biases.size() || ws.empty())
    return outs;
  int64_t width = 0;
  for (size_t i = 0; i < ws.size(); ++i) {
    if (ws[i].dim() != 2 || ws[i].size(1) != x.size(1) || !reads(ws[i], 16) ||
        (biases[i].has_value() &&
         (biases[i]->dim() != 1 || biases[i]->size(0) != ws[i].size(0) ||
          !reads(*biases[i], 2))))
      return outs;
    width = std::gcd(width, ws[i].size(0));
  }
  if (width == 0 || width % FEW.columns != 0 || width > 1 << 20) return outs;
  const c10::DeviceGuard on(x.device());
  Product m{};
  m.M = x.size(0);
  m.N = width;
  m.row = x.size(1) * 2;
  m.n_tiles = width / FEW.columns;
  m.chunks = m.per = m.row / FEW.chunk;
  Many many;
  int n = 0;
  auto launch = [&] {
    if (n > 0)
      run_as<false, false, true, Many>(nullptr, nullptr, x, nullptr, m, n, many);
    n = 0;
  };
  for (size_t i = 0; i < ws.size(); ++i) {
    const int64_t N = ws[i].size(0);
    outs.push_back(torch::empty({m.M, N}, x.options()));
    for (int64_t c = 0; c < N; c += width) {
      auto& one = many.at[n++];
      one.w = (const uint16_t*)ws[i].data_ptr() + c * x.size(1);
      one.bias = biases[i].has_value()
                     ? (const uint16_t*)biases[i]->data_ptr() + c : nullptr;
      one.out = (uint16_t*)outs[i].data_ptr() + c;
      one.ld = N;
      if (n == Many::MOST) launch();
    }
  }
  launch();
  return outs;
}
