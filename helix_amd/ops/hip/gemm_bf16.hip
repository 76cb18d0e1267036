// bf16 MFMA GEMM for gfx950: out[M,N] = act(x[M,K] @ w[N,K]^T + bias).
//
// The encoder's and the image model's projections (act: none or GELU, tanh),
// and Llama's of more than a few rows; deep ones of few tiles are cut into
// stretches of the inner dimension that a later reader adds up (fp32
// [stretch][M][N]).
//
// gemm_ring.h has the kernel, its times and what bounds it. Here are its tiles
// and the rule that chooses one, and the kernel for what it does not take
// (matrices beyond its offsets) or not as fast (small_tiles).
#include "gemm_join.h"
#include "gemm_ring.h"
#include <c10/core/DeviceGuard.h>

using namespace helix;

namespace {

constexpr int GROUP = 4;                      // tiles of rows

struct Gemm {
  const uint16_t* bias;
  int M, N, K, m_tiles, n_tiles, gelu;
};

__device__ __forceinline__ float finish(float v, float b, int gelu) {
  v += b;
  return gelu ? gelu_tanh_f32(v) : v;
}

struct Place {
  int m0, n0;
};
__device__ __forceinline__ Place place(const Gemm& m, int BM, int BN) {
  const int at = xcd_chunk(blockIdx.x, gridDim.x);
  const int first = at / (GROUP * m.n_tiles) * GROUP;
  const int rows = min(GROUP, m.m_tiles - first);
  const int in = at % (GROUP * m.n_tiles);
  Place p;
  p.m0 = (first + in % rows) * BM;
  p.n0 = in / rows * BN;
  return p;
}

// Piece p of a row of 64 elements lies at p ^ cross(row).
__device__ __forceinline__ int cross(int r) { return r >> 1 & 7; }

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
                (e % PR ^ cross(r)) * 8;
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
__device__ __forceinline__ void store(const Gemm& m, uint16_t* out, int row0,
                                      int col0,
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

  xs.load(0, lds);
  ws.load(0, lds + BM * BK);
  for (int k = 0, cur = 0; k < m.K; k += BK, cur ^= 1) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (k + BK < m.K) {
      xs.load(k + BK, lds + (cur ^ 1) * HALF);
      ws.load(k + BK, lds + (cur ^ 1) * HALF + BM * BK);
    }
    const uint16_t* xl = lds + cur * HALF + (wr * MI * 16 + lo) * BK;
    const uint16_t* wl = lds + cur * HALF + (BM + wc * NI * 16 + lo) * BK;
#pragma unroll
    for (int kk = 0; kk < BK / 32; ++kk) {
      const int piece = ((kk * 4 + hi) ^ cross(lo)) * 8;
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
  store<MI, NI>(m, out, p.m0 + wr * MI * 16, p.n0 + wc * NI * 16, acc);
}

template <int BM, int BN, int WM, int WN>
void run_tiles(Gemm m, uint16_t* out, const uint16_t* x, const uint16_t* w) {
  m.m_tiles = cdiv(m.M, BM);
  m.n_tiles = cdiv(m.N, BN);
  hipLaunchKernelGGL((gemm_tiles_kernel<BM, BN, WM, WN>),
                     dim3(m.m_tiles * m.n_tiles), dim3(WM * WN * WAVE),
                     2 * (BM + BN) * 64 * 2, at::hip::getCurrentHIPStream(),
                     out, x, w, m);
}

// Of 23 tiles of 64 to 256 rows and columns these are needed for times within
// 1% of the best of all (150 sizes, see ring_us).
#define HELIX_RING_ROWS(TILE)                                                \
  TILE(2, 2) TILE(3, 4) TILE(4, 2) TILE(4, 8) TILE(5, 2) TILE(5, 4)          \
  TILE(5, 6) TILE(5, 8) TILE(6, 4) TILE(6, 6) TILE(7, 8) TILE(8, 8)
#define HELIX_RING_SUMS(TILE)                                                \
  TILE(2, 2) TILE(2, 4) TILE(3, 4) TILE(4, 2) TILE(4, 4) TILE(4, 8)          \
  TILE(5, 4) TILE(5, 8) TILE(8, 8)
// Any columns, us by the tiles of a workgroup each that had these before -> now:
// 8192 x 4092 x 4096 391 -> 198, 16600 x 3002 x 1024 198 -> 141, 2304 x 766 x
// 3072 30 -> 21, 100 x 1020 x 4096 32 -> 10 (8 stretches), 777 x 4095 x 4096 58
// -> 40.
#define HELIX_RING_ANY(TILE)                                                 \
  TILE(2, 2) TILE(4, 2) TILE(4, 4) TILE(5, 4) TILE(4, 8) TILE(8, 8)
#define HELIX_TILE(MI, NI) {MI, NI},
constexpr int ROWS_TILES[][2] = {HELIX_RING_ROWS(HELIX_TILE)};
constexpr int ANY_TILES[][2] = {HELIX_RING_ANY(HELIX_TILE)};
constexpr int SUMS_TILES[][2] = {HELIX_RING_SUMS(HELIX_TILE)};
#undef HELIX_TILE

void run_ring(const Ring& m, const RingTile& t, int cus) {
#define HELIX_RUN(MI, NI)                                                    \
  if (t.mi == MI && t.ni == NI) return ring_run<MI, NI, ROWS>(m, 1, cus);
  HELIX_RING_ROWS(HELIX_RUN)
#undef HELIX_RUN
  TORCH_CHECK(false, "no tile of ", 32 * t.mi, " x ", 32 * t.ni);
}

void run_ring_any(const Ring& m, const RingTile& t, int cus) {
#define HELIX_RUN(MI, NI)                                                    \
  if (t.mi == MI && t.ni == NI) return ring_run<MI, NI, ANY>(m, 1, cus);
  HELIX_RING_ANY(HELIX_RUN)
#undef HELIX_RUN
  TORCH_CHECK(false, "no tile of ", 32 * t.mi, " x ", 32 * t.ni);
}

void run_ring_sums(const Ring& m, const RingTile& t, int stretches, int cus) {
#define HELIX_RUN(MI, NI)                                                    \
  if (t.mi == MI && t.ni == NI)                                              \
    return ring_run<MI, NI, SUMS>(m, stretches, cus);
  HELIX_RING_SUMS(HELIX_RUN)
#undef HELIX_RUN
  TORCH_CHECK(false, "no tile of ", 32 * t.mi, " x ", 32 * t.ni, " for sums");
}

RingPlan plan_rows(const Ring& m, int cus) {
  return ring_plan(m, ROWS, ROWS_TILES, 1, 1, cus);
}
RingPlan plan_any(const Ring& m, int cus) {
  return ring_plan(m, ANY, ANY_TILES, 1, 1, cus);
}
RingPlan plan_sums(const Ring& m, int from, int cus, double below = 1e30) {
  return ring_plan(m, SUMS, SUMS_TILES, from, std::min(8, m.K / RING_STEP), cus,
                   below);
}

RingCut cut_rows(const Ring& m, int cus, double us) {
  return ring_cut(m, ROWS, ROWS_TILES, cus, ring_cut_below(us, 0.03));
}

// The last stretch may be shorter; there are as many as have something to do.
int cut(Ring& m, int stretches) {
  m.stretch = cdiv(m.K / 64, stretches) * 64;
  return cdiv(m.K, m.stretch);
}

torch::Tensor sums_of(const torch::Tensor& x, Ring& m, const RingTile& t,
                      int stretches, int cus) {
  stretches = cut(m, stretches);
  torch::Tensor sums = torch::empty({stretches, m.M, m.N},
                                    x.options().dtype(torch::kFloat32));
  m.sums = sums.data_ptr<float>();
  run_ring_sums(m, t, stretches, cus);
  return sums;
}

// Whether a product whose rows are stored in parts goes by workgroups of a tile
// each. Their stores overlap with other workgroups' work, which pays where
// columns go one by one and the inner dimension is short, and there is less of
// them to start. us by persistent tiles and by these: 16600 x 3001 x 1024 195
// and 172, 8192 x 765 x 3072 51 and 57, 2304 x 2303 x 768 27 and 27; 64 x 1021 x
// 1024 8.2 and 6.9, 100 of it 8.3 and 8.4; 20 x 100 x 768 6.4 and 5.7, 100 of it
// 6.6 and 6.7, 20 x 3002 x 1024 7.6 and 10.3, 200 x 258 x 256 5.4 and 5.1.
bool small_tiles(const Ring& m) {
  const int64_t work = (int64_t)m.N * m.K;
  if (m.unit == 1)
    return (m.K < 2048 && m.M > 512) || work <= (m.M <= 64 ? 5 << 18 : 5 << 17);
  return m.unit < 8 && work <= (m.M <= 64 ? 1 << 20 : 1 << 17);
}

Ring ring_of(const torch::Tensor& x, const torch::Tensor& w) {
  Ring m{};
  m.M = x.size(0);
  m.K = m.stretch = x.size(1);
  m.N = w.size(0);
  m.x = (const uint16_t*)x.data_ptr();
  m.w = (const uint16_t*)w.data_ptr();
  return m;
}

}  // namespace

// tile: that one of 32 * (tile / 10) rows and 32 * (tile % 10) columns, 0 the
// one that takes least time.
void gemm_bf16(torch::Tensor out, torch::Tensor x, torch::Tensor w,
               c10::optional<torch::Tensor> bias, int64_t act, int64_t tile) {
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
  const c10::DeviceGuard on(x.device());
  // Columns that would be stored one by one, for many rows of a long inner
  // dimension: a copy costs less (4600 x 2304 x 2048 70 us, with it 60).
  if (tile == 0 && (uintptr_t)out.data_ptr() % 4 != 0 && m.N % 4 == 0 &&
      m.K >= 2048 && m.M > 512) {
    torch::Tensor t = torch::empty_like(out);
    gemm_bf16(t, x, w, bias, act, 0);
    out.copy_(t);
    return;
  }
  // tiles are loaded 16 bytes at a time
  if ((uintptr_t)x.data_ptr() % 16 != 0) x = x.clone();
  if ((uintptr_t)w.data_ptr() % 16 != 0) w = w.clone();
  uint16_t* o = (uint16_t*)out.data_ptr();
  Ring r = ring_of(x, w);
  const bool whole = m.N % 8 == 0 && (uintptr_t)o % 16 == 0;
  r.unit = whole ? 8 : 4;
  while (r.unit > 1 && (m.N % r.unit != 0 || (uintptr_t)o % (2 * r.unit) != 0))
    r.unit /= 2;
  if (ring_fits(r, whole ? ROWS : ANY) && (tile != 0 || !small_tiles(r))) {
    if (whole && m.bias != nullptr && (uintptr_t)m.bias % 16 != 0) {
      bias = bias->clone();
      m.bias = (const uint16_t*)bias->data_ptr();
    }
    r.out = o;
    r.gelu = m.gelu;
    const int cus = ring_cus();
    if (tile != 0) {
      r.bias = m.bias;
      const RingTile t{(int)tile / 10, (int)tile % 10, 0};
      return whole ? run_ring(r, t, cus) : run_ring_any(r, t, cus);
    }
    // A launch that joins stretches takes 3 us more than what it reads (with
    // it, and whole: 300 x 1024 x 4096 13 and 18, 288 x 768 x 3072 9.6 and 12.1;
    // 2304 x 768 x 3072 20 and 18).
    const RingPlan rows = whole ? plan_rows(r, cus) : plan_any(r, cus);
    RingPlan sums;
    if (m.N % 4 == 0) sums = plan_sums(r, 2, cus, rows.us - 4);
    if (sums.tile.mi == 0) {
      r.bias = m.bias;
      const RingCut cut = whole ? cut_rows(r, cus, rows.us) : RingCut{};
      if (cut.at > 0) {
        Ring a, b;
        r.ld = r.N;
        ring_parts(r, cut, a, b);
        run_ring(a, cut.first, cus);
        return run_ring(b, cut.rest, cus);
      }
      return whole ? run_ring(r, rows.tile, cus)
                   : run_ring_any(r, rows.tile, cus);
    }
    const torch::Tensor t = sums_of(x, r, sums.tile, sums.stretches, cus);
    const int64_t MN = (int64_t)m.M * m.N;
    hipLaunchKernelGGL(gemm_join_kernel, dim3((MN + 1023) / 1024), dim3(256),
                       0, at::hip::getCurrentHIPStream(), o,
                       t.data_ptr<float>(), m.bias, MN, m.N, (int)t.size(0),
                       m.gelu != 0);
    return;
  }
  TORCH_CHECK(tile == 0, "not a product of tiles");
  const uint16_t* xp = (const uint16_t*)x.data_ptr();
  const uint16_t* wp = (const uint16_t*)w.data_ptr();
  if ((int64_t)cdiv(m.M, 128) * cdiv(m.N, 128) >= 256)
    run_tiles<128, 128, 2, 4>(m, o, xp, wp);
  else if (m.M > 64) run_tiles<64, 64, 2, 2>(m, o, xp, wp);
  else run_tiles<32, 64, 2, 2>(m, o, xp, wp);
}

// Sums [stretches, M, N] for a reader that adds them up, those that take least
// time with it. stretches: that many, by the tile of 32 * (tile / 10) rows and
// 32 * (tile % 10) columns.
torch::Tensor gemm_bf16_sums(torch::Tensor x, torch::Tensor w, int64_t tile,
                             int64_t stretches) {
  const c10::DeviceGuard on(x.device());
  for (const auto& t : {x, w})
    TORCH_CHECK(t.dim() == 2 && t.is_contiguous() && t.is_cuda() &&
                t.device() == x.device() &&
                t.scalar_type() == torch::kBFloat16 &&
                (uintptr_t)t.data_ptr() % 16 == 0);
  Ring m = ring_of(x, w);
  TORCH_CHECK(w.size(1) == m.K && m.K > 0 && m.K % 64 == 0 && m.M >= 1 &&
              m.N >= 4 && m.N % 4 == 0 && (stretches > 0 || tile == 0));
  TORCH_CHECK(ring_fits(m, SUMS), "a product of more than the offsets reach");
  const int cus = ring_cus();
  if (stretches > 0)
    return sums_of(x, m, RingTile{(int)tile / 10, (int)tile % 10, 0},
                   (int)std::min<int64_t>(stretches, m.K / 64), cus);
  const RingPlan p = plan_sums(m, 1, cus);
  return sums_of(x, m, p.tile, p.stretches, cus);
}

// x @ w^T for a layer norm that adds it to something: rows with the bias [M, N], or
// two to four stretches [n, M, N] (fp32) without it where those take less with
// their reader, which would have read rows; half a microsecond is left to rows. The
// norm has a wave to a row, so more stretches cost it 0.5 us each. us with the
// norm, rows and stretches: 100 x 1024 x 4096 13.9 and 13.4, 288 16.6 and 14.8, 576
// 19.8 and 17.5, 1152 24.2 and 21.2, 2000 26.3 and 27.9; 400 x 768 x 3072 15.9 and
// 14.2. Up to 64 rows, and where the inner dimension is not deep, it is 0.5 us at
// most (60 x 1024 x 4096 13.8 and 13.1, 200 x 768 x 768 10.2 and 9.9).
torch::Tensor gemm_bf16_summand(torch::Tensor x, torch::Tensor w,
                                torch::Tensor bias) {
  TORCH_CHECK(x.dim() == 2 && w.dim() == 2 && x.is_cuda() &&
              x.scalar_type() == torch::kBFloat16, "bf16 matrices on the GPU");
  const c10::DeviceGuard on(x.device());
  Ring m = ring_of(x, w);
  if (m.M > 64 && m.N > 0 && m.K >= 2 * m.N && w.size(1) == m.K &&
      m.N % 8 == 0 && (int64_t)m.M * m.N <= 4 << 20 && ring_fits(m, SUMS) &&
      ring_fits(m, ROWS) && x.is_contiguous() && w.is_contiguous() &&
      w.scalar_type() == torch::kBFloat16 && w.device() == x.device() &&
      (uintptr_t)m.x % 16 == 0 && (uintptr_t)m.w % 16 == 0) {
    const int cus = ring_cus();
    const RingPlan rows = plan_rows(m, cus);
    const RingPlan sums = ring_plan(m, SUMS, SUMS_TILES, 2,
                                    std::min(4, m.K / RING_STEP), cus);
    // rows in stretches that a launch of 4 us joins
    if (sums.us + 0.5 <=
        std::min(rows.us, sums.us + 4) + 2. * m.M * m.N / 4.5e6)
      return sums_of(x, m, sums.tile, sums.stretches, cus);
  }
  torch::Tensor out = torch::empty({x.size(0), w.size(0)}, x.options());
  gemm_bf16(out, x, w, bias, 0, 0);
  return out;
}

// What gemm_bf16 (sums false) and gemm_bf16_sums do with a product on so many
// CUs: tile, stretches, us with the reader of those, and how many times were
// worked out to find them. Tile 0: no sums take less than `below`.
std::tuple<int64_t, int64_t, double, int64_t> gemm_bf16_plan(
    int64_t M, int64_t N, int64_t K, bool gelu, bool sums, int64_t cus,
    double below) {
  Ring m{};
  m.M = M;
  m.N = N;
  m.K = K;
  m.gelu = gelu;
  TORCH_CHECK(M > 0 && N > 0 && K > 0 && cus > 0 && M <= INT32_MAX &&
              ring_fits(m, sums ? SUMS : ANY), "a product of tiles");
  RingPlan best, p;
  if (!sums) best = N % 8 == 0 ? plan_rows(m, cus) : plan_any(m, cus);
  if (N % 4 == 0)
    p = sums ? plan_sums(m, 1, cus, below) : plan_sums(m, 2, cus, best.us - 4);
  p.weighed += best.weighed;
  if (!sums && p.tile.mi == 0) best.weighed = p.weighed, p = best;
  return {10 * p.tile.mi + p.tile.ni, p.stretches, p.us, p.weighed};
}

// How gemm_bf16 cuts a product that is not in stretches: whether by rows, behind
// how many (0: not at all), the tiles of both parts and us.
std::tuple<bool, int64_t, int64_t, int64_t, double> gemm_bf16_cut(
    int64_t M, int64_t N, int64_t K, bool gelu, int64_t cus) {
  Ring m{};
  m.M = M;
  m.N = N;
  m.K = K;
  m.gelu = gelu;
  TORCH_CHECK(M > 0 && N > 0 && K > 0 && cus > 0 && M <= INT32_MAX &&
              ring_fits(m, ROWS), "a product of tiles");
  const RingCut c = cut_rows(m, cus, plan_rows(m, cus).us);
  return {c.rows, c.at, 10 * c.first.mi + c.first.ni, 10 * c.rest.mi + c.rest.ni,
          c.us};
}

// Places along the inner dimension that a workgroup orders in so many steps, of
// items from k[2 i] to k[2 i + 1], `turn` after their start, and after the last
// of them.
std::vector<int64_t> gemm_ring_places(std::vector<int64_t> k, int64_t steps,
                                      int64_t turn) {
  RingAt at;
  size_t item = 0;
  auto next = [&] {
    at.close();
    if (item + 1 < k.size()) at.open((int)k[item], (int)k[item + 1], (int)turn);
    item += 2;
  };
  next();
  std::vector<int64_t> places;
  for (int64_t i = 0; i < steps; ++i) {
    places.push_back(at.k);
    if (at.step()) next();
  }
  return places;
}
