// The gated half of a feed-forward block for more rows than gemm_rows.hip
// takes: out[M,N] = silu(x w[:N]^T) * (x w[N:]^T), bf16.
//
// The kernel of gemm_ring.h with as many columns of the gate as of the other
// factor in a wave: both halves of a product meet in registers and are not
// rounded before, and neither is written, read and written again by a launch of
// its own (8192 rows of 2 x 14336: 125 us of 1395). That form knows no stretches:
// where its tiles leave CUs idle both halves are cut along the inner dimension
// and meet in a launch that adds the stretches up. us of one launch and of both:
// 80 x 2 x 1024 x 8192 43 and 15 (8 stretches), 512 x 2 x 512 x 16384 90 and 30,
// 100 x 2 x 2048 x 14336 79 and 37, 1024 x 2 x 4224 x 14592 254 and 259. Of 555
// sizes 4 take over 5% longer than in one launch, all together 0.84 of the time.
#include "gemm_ring.h"
#include <c10/core/DeviceGuard.h>

using namespace helix;

// of gemm_bf16.hip
torch::Tensor gemm_bf16_sums(torch::Tensor x, torch::Tensor w, int64_t tile,
                             int64_t stretches);
std::tuple<int64_t, int64_t, double, int64_t> gemm_bf16_plan(
    int64_t M, int64_t N, int64_t K, bool gelu, bool sums, int64_t cus,
    double below);

namespace {

#define HELIX_RING_GATED(TILE)                                               \
  TILE(1, 4) TILE(2, 4) TILE(3, 4) TILE(4, 8) TILE(5, 4) TILE(5, 8)           \
  TILE(6, 4) TILE(7, 8) TILE(8, 8)
#define HELIX_TILE(MI, NI) {MI, NI},
constexpr int GATED_TILES[][2] = {HELIX_RING_GATED(HELIX_TILE)};
#undef HELIX_TILE

// out[M,N] of sums [stretches][M][2 N], 4 columns a thread. Bound by their
// bytes and a launch.
__global__ __launch_bounds__(256) void glu_join_kernel(
    uint16_t* __restrict__ out, const float* __restrict__ sums, int M, int N,
    int stretches, Divide by_row) {
  const uint32_t i = blockIdx.x * 256 + threadIdx.x;
  const int row = by_row(i);
  if (row >= M) return;
  const int c = (int)(i - (uint32_t)row * (N / 4)) * 4;
  const float* p = sums + (int64_t)row * 2 * N + c;
  f32x4 g = {0, 0, 0, 0}, u = {0, 0, 0, 0};
#pragma unroll 4
  for (int s = 0; s < stretches; ++s, p += (int64_t)M * 2 * N) {
    g += *reinterpret_cast<const f32x4*>(p);
    u += *reinterpret_cast<const f32x4*>(p + N);
  }
  float v[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) v[j] = silu_f32(g[j]) * u[j];
  st_bf16x4(out + (int64_t)row * N + c, v);
}

// Tile of one launch, or tile and number of stretches of two. The second
// launch takes 4 us beside what it reads.
struct GluPlan {
  int tile, stretches;
  double us;
};
GluPlan plan_glu(const Ring& m, int cus) {
  const RingPlan one = ring_plan(m, GATED, GATED_TILES, 1, 1, cus);
  GluPlan p{10 * one.tile.mi + one.tile.ni, 0, one.us};
  if (m.N <= 1 << 19 && (int64_t)m.M * (m.N / 4) < 1 << 30) {
    const auto two = gemm_bf16_plan(m.M, 2 * m.N, m.K, false, true, cus,
                                    one.us - 4);
    if (std::get<0>(two) != 0)
      p = GluPlan{(int)std::get<0>(two), (int)std::get<1>(two),
                  std::get<2>(two)};
  }
  return p;
}

RingCut cut_glu(const Ring& m, int cus, double us) {
  return ring_cut(m, GATED, GATED_TILES, cus, ring_cut_below(us, 0.02));
}

void run_glu(const Ring& m, const RingTile& t, int cus) {
#define HELIX_RUN(MI, NI)                                                    \
  if (t.mi == MI && t.ni == NI) return ring_run<MI, NI, GATED>(m, 1, cus);
  HELIX_RING_GATED(HELIX_RUN)
#undef HELIX_RUN
  TORCH_CHECK(false, "no tile of ", 32 * t.mi, " x ", 16 * t.ni);
}

}  // namespace

// As gemm_bf16_cut, of one launch.
std::tuple<bool, int64_t, int64_t, int64_t, double> gemm_bf16_glu_cut(
    int64_t M, int64_t N, int64_t K, int64_t cus) {
  Ring m{};
  m.M = M;
  m.N = N;
  m.K = K;
  TORCH_CHECK(M > 0 && N > 0 && K > 0 && cus > 0 && M <= INT32_MAX &&
              ring_fits(m, GATED), "a product of tiles");
  const GluPlan p = plan_glu(m, cus);
  const RingCut c = p.stretches > 0 ? RingCut{} : cut_glu(m, cus, p.us);
  return {c.rows, c.at, 10 * c.first.mi + c.first.ni, 10 * c.rest.mi + c.rest.ni,
          c.us};
}

std::tuple<int64_t, int64_t> gemm_bf16_glu_plan(int64_t M, int64_t N,
                                                         int64_t K,
                                                         int64_t cus) {
  Ring m{};
  m.M = M;
  m.N = N;
  m.K = K;
  TORCH_CHECK(M > 0 && N > 0 && K > 0 && cus > 0 && M <= INT32_MAX &&
              ring_fits(m, GATED), "a product of tiles");
  const GluPlan p = plan_glu(m, cus);
  return {p.tile, p.stretches};
}

// tile: 32 * (tile / 10) rows and 16 * (tile % 10) columns, 0 the one that
// takes least time.
void gemm_bf16_glu(torch::Tensor out, torch::Tensor x, torch::Tensor w,
                   int64_t tile) {
  const c10::DeviceGuard on(x.device());
  for (const auto& t : {x, w, out})
    TORCH_CHECK(t.dim() == 2 && t.is_contiguous() && t.is_cuda() &&
                t.device() == x.device() &&
                t.scalar_type() == torch::kBFloat16 &&
                (uintptr_t)t.data_ptr() % 16 == 0,
                "packed bf16 matrices on one GPU");
  Ring m{};
  m.M = x.size(0);
  m.K = m.stretch = x.size(1);
  m.N = w.size(0) / 2;
  m.x = (const uint16_t*)x.data_ptr();
  m.w = (const uint16_t*)w.data_ptr();
  m.out = (uint16_t*)out.data_ptr();
  TORCH_CHECK(w.size(1) == m.K && w.size(0) % 2 == 0 && m.M > 0 && m.N > 0 &&
              m.K > 0 && out.size(0) == m.M && out.size(1) == m.N,
              "out is [M, N], w [2 N, K]");
  TORCH_CHECK(ring_fits(m, GATED), "columns are a multiple of 8, and K of 64");
  const int cus = ring_cus();
  GluPlan plan{(int)tile, 0, 0};
  if (tile == 0) plan = plan_glu(m, cus);
  if (plan.stretches > 0) {
    const torch::Tensor sums = gemm_bf16_sums(x, w, plan.tile, plan.stretches);
    const int64_t parts = (int64_t)m.M * (m.N / 4);
    hipLaunchKernelGGL(glu_join_kernel, dim3((parts + 255) / 256), dim3(256), 0,
                       at::hip::getCurrentHIPStream(), m.out,
                       sums.data_ptr<float>(), m.M, m.N, (int)sums.size(0),
                       Divide(m.N / 4));
    return;
  }
  const RingCut cut = tile == 0 ? cut_glu(m, cus, plan.us) : RingCut{};
  if (cut.at > 0) {
    Ring a, b;
    m.ld = m.up = m.N;
    ring_parts(m, cut, a, b);
    run_glu(a, cut.first, cus);
    return run_glu(b, cut.rest, cus);
  }
  run_glu(m, RingTile{plan.tile / 10, plan.tile % 10, 0}, cus);
}
