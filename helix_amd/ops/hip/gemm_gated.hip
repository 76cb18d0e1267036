// The gated half of a feed-forward block for more rows than gemm_rows.hip
// takes: out[M,N] = silu(x w[:N]^T) * (x w[N:]^T), bf16.
//
// The kernel of gemm_ring.h with as many columns of the gate as of the other
// factor in a wave: both halves of a product meet in registers and are not
// rounded before, and neither is written, read and written again by a launch of
// its own (8192 rows of 2 x 14336: 125 us of 1395).
#include "gemm_ring.h"
#include <c10/core/DeviceGuard.h>

using namespace helix;

namespace {

#define HELIX_RING_GATED(TILE)                                               \
  TILE(1, 4) TILE(2, 4) TILE(3, 4) TILE(4, 8) TILE(5, 4) TILE(5, 8)           \
  TILE(6, 4) TILE(7, 8) TILE(8, 8)
#define HELIX_TILE(MI, NI) {MI, NI},
constexpr int GATED_TILES[][2] = {HELIX_RING_GATED(HELIX_TILE)};
#undef HELIX_TILE

}  // namespace

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
  const RingTile best =
      tile == 0 ? ring_plan(m, GATED, GATED_TILES, 1, 1, cus).tile
                : RingTile{(int)tile / 10, (int)tile % 10, 0};
#define HELIX_RUN(MI, NI)                                                    \
  if (best.mi == MI && best.ni == NI)                                        \
    return ring_run<MI, NI, GATED>(m, 1, cus);
  HELIX_RING_GATED(HELIX_RUN)
#undef HELIX_RUN
  TORCH_CHECK(false, "no tile of ", 32 * best.mi, " x ", 16 * best.ni);
}
