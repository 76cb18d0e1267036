// Prompt attention, see attn_prefill.h.
#include "attn_prefill.h"

using namespace helix;
using namespace helix::prefill;

namespace {

// TILES: a grid of XCDs and heads of a group, tiles and rounds, without a division (28
// heads on 4, 8 x 128 9.75 us and 9.5), but it should have more than 8 along x (16
// heads of 64, 8 x 288 11.7 us and 12.0). Else of a round's workgroups and rounds, or
// flat. (All three as values of one argument came out of the compiler with y for z.)
template <int D, bool CAUSAL, bool TILES>
__global__ __launch_bounds__(NT, 2) void attn_prefill_kernel(
    uint16_t* __restrict__ out, const uint16_t* __restrict__ q,
    const uint16_t* __restrict__ k, const uint16_t* __restrict__ v,
    Prefill m, bool flat) {
  extern __shared__ __attribute__((aligned(16))) uint16_t tiles[];
  const int x = blockIdx.x, y = blockIdx.y;
  Place at;
  if constexpr (TILES)
    at = Place{x & 7, x >> 3, y, (int)blockIdx.z};
  else
    at = flat ? place_of(m, x) : place_of(m, x, y);
  queries<D, CAUSAL>(out, q, k, v, m, at, tiles);
}

}  // namespace

void attn_prefill(torch::Tensor out, torch::Tensor q, torch::Tensor k,
                  torch::Tensor v, torch::Tensor cu_seqlens,
                  torch::Tensor cu_seqlens_k, int64_t max_seqlen,
                  double scale, bool causal, int64_t window) {
  const Plan p = plan(out, q, k, v, cu_seqlens, cu_seqlens_k, max_seqlen,
                      scale, window);
  if (p.blocks() == 0) return;
  // a grid has no more than 2^16 along y and z
  const bool flat = p.rounds >= 1 << 16;
  const bool by_tiles = !flat && p.m.spread && p.m.G >= 4 &&
                        p.m.q_tiles < 1 << 16;
  const dim3 grid = by_tiles ? dim3(8 * p.m.G, p.m.q_tiles, p.rounds)
                    : flat   ? dim3(p.blocks())
                             : dim3(p.m.in_round, p.rounds);
  const int D = q.size(2);
  auto stream = at::hip::getCurrentHIPStream();
#define LAUNCH2(DH, C, T)                                                    \
  hipLaunchKernelGGL((attn_prefill_kernel<DH, C, T>), grid, dim3(NT),        \
                     lds_of(DH), stream, (uint16_t*)out.data_ptr(),          \
                     (const uint16_t*)q.data_ptr(),                          \
                     (const uint16_t*)k.data_ptr(),                          \
                     (const uint16_t*)v.data_ptr(), p.m, flat)
#define LAUNCH(DH, C)                                                        \
  if (by_tiles) LAUNCH2(DH, C, true); else LAUNCH2(DH, C, false)
  if (D == 128) {
    if (causal) { LAUNCH(128, true); } else { LAUNCH(128, false); }
  } else {
    if (causal) { LAUNCH(64, true); } else { LAUNCH(64, false); }
  }
#undef LAUNCH2
#undef LAUNCH
}
