// Prompt attention, see attn_prefill.h.
#include "attn_prefill.h"

using namespace helix;
using namespace helix::prefill;

namespace {

template <int D, bool CAUSAL>
__global__ __launch_bounds__(NT, 2) void attn_prefill_kernel(
    uint16_t* __restrict__ out, const uint16_t* __restrict__ q,
    const uint16_t* __restrict__ k, const uint16_t* __restrict__ v,
    Prefill m, bool flat) {
  extern __shared__ __attribute__((aligned(16))) uint16_t tiles[];
  const Place at = flat ? place_of(m, blockIdx.x)
                        : Place{(int)blockIdx.x & 7, (int)blockIdx.x >> 3,
                                (int)blockIdx.y, (int)blockIdx.z};
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
  // a grid has no more along y and z
  const bool flat = p.grid.y >= 1 << 16 || p.grid.z >= 1 << 16;
  const dim3 grid = flat ? dim3(p.blocks()) : p.grid;
  const int D = q.size(2);
  auto stream = at::hip::getCurrentHIPStream();
#define LAUNCH(DH, C)                                                        \
  hipLaunchKernelGGL((attn_prefill_kernel<DH, C>), grid, dim3(NT),           \
                     lds_of(DH), stream, (uint16_t*)out.data_ptr(),      \
                     (const uint16_t*)q.data_ptr(),                          \
                     (const uint16_t*)k.data_ptr(),                          \
                     (const uint16_t*)v.data_ptr(), p.m, flat)
  if (causal) {
    if (D == 128) LAUNCH(128, true); else LAUNCH(64, true);
  } else {
    if (D == 128) LAUNCH(128, false); else LAUNCH(64, false);
  }
#undef LAUNCH
}
