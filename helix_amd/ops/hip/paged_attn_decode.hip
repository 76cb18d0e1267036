// Decode attention, see paged_rows.h.
#include "paged_rows.h"

using namespace helix;
using namespace helix::paged;

namespace {

template <int D, int G, bool F8, bool PAGE8>
__global__ __launch_bounds__(NT, waves_per_simd(D, G)) void paged_rows_kernel(
    const uint16_t* __restrict__ q, const void* __restrict__ kc,
    const void* __restrict__ vc, Rows m) {
  __shared__ Shared<D, G> lds;
  // by the grid's two dimensions; dividing one number takes longer (32 heads on 8, 1
  // row of 1500 10.8 us for 10.5, e4m3 10.2 for 10.0, 32 of 1025..1044 33.0 for 30.1)
  rows<D, G, F8, PAGE8>(q, kc, vc, m, m.heads_first ? blockIdx.y : blockIdx.x,
                        m.heads_first ? blockIdx.x : blockIdx.y, lds);
}

template <int D, int G>
void launch(const uint16_t* q, const void* kc, const void* vc, const Rows& m,
            bool f8, dim3 grid, hipStream_t stream) {
#define HELIX_PD(F8, P8)                                                     \
  hipLaunchKernelGGL((paged_rows_kernel<D, G, F8, P8>), grid, dim3(NT), 0,   \
                     stream, q, kc, vc, m)
  if (m.shift >= 3) {
    if (f8) HELIX_PD(true, true);
    else HELIX_PD(false, true);
  } else {
    if (f8) HELIX_PD(true, false);
    else HELIX_PD(false, false);
  }
#undef HELIX_PD
}

}  // namespace

void paged_attn_decode(torch::Tensor out, torch::Tensor q,
                       torch::Tensor k_cache, torch::Tensor v_cache,
                       torch::Tensor block_tables, torch::Tensor seq_lens,
                       double scale, torch::Tensor tmp_out,
                       torch::Tensor tmp_ml, int64_t max_len_hint,
                       int64_t window) {
  const Plan p = plan(out, q, k_cache, v_cache, block_tables, seq_lens, scale,
                      tmp_out, tmp_ml, max_len_hint, window);
  if (p.m.B == 0) return;
  const dim3 grid = p.m.heads_first ? dim3(p.m.Hkv, p.pieces)
                                    : dim3(p.pieces, p.m.Hkv);
  auto stream = at::hip::getCurrentHIPStream();
#define DISPATCH(DH, GG)                                                     \
  launch<DH, GG>((const uint16_t*)q.data_ptr(), k_cache.data_ptr(),          \
                 v_cache.data_ptr(), p.m, p.f8, grid, stream)
  if (p.D == 128) {
    if (p.G == 1) DISPATCH(128, 1);
    else if (p.G == 2) DISPATCH(128, 2);
    else if (p.G == 4) DISPATCH(128, 4);
    else DISPATCH(128, 8);
  } else {
    if (p.G == 1) DISPATCH(64, 1);
    else if (p.G == 2) DISPATCH(64, 2);
    else if (p.G == 4) DISPATCH(64, 4);
    else DISPATCH(64, 8);
  }
#undef DISPATCH
  merge(p, stream);
}
