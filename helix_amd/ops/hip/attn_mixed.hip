// Attention of a mixed step in one launch: prompt portions (attn_prefill.h), which
// are bound by instruction issue, and replies (paged_rows.h), which are bound by the
// memory. The portions' workgroups come first; the replies' fill the places that
// these leave (a CU has two) and come after them. Never slower than one behind the
// other, so all sizes go here; us, 32 heads on 8 of 128: 40 replies of 100..3000 and
// 1500 tokens behind 5001 with a window of 4096 186 -> 157, and 600 new ones 72 ->
// 59; 64 of 300..4000 and 200 behind 5000 205 -> 143, and 200 120 -> 110; 10 of them
// and 2000 80 -> 66; 2 of 300 and 17 14.5 -> 10.0. Results are the same bits.
#include "attn_prefill.h"
#include "paged_rows.h"

using namespace helix;

namespace {

constexpr int D = 128;

template <int G, bool F8>
__global__ __launch_bounds__(prefill::NT, 2) void attn_mixed_kernel(
    uint16_t* __restrict__ out, const uint16_t* __restrict__ qp,
    const uint16_t* __restrict__ k, const uint16_t* __restrict__ v,
    prefill::Prefill pm, int portions, const uint16_t* __restrict__ qd,
    const void* __restrict__ kc, const void* __restrict__ vc, paged::Rows dm,
    int pieces) {
  static_assert(prefill::NT == paged::NT && sizeof(paged::Shared<D, G>) <=
                    prefill::lds_of(D), "one shape of workgroup");
  extern __shared__ __attribute__((aligned(16))) uint16_t lds[];
  const int at = (int)blockIdx.x - portions;
  if (at < 0) {
    prefill::queries<D, true>(out, qp, k, v, pm, blockIdx.x, lds);
  } else {
    paged::rows<D, G, F8, true>(qd, kc, vc, dm, at, pieces,
                                *reinterpret_cast<paged::Shared<D, G>*>(lds));
  }
}

}  // namespace

// Both, as attn_prefill (causal) and paged_attn_decode do them. False, and nothing
// done, for other heads, groups and pages.
bool attn_mixed(torch::Tensor out_p, torch::Tensor q_p, torch::Tensor k,
                torch::Tensor v, torch::Tensor cu_seqlens,
                torch::Tensor cu_seqlens_k, int64_t max_seqlen,
                torch::Tensor out_d, torch::Tensor q_d, torch::Tensor k_cache,
                torch::Tensor v_cache, torch::Tensor block_tables,
                torch::Tensor seq_lens, torch::Tensor tmp_out,
                torch::Tensor tmp_ml, int64_t max_len, double scale,
                int64_t window) {
  if (q_p.dim() != 3 || q_d.dim() != 3 || k_cache.dim() != 4 ||
      q_p.size(2) != D || q_d.size(2) != D || q_p.device() != q_d.device() ||
      k_cache.size(1) < 1)
    return false;
  const int64_t G = q_d.size(1) / k_cache.size(1), bs = k_cache.size(2);
  if ((G != 4 && G != 8) || bs < 8 || (bs & (bs - 1)) != 0) return false;
  const prefill::Plan p = prefill::plan(out_p, q_p, k, v, cu_seqlens,
                                        cu_seqlens_k, max_seqlen, scale, window);
  const paged::Plan d = paged::plan(out_d, q_d, k_cache, v_cache, block_tables,
                                    seq_lens, scale, tmp_out, tmp_ml, max_len,
                                    window);
  if (p.grid == 0 || d.m.B == 0) return false;
  auto stream = at::hip::getCurrentHIPStream();
#define HELIX_AM(G, F8)                                                      \
  hipLaunchKernelGGL((attn_mixed_kernel<G, F8>),                             \
                     dim3(p.grid + d.pieces * d.m.Hkv), dim3(prefill::NT),   \
                     prefill::lds_of(D), stream, (uint16_t*)out_p.data_ptr(),\
                     (const uint16_t*)q_p.data_ptr(),                        \
                     (const uint16_t*)k.data_ptr(),                          \
                     (const uint16_t*)v.data_ptr(), p.m, p.grid,             \
                     (const uint16_t*)q_d.data_ptr(), k_cache.data_ptr(),    \
                     v_cache.data_ptr(), d.m, d.pieces)
  if (G == 4) {
    if (d.f8) HELIX_AM(4, true); else HELIX_AM(4, false);
  } else {
    if (d.f8) HELIX_AM(8, true); else HELIX_AM(8, false);
  }
#undef HELIX_AM
  paged::merge(d, stream);
  return true;
}
