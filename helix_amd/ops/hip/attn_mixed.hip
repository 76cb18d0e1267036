// Attention of a mixed step in one launch: prompt portions (attn_prefill.h), which
// are bound by instruction issue, and replies (paged_rows.h), which are bound by the
// memory. The portions' workgroups come first; the replies' fill the places that
// these leave (a CU has two) and come after them. us one behind the other and at
// once, 32 heads on 8 of 128: 40 replies of 100..3000 and 1500 tokens behind 5001
// with a window of 4096 186 and 157, and 600 new ones 72 and 59; 64 of 300..4000 and
// 200 behind 5000 205 and 143, and 200 120 and 110; 10 of them and 2000 80 and 66; 2
// of 300 and 17 14.5 and 10.0. Not for many short replies beside short portions (see
// `joins`). Results are the same bits.
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
    prefill::queries<D, true>(out, qp, k, v, pm,
                              prefill::place_of(pm, blockIdx.x), lds);
  } else {
    const int per = dm.heads_first ? dm.Hkv : pieces;
    const int high = at / per, low = at - high * per;
    paged::rows<D, G, F8, true>(qd, kc, vc, dm, dm.heads_first ? high : low,
                                dm.heads_first ? low : high,
                                *reinterpret_cast<paged::Shared<D, G>*>(lds));
  }
}

// Whether one launch takes no longer than two. It hides the portions' chain of key
// tiles, some 4 us and 1.2 a tile, behind the replies. But these have two workgroups
// on a CU here and, in groups of four heads, three alone, which many short ones need
// to hide their latency: 3 ns a workgroup with e4m3 up to 1024 tokens (1536 where
// rows are cut), 2 with bf16 up to 384. With eight heads alone it is two as well. us
// of two launches and of one, 32 heads on 8, up to 300 tokens unless said:
//   e4m3  512 replies and 17 tokens 46.5 and 55.7, 300 51.5 and 57.5, 600 58.1 and
//         60.0, 17 behind 700 58.6 and 56.6, 64 behind 1000 65.4 and 57.8; 384 and 300
//         43.9 and 45.5, 600 51.0 and 48.9; 256 and 17 30.4 and 31.5, 300 35.7 and
//         33.6; 128 of 1500 (cut) and 17 60.8 and 63.0, 300 66.0 and 64.5; 300 of 1500
//         (whole) and 17 99.1 and 95.2; 512 of 640 and 17 110 and 115, 300 118.5 and
//         117.3; 1024 and 600 100 and 113
//   bf16  512 and 17 77.2 and 79.4, 300 82.6 and 81.4, of 500 and 17 132.6 and 126.5;
//         384 and 17 63.2 and 62.6; 1024 and 300 150.6 and 154.5, 600 158.2 and 157.6
//   64 heads on 8, 512 and 17: e4m3 85.8 and 81.0, bf16 105.4 and 95.8
// Lengths on the device are not known: the bound stands for them, and the mean of
// portions for each.
bool joins(const paged::Plan& d, int64_t bound, int64_t keys) {
  if (d.G != 4) return true;
  const int64_t replies = (int64_t)d.pieces * d.m.Hkv;
  const int64_t tiles = (keys + prefill::KT - 1) / prefill::KT;
  if (d.f8)
    return bound > (d.m.split ? 1536 : 1024) || replies <= 1600 + 250 * tiles;
  return bound > 384 || replies <= 3000 + 600 * tiles;
}

}  // namespace

// Both, as attn_prefill (causal) and paged_attn_decode do them. False, and nothing
// done, for other heads, groups and pages, and where two launches are faster.
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
  const int portions = p.blocks();
  if (portions == 0 || d.m.B == 0) return false;
  const auto seen = [&](int64_t n, int64_t more) {
    return window > 0 ? std::min(n, window + more) : n;
  };
  if (!joins(d, seen(max_len, 0), seen(k.size(0) / p.m.seqs, max_seqlen)))
    return false;
  auto stream = at::hip::getCurrentHIPStream();
#define HELIX_AM(G, F8)                                                      \
  hipLaunchKernelGGL((attn_mixed_kernel<G, F8>),                             \
                     dim3(portions + d.pieces * d.m.Hkv), dim3(prefill::NT), \
                     prefill::lds_of(D), stream, (uint16_t*)out_p.data_ptr(),\
                     (const uint16_t*)q_p.data_ptr(),                        \
                     (const uint16_t*)k.data_ptr(),                          \
                     (const uint16_t*)v.data_ptr(), p.m, portions,           \
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
