// A block of the text encoder and one of the image model as one call from Python:
// the launches of their steps, in order, with nothing else between them.
//
// A small batch is bound by the host: views, allocations and the arguments of seven
// calls a block. us of the host, step by step -> by one call: one image through 12
// blocks 890 -> 563, eight 848 -> 561; a text of 60 tokens through 12 blocks, which
// the GPU now takes as long for, 748 -> 526. The kernels are those of the steps, but
// that sums behind deep products take these in stretches (gemm_bf16_summand).
#include "common.h"
#include <torch/extension.h>
#include <c10/core/DeviceGuard.h>

using OptT = c10::optional<torch::Tensor>;
using Tensors = std::vector<torch::Tensor>;
using OptTs = std::vector<OptT>;

// of gemm_bf16.hip, gemm_rows.hip, attn_prefill.hip, embed.hip and encoder.hip
void text_first(torch::Tensor out, torch::Tensor starts, torch::Tensor x,
                torch::Tensor cu);
void gemm_bf16(torch::Tensor out, torch::Tensor x, torch::Tensor w, OptT bias,
               int64_t act, int64_t tile);
void gemm_rows(torch::Tensor out, torch::Tensor x, torch::Tensor w, OptT bias,
               OptT x_scale, OptT w_scale, bool gelu);
void attn_prefill(torch::Tensor out, torch::Tensor q, torch::Tensor k,
                  torch::Tensor v, torch::Tensor cu_seqlens,
                  torch::Tensor cu_seqlens_k, int64_t max_seqlen, double scale,
                  bool causal, int64_t window);
bool add_norm(OptT sum, torch::Tensor out, torch::Tensor x, OptT y, OptT gate,
              torch::Tensor a, torch::Tensor b, int64_t L, double eps,
              OptT y_bias);
torch::Tensor gemm_bf16_summand(torch::Tensor x, torch::Tensor w,
                                torch::Tensor bias);

namespace {

// Packed bf16 of that size on 16-byte boundaries, beside x.
bool packed(const torch::Tensor& t, const torch::Tensor& x,
            at::IntArrayRef sizes) {
  return t.scalar_type() == torch::kBFloat16 && t.device() == x.device() &&
         t.sizes() == sizes && t.is_contiguous() &&
         (uintptr_t)t.data_ptr() % 16 == 0;
}
// The first n of p: none where one of them is missing (a bias that is None).
Tensors present(const OptTs& p, size_t n) {
  if (p.size() < n) return {};
  Tensors all;
  for (size_t i = 0; i < n; ++i) {
    if (!p[i].has_value()) return {};
    all.push_back(*p[i]);
  }
  return all;
}
bool layer(const Tensors& p, size_t i, const torch::Tensor& x, int64_t out,
           int64_t in) {
  return packed(p[i], x, {out, in}) && packed(p[i + 1], x, {out});
}

// What ops.gemm_bf16 does with packed rows.
torch::Tensor product(const torch::Tensor& x, const torch::Tensor& w,
                      const torch::Tensor& b, int act) {
  const int64_t M = x.size(0), K = x.size(1), N = w.size(0);
  torch::Tensor out = at::empty({M, N}, x.options());
  if (M <= 64 && K >= 2 * N && N * K <= 8 << 20 && N % 8 == 0 && K % 256 == 0)
    gemm_rows(out, x, w, b, {}, {}, act == 1);
  else
    gemm_bf16(out, x, w, b, act, 0);
  return out;
}

// The same for a norm that adds it to something: rows, or stretches of them that
// the norm adds up (add_norm's y_bias).
struct Summand {
  torch::Tensor y;
  OptT bias;                   // still to be added
};
Summand summand(const torch::Tensor& x, const torch::Tensor& w,
                const torch::Tensor& b) {
  Summand s;
  s.y = x.size(0) <= 64 ? product(x, w, b, 0) : gemm_bf16_summand(x, w, b);
  if (s.y.dim() == 3) s.bias = b;
  return s;
}

torch::Tensor attend(const torch::Tensor& x, const torch::Tensor& w,
                     const torch::Tensor& b, const torch::Tensor& cu,
                     int64_t max_len, int64_t heads, double scale) {
  const int64_t T = x.size(0), H = x.size(1), D = H / heads;
  const torch::Tensor qkv = product(x, w, b, 0);
  const int64_t at = qkv.storage_offset();
  auto part = [&](int64_t i) {
    return qkv.as_strided({T, heads, D}, {3 * H, D, 1}, at + i * H);
  };
  torch::Tensor o = at::empty({T, heads, D}, x.options());
  attn_prefill(o, part(0), part(1), part(2), cu, cu, max_len, scale, false, 0);
  return o.view({T, H});
}

bool rows_of(const torch::Tensor& x, const torch::Tensor& cu, int64_t heads) {
  if (!x.is_cuda() || x.dim() != 2) return false;
  const int64_t T = x.size(0), H = x.size(1);
  return T > 0 && H > 0 && H % 64 == 0 && H <= 4096 && heads > 0 &&
         (H == heads * 64 || H == heads * 128) && packed(x, x, {T, H}) &&
         cu.scalar_type() == torch::kInt32 && cu.device() == x.device() &&
         cu.dim() == 1 && cu.numel() >= 2 && cu.is_contiguous();
}


// p: weight and bias of q k v, attention's end, its norm, the way up, the way down,
// the last norm. first: only the first row of each text, which has one, and the
// boundaries of texts of a row each. Keys and values are of all rows then, and the
// rest is of as many rows as there are texts: 16000 tokens of 64 texts, 768 columns,
// 273 us -> 90.
Tensors through_text(torch::Tensor x, const torch::Tensor& cu, int64_t max_len,
                     int64_t heads, double scale, double eps,
                     const OptTs& params, bool first) {
  const Tensors p = present(params, 12);
  if (p.empty() || params.size() != 12 || !rows_of(x, cu, heads) ||
      p[6].dim() != 2)
    return {};
  const int64_t H = x.size(1), I = p[6].size(0);
  if (I < 1 || I % 64 != 0 || !layer(p, 0, x, 3 * H, H) ||
      !layer(p, 2, x, H, H) || !layer(p, 6, x, I, H) || !layer(p, 8, x, H, I))
    return {};
  for (int i : {4, 5, 10, 11})
    if (!packed(p[i], x, {H})) return {};
  const c10::DeviceGuard on(x.device());
  auto norm = [&](const torch::Tensor& a, const Summand& b, int i) {
    torch::Tensor out = at::empty_like(a);
    TORCH_CHECK(add_norm({}, out, a, b.y, {}, p[i], p[i + 1], 0, eps, b.bias),
                "a norm of other operands");
    return out;
  };
  torch::Tensor o, starts;
  if (first) {
    const int64_t T = x.size(0), B = cu.numel() - 1, D = H / heads;
    const torch::Tensor rows = at::empty({B, H}, x.options());
    starts = at::empty({B + 1}, cu.options());
    text_first(rows, starts, x, cu);
    const torch::Tensor kv = product(x, p[0].narrow(0, H, 2 * H),
                                     p[1].narrow(0, H, 2 * H), 0);
    const torch::Tensor q = product(rows, p[0].narrow(0, 0, H),
                                    p[1].narrow(0, 0, H), 0);
    auto part = [&](int64_t i) {
      return kv.as_strided({T, heads, D}, {2 * H, D, 1},
                           kv.storage_offset() + i * H);
    };
    o = at::empty({B, heads, D}, x.options());
    attn_prefill(o, q.view({B, heads, D}), part(0), part(1), starts, cu, 1,
                 scale, false, 0);
    o = o.view({B, H});
    x = rows;
  } else {
    o = attend(x, p[0], p[1], cu, max_len, heads, scale);
  }
  x = norm(x, summand(o, p[2], p[3]), 4);
  const torch::Tensor up = product(x, p[6], p[7], 1);
  x = norm(x, summand(up, p[8], p[9]), 10);
  if (first) return {x, starts};
  return {x};
}

}  // namespace

// All: nothing, and nothing done, for other forms of operands than all of the
// steps' kernels read.

OptT text_block(torch::Tensor x, torch::Tensor cu, int64_t max_len,
                int64_t heads, double scale, double eps, OptTs params) {
  const Tensors out = through_text(x, cu, max_len, heads, scale, eps, params,
                                   false);
  return out.empty() ? OptT{} : out[0];
}

// Its result for the first row of each text, which has one, and the boundaries of
// texts of a row each.
Tensors text_block_first(torch::Tensor x, torch::Tensor cu, int64_t max_len,
                         int64_t heads, double scale, double eps,
                         OptTs params) {
  return through_text(x, cu, max_len, heads, scale, eps, params, true);
}

// x (+ gate y) through a block: the result as x, y and gate of a sum that is still
// to be taken, and where y is in stretches the bias that is still to be added to
// it. mod: shift, scale and gate of either half, a row for every L of x. p: weight
// and bias of q k v, attention's end, the way up, the way down. stretches: whether y
// may be in such.
Tensors image_block(torch::Tensor x, OptT y, OptT gate, OptT y_bias,
                    torch::Tensor mod, torch::Tensor cu, int64_t L,
                    int64_t heads, double scale, double eps, OptTs params,
                    bool stretches) {
  const Tensors p = present(params, 8);
  if (p.empty() || !rows_of(x, cu, heads) || p[4].dim() != 2) return {};
  const int64_t T = x.size(0), H = x.size(1), I = p[4].size(0);
  if (I < 1 || I % 64 != 0 || L < 1 || T % L != 0 ||
      !packed(mod, x, {T / L, 6 * H}) || !layer(p, 0, x, 3 * H, H) ||
      !layer(p, 2, x, H, H) || !layer(p, 4, x, I, H) ||
      !layer(p, 6, x, H, I) || y.has_value() != gate.has_value() ||
      (y_bias.has_value() && !y.has_value()))
    return {};
  if (y.has_value()) {
    const bool rows = !y_bias.has_value();
    if (rows ? !packed(*y, x, x.sizes())
             : !packed(*y_bias, x, {H}) || y->dim() != 3 || y->size(0) < 1 ||
                   y->size(1) != T || y->size(2) != H ||
                   y->scalar_type() != torch::kFloat32 ||
                   y->device() != x.device() || !y->is_contiguous() ||
                   (uintptr_t)y->data_ptr() % 16 != 0)
      return {};
    if (gate->dim() != 2 || gate->device() != x.device() ||
        gate->scalar_type() != torch::kBFloat16 || gate->size(0) != T / L ||
        gate->size(1) != H || gate->stride(1) != 1 ||
        gate->stride(0) % 8 != 0 || (uintptr_t)gate->data_ptr() % 16 != 0)
      return {};
  }
  const c10::DeviceGuard on(x.device());
  auto of = [&](int64_t i) {
    return mod.as_strided({T / L, H}, {6 * H, 1}, mod.storage_offset() + i * H);
  };
  auto norm = [&](const OptT& b, const OptT& bias, const OptT& g, int shift) {
    torch::Tensor out = at::empty_like(x);
    OptT sum;
    if (b.has_value()) sum = at::empty_like(x);
    TORCH_CHECK(add_norm(sum, out, x, b, g, of(shift + 1), of(shift), L, eps,
                         bias),
                "a norm of other operands");
    if (sum.has_value()) x = *sum;
    return out;
  };
  const torch::Tensor o =
      attend(norm(y, y_bias, gate, 0), p[0], p[1], cu, L, heads, scale);
  const Summand a = summand(o, p[2], p[3]);
  const torch::Tensor up = product(norm(a.y, a.bias, of(2), 3), p[4], p[5], 1);
  if (!stretches) return {x, product(up, p[6], p[7], 0), of(5)};
  const Summand m = summand(up, p[6], p[7]);
  if (!m.bias.has_value()) return {x, m.y, of(5)};
  return {x, m.y, of(5), *m.bias};
}
