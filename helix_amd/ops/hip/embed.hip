// What stands before and behind the blocks of the text encoder and the image
// model (bf16). Each was a chain of torch's gathers, casts, copies and sums, 3 to
// 10 launches that hold almost nothing; here it is one, bound by its start, or for
// large batches of texts by writing them. us of chain -> launch on the GPU:
// text_embed of 60 x 768 23 -> 3.7, of 6044 x 768 46 -> 7, text_pool of 64 texts 14
// -> 3.2; of 8 images image_rows 8.7 -> 2.6, image_tokens 35 -> 6.5, time_embed 17 ->
// 2.3, image_velocity 7.7 -> 2.5. Roundings are those of the chains: what torch
// rounds to bf16 between two steps is rounded here.
#include "common.h"
#include <torch/extension.h>
#include <ATen/hip/HIPContext.h>
#include <c10/core/DeviceGuard.h>

using namespace helix;

namespace {

constexpr int NT = 256;

// Rows of a bf16 table, packed and on 16-byte boundaries.
bool table(const torch::Tensor& t, const torch::Tensor& like, int64_t rows,
           int64_t columns) {
  return t.scalar_type() == torch::kBFloat16 && t.device() == like.device() &&
         t.is_contiguous() && (uintptr_t)t.data_ptr() % 16 == 0 &&
         t.dim() == 2 && t.size(1) == columns &&
         (rows < 0 ? t.size(0) > 0 : t.size(0) == rows);
}
bool numbers(const torch::Tensor& t, torch::ScalarType type,
             const torch::Tensor& like) {
  return t.scalar_type() == type && t.device() == like.device() &&
         t.is_contiguous();
}

__device__ __forceinline__ int clamp_to(int64_t i, int n) {
  return i < 0 ? 0 : i >= n ? n - 1 : (int)i;
}

struct Text {
  const int64_t* ids;          // [T]
  const int* cu;               // [B + 1]
  const uint16_t *word, *pos, *w, *b;
  uint16_t* out;
  int T, B, H, V, P;
  float eps;
};

// Norm of word + position, a wave to a token; NV: vectors of 8 that a lane has. A
// word or place outside its table reads a row that is there and gives no number.
template <int NV>
__global__ __launch_bounds__(NT) void text_embed_kernel(Text m) {
  const int t = blockIdx.x * (NT / WAVE) + threadIdx.x / WAVE;
  if (t >= m.T) return;
  const int lane = threadIdx.x & (WAVE - 1), nvec = m.H / 8;
  int seq = 0;                 // texts that end at or before this token
  for (int i = 0; i < m.B; i += WAVE) {
    const int n = __popcll(__ballot(i + lane < m.B && m.cu[i + lane + 1] <= t));
    seq += n;
    if (n < WAVE) break;
  }
  const int at = t - m.cu[min(seq, m.B - 1)];
  const int64_t id = m.ids[t];
  const bool known = id >= 0 && id < m.V && at >= 0 && at < m.P;
  const uint16_t* word = m.word + (int64_t)clamp_to(id, m.V) * m.H;
  const uint16_t* pos = m.pos + (int64_t)clamp_to(at, m.P) * m.H;
  float v[NV][8], total = known ? 0.f : __builtin_nanf("");
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int c = (i * WAVE + lane) * 8;
    if (i * WAVE + lane < nvec) {
      float p[8];
      load_bf16x8(word + c, v[i]);
      load_bf16x8(pos + c, p);
#pragma unroll
      for (int j = 0; j < 8; ++j)
        v[i][j] = bf16_to_f32(f32_to_bf16(v[i][j] + p[j]));
    } else {
#pragma unroll
      for (int j = 0; j < 8; ++j) v[i][j] = 0.f;
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) total += v[i][j];
  }
  const float mean = wave_reduce_sum(total) / m.H;
  float square = 0.f;
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    if (i * WAVE + lane >= nvec) continue;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      v[i][j] -= mean;
      square += v[i][j] * v[i][j];
    }
  }
  const float inv = rsqrtf(wave_reduce_sum(square) / m.H + m.eps);
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int c = (i * WAVE + lane) * 8;
    if (i * WAVE + lane >= nvec) continue;
    float w[8], b[8];
    load_bf16x8(m.w + c, w);
    load_bf16x8(m.b + c, b);
#pragma unroll
    for (int j = 0; j < 8; ++j) b[j] += v[i][j] * inv * w[j];
    store_bf16x8(m.out + (int64_t)t * m.H + c, b);
  }
}

// A text's first row, divided by its length, a wave each.
__global__ __launch_bounds__(NT) void text_pool_kernel(
    float* __restrict__ out, const uint16_t* __restrict__ x,
    const int* __restrict__ cu, int B, int H) {
  const int s = blockIdx.x * (NT / WAVE) + threadIdx.x / WAVE;
  if (s >= B) return;
  const int lane = threadIdx.x & (WAVE - 1);
  const uint16_t* row = x + (int64_t)cu[s] * H;
  float square = 0.f;
  for (int c = lane * 8; c < H; c += WAVE * 8) {
    float v[8];
    load_bf16x8(row + c, v);
#pragma unroll
    for (int j = 0; j < 8; ++j) square += v[j] * v[j];
  }
  const float root = sqrtf(wave_reduce_sum(square));
  const float length = root < 1e-12f ? 1e-12f : root;     // NaN stays NaN
  for (int c = lane * 8; c < H; c += WAVE * 8) {
    float v[8];
    load_bf16x8(row + c, v);
    f32x4* o = reinterpret_cast<f32x4*>(out + (int64_t)s * H + c);
    o[0] = f32x4{v[0] / length, v[1] / length, v[2] / length, v[3] / length};
    o[1] = f32x4{v[4] / length, v[5] / length, v[6] / length, v[7] / length};
  }
}

// Rows cu[:-1] of x side by side, and their boundaries 0, 1, ..: a workgroup each,
// and one more for the last of those. A text without tokens, or with its first
// outside of x, is no number: the host has not seen the boundaries.
__global__ __launch_bounds__(NT) void text_first_kernel(
    uint16_t* __restrict__ out, int* __restrict__ starts,
    const uint16_t* __restrict__ x, const int* __restrict__ cu, int B, int T,
    int H) {
  const int s = blockIdx.x;
  if (threadIdx.x == 0) starts[s] = s;
  if (s == B) return;
  const int first = cu[s];
  const bool there = first >= 0 && first < T && cu[s + 1] > first;
  const int64_t from = (int64_t)(there ? first : 0) * H, to = (int64_t)s * H;
  for (int c = threadIdx.x * 8; c < H; c += NT * 8) {
    u16x8 v = *reinterpret_cast<const u16x8*>(x + from + c);
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = there ? v[i] : (uint16_t)0x7FC0;
    *reinterpret_cast<u16x8*>(out + to + c) = v;
  }
}

struct Image {
  int B, C, S, p;              // latents [B, C, S, S] in patches of p x p
  int L, text;                 // tokens of an image, of them text
  int K;                       // columns of a patch's row
};

// Element c of patch n of image b in the latents; columns past the patch: -1.
__device__ __forceinline__ int64_t latent_at(const Image& m, int64_t b, int n,
                                             int c) {
  const int g = m.S / m.p, pp = m.p * m.p;
  if (c >= m.C * pp) return -1;
  const int y = n / g * m.p + c % pp / m.p, x = n % g * m.p + c % m.p;
  return ((b * m.C + c / pp) * m.S + y) * m.S + x;
}

// Patches as rows of K columns, zeros behind them.
template <typename T>
__global__ __launch_bounds__(NT) void image_rows_kernel(
    uint16_t* __restrict__ out, const T* __restrict__ lat, Image m,
    int64_t total) {
  const int64_t i = (int64_t)blockIdx.x * NT + threadIdx.x;
  if (i >= total) return;
  const int patches = m.L - m.text;
  const int64_t row = i / m.K;
  const int64_t at = latent_at(m, row / patches, row % patches, i % m.K);
  if constexpr (sizeof(T) == 2) out[i] = at < 0 ? 0 : lat[at];
  else out[i] = at < 0 ? 0 : f32_to_bf16(lat[at]);
}

// Rows of the image tokens back to latents (fp32).
__global__ __launch_bounds__(NT) void image_velocity_kernel(
    float* __restrict__ out, const uint16_t* __restrict__ rows, Image m,
    int64_t total) {
  const int64_t i = (int64_t)blockIdx.x * NT + threadIdx.x;
  if (i >= total) return;
  const int patches = m.L - m.text;
  const int c = i % m.K;
  const int64_t row = i / m.K, b = row / patches;
  const int n = row % patches;
  out[latent_at(m, b, n, c)] =
      bf16_to_f32(rows[(b * m.L + m.text + n) * m.K + c]);
}

struct Tokens {
  const int64_t* ids;          // [B, text]
  const uint16_t *word, *pos, *image;         // [V, H], [L, H], [B patches, H]
  uint16_t *x, *mean;          // [B L, H], [B, H]
  int* cu;                     // [B + 1]
  int B, L, text, H, V;
};

// The text's rows, then the image's, with their places; behind those B more, the
// means of the texts' rows without places; and the images' boundaries.
__global__ __launch_bounds__(NT) void image_tokens_kernel(Tokens m,
                                                          int64_t total) {
  const int64_t i = (int64_t)blockIdx.x * NT + threadIdx.x;
  if (i <= m.B) m.cu[i] = (int)i * m.L;
  if (i >= total) return;
  const int nvec = m.H / 8;
  const int64_t row = i / nvec;
  const int c = (int)(i - row * nvec) * 8;
  const int64_t tokens = (int64_t)m.B * m.L;
  auto word = [&](int64_t b, int l, float* v) {
    load_bf16x8(m.word +
                    (int64_t)clamp_to(m.ids[b * m.text + l], m.V) * m.H + c, v);
  };
  float v[8];
  if (row >= tokens) {
    const int64_t b = row - tokens;
    float sum[8] = {0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll 4
    for (int l = 0; l < m.text; ++l) {
      word(b, l, v);
#pragma unroll
      for (int j = 0; j < 8; ++j) sum[j] += v[j];
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) sum[j] /= m.text;
    float add[8];
    load_bf16x8(m.mean + b * m.H + c, add);
#pragma unroll
    for (int j = 0; j < 8; ++j) add[j] += sum[j];
    store_bf16x8(m.mean + b * m.H + c, add);
    return;
  }
  const int64_t b = row / m.L;
  const int l = (int)(row - b * m.L);
  float p[8];
  if (l < m.text) word(b, l, v);
  else load_bf16x8(m.image + (b * (m.L - m.text) + l - m.text) * m.H + c, v);
  load_bf16x8(m.pos + (int64_t)l * m.H + c, p);
#pragma unroll
  for (int j = 0; j < 8; ++j) v[j] += p[j];
  store_bf16x8(m.x + row * m.H + c, v);
}

// cos and sin of 1000 t 10000^(-i / half), half of the columns each.
__global__ __launch_bounds__(NT) void time_embed_kernel(
    uint16_t* __restrict__ out, const float* __restrict__ t, int B, int half) {
  const int i = blockIdx.x * NT + threadIdx.x;
  if (i >= B * half) return;
  const int b = i / half, c = i % half;
  const float f = expf(-9.210340371976184f * (float)c / (float)half);
  const float a = t[b] * 1000.f * f;
  out[(int64_t)b * 2 * half + c] = f32_to_bf16(cosf(a));
  out[(int64_t)b * 2 * half + half + c] = f32_to_bf16(sinf(a));
}

dim3 blocks(int64_t threads) { return dim3((threads + NT - 1) / NT); }

bool image_of(const torch::Tensor& lat, int64_t patch, int64_t text, int64_t K,
              Image& m) {
  if (!lat.is_cuda() || lat.dim() != 4 || !lat.is_contiguous() ||
      lat.size(2) != lat.size(3) || patch < 1 || lat.size(2) % patch != 0 ||
      lat.numel() == 0 || lat.size(0) > 1 << 16 || lat.size(2) > 1 << 12 ||
      text < 0)
    return false;
  m.B = lat.size(0);
  m.C = lat.size(1);
  m.S = lat.size(2);
  m.p = patch;
  m.text = text;
  m.L = text + (m.S / m.p) * (m.S / m.p);
  m.K = K;
  return (int64_t)m.C * m.p * m.p <= K;
}

}  // namespace

// Below: false (or nothing), and nothing done, for other forms of operands than
// the kernels read.

// out[T, H] = layer norm of word[ids] + pos[place within the text].
bool text_embed(torch::Tensor out, torch::Tensor ids, torch::Tensor cu,
                torch::Tensor word, torch::Tensor pos, torch::Tensor w,
                torch::Tensor b, double eps) {
  Text m{};
  if (!out.is_cuda() || out.dim() != 2) return false;
  m.T = out.size(0);
  m.H = out.size(1);
  if (!table(out, out, m.T, m.H) || !table(word, out, -1, m.H) ||
      !table(pos, out, -1, m.H) || m.H % 8 != 0 || m.H > 4096 ||
      !numbers(ids, torch::kInt64, out) || ids.dim() != 1 ||
      ids.numel() != m.T || !numbers(cu, torch::kInt32, out) ||
      cu.dim() != 1 || cu.numel() < 2 || word.size(0) > INT32_MAX ||
      pos.size(0) > INT32_MAX)
    return false;
  for (const auto& t : {w, b})
    if (!numbers(t, torch::kBFloat16, out) || t.dim() != 1 ||
        t.numel() != m.H || (uintptr_t)t.data_ptr() % 16 != 0)
      return false;
  if (m.T == 0) return true;
  m.ids = ids.data_ptr<int64_t>();
  m.cu = cu.data_ptr<int>();
  m.word = (const uint16_t*)word.data_ptr();
  m.pos = (const uint16_t*)pos.data_ptr();
  m.w = (const uint16_t*)w.data_ptr();
  m.b = (const uint16_t*)b.data_ptr();
  m.out = (uint16_t*)out.data_ptr();
  m.B = cu.numel() - 1;
  m.V = word.size(0);
  m.P = pos.size(0);
  m.eps = (float)eps;
  const c10::DeviceGuard on(out.device());
  const dim3 grid(cdiv(m.T, NT / WAVE));
  auto stream = at::hip::getCurrentHIPStream();
#define HELIX_TE(NV)                                                         \
  hipLaunchKernelGGL(text_embed_kernel<NV>, grid, dim3(NT), 0, stream, m)
  if (m.H <= 512) HELIX_TE(1);
  else if (m.H <= 1024) HELIX_TE(2);
  else if (m.H <= 2048) HELIX_TE(4);
  else HELIX_TE(8);
#undef HELIX_TE
  return true;
}

// out[B, H] (fp32): rows cu[:-1] of x, each divided by its length.
bool text_pool(torch::Tensor out, torch::Tensor x, torch::Tensor cu) {
  if (!x.is_cuda() || x.dim() != 2 || !table(x, x, x.size(0), x.size(1)) ||
      x.size(1) % 8 != 0 || !numbers(cu, torch::kInt32, x) || cu.dim() != 1 ||
      cu.numel() < 2 || !numbers(out, torch::kFloat32, x) || out.dim() != 2 ||
      out.size(0) != cu.numel() - 1 || out.size(1) != x.size(1))
    return false;
  const c10::DeviceGuard on(x.device());
  const int B = out.size(0);
  hipLaunchKernelGGL(text_pool_kernel, dim3(cdiv(B, NT / WAVE)), dim3(NT), 0,
                     at::hip::getCurrentHIPStream(), out.data_ptr<float>(),
                     (const uint16_t*)x.data_ptr(), cu.data_ptr<int>(), B,
                     (int)x.size(1));
  return true;
}

// out[B, H], starts[B + 1]: rows cu[:-1] of x and the boundaries of texts of a token
// each. A text without tokens is NaN; x and out are packed rows on 16-byte boundaries.
void text_first(torch::Tensor out, torch::Tensor starts, torch::Tensor x,
                torch::Tensor cu) {
  const int64_t B = cu.numel() - 1;
  TORCH_CHECK(x.is_cuda() && x.dim() == 2 &&
              table(x, x, x.size(0), x.size(1)) && x.size(1) % 8 == 0 &&
              x.size(0) >= 1 && x.size(0) <= INT32_MAX &&
              numbers(cu, torch::kInt32, x) && cu.dim() == 1 && B >= 1 &&
              table(out, x, B, x.size(1)) &&
              numbers(starts, torch::kInt32, x) && starts.numel() == B + 1,
              "rows of texts");
  hipLaunchKernelGGL(text_first_kernel, dim3(B + 1), dim3(NT), 0,
                     at::hip::getCurrentHIPStream(), (uint16_t*)out.data_ptr(),
                     starts.data_ptr<int>(), (const uint16_t*)x.data_ptr(),
                     cu.data_ptr<int>(), (int)B, (int)x.size(0),
                     (int)x.size(1));
}

// out[B patches, K]: patches of the latents (bf16 or fp32) as rows.
bool image_rows(torch::Tensor out, torch::Tensor lat, int64_t patch) {
  Image m{};
  if (out.dim() != 2 || !image_of(lat, patch, 0, out.size(1), m) ||
      !numbers(out, torch::kBFloat16, lat) ||
      out.size(0) != (int64_t)m.B * m.L)
    return false;
  const c10::DeviceGuard on(lat.device());
  auto stream = at::hip::getCurrentHIPStream();
  uint16_t* o = (uint16_t*)out.data_ptr();
  const int64_t n = out.numel();
  if (lat.scalar_type() == torch::kBFloat16)
    hipLaunchKernelGGL(image_rows_kernel<uint16_t>, blocks(n), dim3(NT), 0,
                       stream, o, (const uint16_t*)lat.data_ptr(), m, n);
  else if (lat.scalar_type() == torch::kFloat32)
    hipLaunchKernelGGL(image_rows_kernel<float>, blocks(n), dim3(NT), 0, stream,
                       o, lat.data_ptr<float>(), m, n);
  else
    return false;
  return true;
}

// out[B, C, S, S] (fp32) of the image tokens' rows [B L, C patch patch].
bool image_velocity(torch::Tensor out, torch::Tensor rows, int64_t patch,
                    int64_t text) {
  Image m{};
  if (rows.dim() != 2 || !image_of(out, patch, text, rows.size(1), m) ||
      out.scalar_type() != torch::kFloat32 ||
      !numbers(rows, torch::kBFloat16, out) || m.K != m.C * m.p * m.p ||
      rows.size(0) != (int64_t)m.B * m.L)
    return false;
  const c10::DeviceGuard on(out.device());
  const int64_t n = out.numel();
  hipLaunchKernelGGL(image_velocity_kernel, blocks(n), dim3(NT), 0,
                     at::hip::getCurrentHIPStream(), out.data_ptr<float>(),
                     (const uint16_t*)rows.data_ptr(), m, n);
  return true;
}

// x[B L, H] = word[ids] and then image, each with pos; cond[B, H] += mean of
// word[ids]; cu[B + 1] = 0, L, ..
bool image_tokens(torch::Tensor x, torch::Tensor cond, torch::Tensor cu,
                  torch::Tensor ids, torch::Tensor word, torch::Tensor pos,
                  torch::Tensor image) {
  Tokens m{};
  if (!x.is_cuda() || x.dim() != 2 || ids.dim() != 2) return false;
  m.B = ids.size(0);
  m.text = ids.size(1);
  m.L = pos.size(0);
  m.H = x.size(1);
  if (m.B < 1 || m.text < 1 || m.L <= m.text || m.H % 8 != 0 ||
      !table(x, x, (int64_t)m.B * m.L, m.H) || !table(cond, x, m.B, m.H) ||
      !table(word, x, -1, m.H) || !table(pos, x, m.L, m.H) ||
      !table(image, x, (int64_t)m.B * (m.L - m.text), m.H) ||
      !numbers(ids, torch::kInt64, x) || !numbers(cu, torch::kInt32, x) ||
      cu.numel() != m.B + 1 || word.size(0) > INT32_MAX ||
      (int64_t)m.B * m.L > INT32_MAX)
    return false;
  m.ids = ids.data_ptr<int64_t>();
  m.word = (const uint16_t*)word.data_ptr();
  m.pos = (const uint16_t*)pos.data_ptr();
  m.image = (const uint16_t*)image.data_ptr();
  m.x = (uint16_t*)x.data_ptr();
  m.mean = (uint16_t*)cond.data_ptr();
  m.cu = cu.data_ptr<int>();
  m.V = word.size(0);
  const c10::DeviceGuard on(x.device());
  const int64_t total = (int64_t)m.B * (m.L + 1) * (m.H / 8);
  hipLaunchKernelGGL(image_tokens_kernel, blocks(std::max<int64_t>(total, m.B + 1)),
                     dim3(NT), 0, at::hip::getCurrentHIPStream(), m, total);
  return true;
}

// out[B, 2 half]: the sinusoidal embedding of t[B] (fp32).
bool time_embed(torch::Tensor out, torch::Tensor t) {
  if (!t.is_cuda() || t.dim() != 1 || !numbers(t, torch::kFloat32, t) ||
      !numbers(out, torch::kBFloat16, t) || out.dim() != 2 ||
      out.size(0) != t.size(0) || out.size(1) % 2 != 0 || out.size(1) < 2 ||
      out.numel() == 0 || out.numel() > INT32_MAX)
    return false;
  const int half = out.size(1) / 2;
  const c10::DeviceGuard on(t.device());
  hipLaunchKernelGGL(time_embed_kernel, blocks(t.size(0) * half), dim3(NT), 0,
                     at::hip::getCurrentHIPStream(), (uint16_t*)out.data_ptr(),
                     t.data_ptr<float>(), (int)t.size(0), half);
  return true;
}
