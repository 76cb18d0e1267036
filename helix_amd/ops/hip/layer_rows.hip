// Projections of a few rows of a language model's layer, bf16 with fp32 sums, up to 16,
// with what comes before and behind them: x[M,K] @ w[N,K]^T and
//   JOIN  the residual is added, and rows leave times the next norm's weight, with
//         sums of squares beside them; whoever multiplies them divides by their
//         root, which is one factor a row and can wait for the sums;
//   QKV   heads are turned and written to the cache (rope_qkv.hip);
//   GLU   silu(gate) * other factor.
// A layer of a few rows is bound by reading its weights and by its launches: each
// takes 3 us more than its bytes. Norm and rotation as launches of their own took
// 4.4 us each, three of nine launches of a layer.
//
// A workgroup has all of the inner dimension, so that it sees whole sums: its four
// waves have a quarter each, for the same columns, and pass their sums through LDS.
// Columns are 16 (JOIN, QKV of up to 4 rows) or 32 (QKV of more; GLU, of either
// factor). Waves begin at the start of their quarter: with groups of columns beginning
// at different chunks, chunks dealt to the waves one by one, or eight waves, 1 row of
// 4096 x 4096 took 7.6 to 11.5 us instead of 7.5. GLU's groups do begin apart (`turn`).
// Weights go straight to MFMA operands, a chunk of the inner dimension ahead, which is
// 512 bytes, and 256 of GLU and of more than 16 rows (see `run`). Rows of x come by
// whole lines and become operands through a wave's own LDS: by loads in operand order,
// which take half lines, 16 rows of it took 11.0 us instead of 9.5, 8 rows of 4096 x
// 14336 27.5 instead of 25.2.
//
// us of a product and the launch before or behind it (gemm_rows.hip with norm.hip
// or rope_qkv.hip), and of all here, weights from memory:
//         6144 x 4096    4096 x 4096    4096 x 14336   2 x 14336 x 4096
//         (QKV)          (JOIN)         (JOIN)         (GLU, alone)
//   M  1  15.0  13.6     13.4  10.0     27.7  23.5     43.1  43.5
//   M  4  15.1  13.4     13.6   9.7     27.9  23.9     43.3  43.3
//   M  8  15.6  13.4     13.8   9.7     28.3  25.0     43.5  44.7
//   M 16  15.9  14.9     14.2  10.6     29.2  28.5     44.7  45.8
// GLU gains nothing by itself: it is here to take rows whose division is still to come,
// which is what spares JOIN a norm behind it.
// QKV goes on to 32 rows, without squares, and takes e4m3 (scaled 16x16x128 with
// unity scales; those of rows meet the sums): 32 rows of 6144 x 4096 16.4 us apart
// and 15.6, e4m3 13.4 and 10.3. The other forms would not gain there: 24 rows of
// 4096 x 14336 29 and 31, the gated product of e4m3 26 and 29.
#include "hybrid/tile.h"
#include <torch/extension.h>
#include <ATen/hip/HIPContext.h>
#include <c10/core/DeviceGuard.h>
#include <type_traits>

using namespace helix;

namespace {

constexpr int NW = 4, NT = NW * WAVE;
constexpr int MOST_ROWS = 16, MOST_PARTS = 512;
constexpr int MOST_ROWS_QKV = 32;
constexpr int UNITY = 0x7F7F7F7F;             // e8m0 2^0 in all four bytes

enum Form { JOIN, QKV, GLU };

struct LayerRows {
  const char *x, *w;           // [M, K]; [N, K], GLU [2 N, K]
  const float* squares;        // [M, parts] of x's rows, or null
  const float *xs, *ws;        // e4m3: scales of rows of x and of w
  uint16_t* out;               // JOIN and GLU [M, N]
  int M, N, K, parts;
  float eps;
  // JOIN
  uint16_t* residual;          // [M, N]
  const uint16_t* norm;        // [N]
  float* squares_out;          // [M, N / 16]
  // QKV
  const uint16_t* bias;        // [N] or null
  const int64_t *positions, *slots;           // slots may be null
  uint16_t *q, *k, *v;         // compact; k and v may be null
  void *kc, *vc;               // pages, with slots
  const float* cs;             // [positions, D]
  int Hq, Hkv, D, bs, shift;   // bs is 1 << shift, or shift -1
};

template <bool F8>
__device__ __forceinline__ void write_cache4(void* c, int64_t at,
                                             const float* v) {
  if constexpr (F8) {
    uint32_t p = 0;
    p = __builtin_amdgcn_cvt_pk_fp8_f32(v[0], v[1], p, false);
    p = __builtin_amdgcn_cvt_pk_fp8_f32(v[2], v[3], p, true);
    *reinterpret_cast<uint32_t*>((uint8_t*)c + at) = p;
  } else {
    st_bf16x4((uint16_t*)c + at, v);
  }
}

typedef int v8i __attribute__((ext_vector_type(8)));
__device__ __forceinline__ v8i both(u32x4 a, u32x4 b) {
  return v8i{(int)a[0], (int)a[1], (int)a[2], (int)a[3],
             (int)b[0], (int)b[1], (int)b[2], (int)b[3]};
}

// MR: rows that there is room for, at least M; more than 16 only without squares.
// NI: tiles of 16 rows of w of a workgroup, which go to half as many columns of GLU.
// CHUNK: bytes of the inner dimension. F8: e4m3 pages (QKV). F8X: x and w are e4m3.
template <int MR, int NI, int CHUNK, Form FORM, bool F8, bool F8X>
__global__ __launch_bounds__(NT) void layer_rows_kernel(LayerRows m) {
  constexpr int U = CHUNK / 64, PIECES = CHUNK / 16, XL = MR * PIECES / WAVE;
  constexpr int MI = MR > 16 ? MR / 16 : 1;   // tiles of 16 rows of x
  constexpr bool SQUARES = FORM != JOIN && MI == 1 && !F8X;
  constexpr int PART = MOST_PARTS / (4 * WAVE);
  __shared__ f32x4 red[NW][MI * NI][WAVE];
  __shared__ u32x4 xs[NW][MR * PIECES];
  __shared__ float inv[MOST_ROWS];
  const int tid = threadIdx.x, lane = tid & (WAVE - 1);
  const int wid = __builtin_amdgcn_readfirstlane(tid / WAVE);
  const int lo = lane & 15, hi = lane >> 4;
  const int tile = blockIdx.x, half = m.D / 2;
  // of the tile of x that this wave ends
  const int r_end = (MI > 1 ? wid * 16 : 0) + lo, row = min(r_end, m.M - 1);
  // QKV: a workgroup has pairs that are turned together, x and then y
  constexpr int PAIRS = 8 * NI;
  const int per = FORM == QKV ? half / PAIRS : 1;
  const int head = tile / per, d0 = tile % per * PAIRS;
  // row of w
  auto row_of = [&](int j) {
    if constexpr (FORM == JOIN) return tile * 16 + lo;
    if constexpr (FORM == GLU)
      return (j & 1) * m.N + (tile * (NI / 2) + j / 2) * 16 + lo;
    const int i = j * 16 + lo;
    return head * m.D + d0 + (i < PAIRS ? i : half + i - PAIRS);
  };

  // Loads come back in order, so what else is read goes before the weights.
  f32x4 part[SQUARES ? MR / NW : 1][PART];
  if (SQUARES && m.squares != nullptr) {
#pragma unroll
    for (int r = 0; r < MR / NW; ++r)
      if (r * NW + wid < m.M)
#pragma unroll
        for (int i = 0; i < PART; ++i) {
          const int at = (i * WAVE + lane) * 4;
          part[r][i] = at < m.parts ? *reinterpret_cast<const f32x4*>(
                                          m.squares + (r * NW + wid) * m.parts +
                                          at)
                                    : f32x4{0, 0, 0, 0};
        }
  }
  u16x4 added = {0, 0, 0, 0}, factor = {0, 0, 0, 0};
  int64_t position = 0, slot = -1;
  if constexpr (FORM == JOIN) {
    const int c = tile * 16 + hi * 4;
    added = *reinterpret_cast<const u16x4*>(m.residual + row * m.N + c);
    factor = *reinterpret_cast<const u16x4*>(m.norm + c);
  } else if constexpr (FORM == QKV) {
    position = m.positions[row];
    if (m.slots != nullptr) slot = m.slots[row];
  }

  // A lane's 16 bytes u of a chunk's row: bf16 has four lane groups to 64 bytes,
  // e4m3 two pieces side by side to 128.
  auto piece = [&](int u) {
    return F8X ? (u >> 1) * 8 + hi * 2 + (u & 1) : u * 4 + hi;
  };
  const int64_t bytes = (int64_t)m.K * (F8X ? 1 : 2);
  const char* wp[NI];
#pragma unroll
  for (int j = 0; j < NI; ++j)
    wp[j] = m.w + row_of(j) * bytes;
  // 16-byte piece p of row r lies at p ^ r % 16: operands leave LDS without bank
  // conflicts
  const char* xp[XL];
#pragma unroll
  for (int i = 0; i < XL; ++i) {
    const int e = i * WAVE + lane, r = e / PIECES;
    xp[i] = m.x + min(r, m.M - 1) * bytes + (e % PIECES ^ (r & 15)) * 16;
  }
  const int chunks = (int)(bytes / CHUNK), share = cdiv(chunks, NW);
  const int start = min(chunks, wid * share), end = min(chunks, start + share);
  const int turn = FORM == GLU && end > start ? tile % (end - start) : 0;
  u32x4 wr[2][U][NI], xr[2][XL];
  auto load = [&](int c, auto buf) {
    constexpr int b = decltype(buf)::value;
    if constexpr (FORM == GLU)
      c = c + turn < end ? c + turn : c + turn - end + start;
#pragma unroll
    for (int i = 0; i < XL; ++i)
      xr[b][i] = *reinterpret_cast<const u32x4*>(xp[i] + c * CHUNK);
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int j = 0; j < NI; ++j)
        wr[b][u][j] = *reinterpret_cast<const u32x4*>(wp[j] + c * CHUNK +
                                                      piece(u) * 16);
    __builtin_amdgcn_sched_barrier(0);
  };
  floatx4 acc[MI][NI];
#pragma unroll
  for (int t = 0; t < MI; ++t)
#pragma unroll
    for (int j = 0; j < NI; ++j) acc[t][j] = floatx4{0, 0, 0, 0};
  u32x4* const mine = xs[wid];
  auto multiply = [&](auto buf) {
    constexpr int b = decltype(buf)::value;
#pragma unroll
    for (int i = 0; i < XL; ++i) mine[i * WAVE + lane] = xr[b][i];
#pragma unroll
    for (int t = 0; t < MI; ++t) {
      // columns past the last row repeat others, and nobody looks at them
      const int r = MI > 1 ? t * 16 + lo : lo & (MR - 1);
      u32x4 xf[U];
#pragma unroll
      for (int u = 0; u < U; ++u)
        xf[u] = mine[r * PIECES + (piece(u) ^ (r & 15))];
#pragma unroll
      for (int u = 0; u < U; u += F8X ? 2 : 1)
#pragma unroll
        for (int j = 0; j < NI; ++j) {
          if constexpr (F8X)
            acc[t][j] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(
                both(wr[b][u][j], wr[b][u + 1][j]), both(xf[u], xf[u + 1]),
                acc[t][j], 0, 0, 0, UNITY, 0, UNITY);
          else
            acc[t][j] = mfma16(__builtin_bit_cast(u16x8, wr[b][u][j]),
                               __builtin_bit_cast(u16x8, xf[u]), acc[t][j]);
        }
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  constexpr std::integral_constant<int, 0> A;
  constexpr std::integral_constant<int, 1> B;
  int c = start;
  if (c < end) load(c, A);
  float cosine[4], sine[4];
  if constexpr (FORM == QKV) {
    const float* cs = m.cs + position * m.D + d0 + (NI == 1 ? hi & 1 : hi) * 4;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      cosine[q] = cs[q];
      sine[q] = cs[half + q];
    }
  }
  if (SQUARES && m.squares != nullptr) {
#pragma unroll
    for (int r = 0; r < MR / NW; ++r)
      if (r * NW + wid < m.M) {
        float s = 0.f;
#pragma unroll
        for (int i = 0; i < PART; ++i)
          s += part[r][i][0] + part[r][i][1] + part[r][i][2] + part[r][i][3];
        s = wave_reduce_sum(s);
        if (lane == 0) inv[r * NW + wid] = rsqrtf(s / m.K + m.eps);
      }
  }
  __builtin_amdgcn_sched_barrier(0);
  if (c < end) {
    for (; c + 2 < end; c += 2) {
      load(c + 1, B);
      multiply(A);
      load(c + 2, A);
      multiply(B);
    }
    if (c + 1 < end) {
      load(c + 1, B);
      multiply(A);
      multiply(B);
    } else {
      multiply(A);
    }
  }
#pragma unroll
  for (int t = 0; t < MI; ++t)
#pragma unroll
    for (int j = 0; j < NI; ++j)
      red[wid][t * NI + j][lane] = __builtin_bit_cast(f32x4, acc[t][j]);
  __syncthreads();
  if (wid >= MI) return;
  // lane: columns 4 hi + i of row lo of a tile
  f32x4 s[NI];
#pragma unroll
  for (int j = 0; j < NI; ++j) {
    s[j] = red[0][wid * NI + j][lane];
#pragma unroll
    for (int w = 1; w < NW; ++w) s[j] += red[w][wid * NI + j][lane];
  }
  const bool there = r_end < m.M;
  float v[4];
  if constexpr (FORM == JOIN) {
    const int64_t at = (int64_t)row * m.N + tile * 16 + hi * 4;
    float ss = 0.f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      v[i] = s[0][i] + bf16_to_f32(added[i]);
      ss += v[i] * v[i];
      added[i] = f32_to_bf16(v[i]);
      v[i] *= bf16_to_f32(factor[i]);
    }
    ss += __shfl_xor(ss, 16, WAVE);
    ss += __shfl_xor(ss, 32, WAVE);
    if (!there) return;
    *reinterpret_cast<u16x4*>(m.residual + at) = added;
    st_bf16x4(m.out + at, v);
    if (hi == 0) m.squares_out[row * gridDim.x + tile] = ss;
    return;
  }
  const float f = F8X ? m.xs[row]
                  : SQUARES && m.squares != nullptr ? inv[row] : 1.f;
  if constexpr (FORM == GLU) {
    if (!there) return;
#pragma unroll
    for (int j = 0; j < NI; j += 2) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float g = s[j][i] * f;
        v[i] = g / (1.f + __expf(-g)) * (s[j + 1][i] * f);
      }
      st_bf16x4(m.out + (int64_t)row * m.N + tile * 8 * NI + j * 8 + hi * 4, v);
    }
  } else if constexpr (FORM == QKV) {
    // lane: four pairs; of those of one tile, x or y
    const bool second = NI == 1 && hi >= 2, value = head >= m.Hq + m.Hkv;
    const int d = d0 + (NI == 1 ? hi & 1 : hi) * 4;
    float o[NI][4];
#pragma unroll
    for (int j = 0; j < NI; ++j)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int n = head * m.D + (second || j == 1 ? half : 0) + d + i;
        o[j][i] = s[j][i] * f;
        if constexpr (F8X) o[j][i] *= m.ws[n];
        if (m.bias != nullptr) o[j][i] += bf16_to_f32(m.bias[n]);
      }
    if (!value) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float a = o[0][i];
        const float b = NI == 1 ? __shfl_xor(a, 32, WAVE) : o[NI - 1][i];
        o[0][i] = second ? a * cosine[i] + b * sine[i]
                         : a * cosine[i] - b * sine[i];
        if constexpr (NI == 2) o[1][i] = b * cosine[i] + a * sine[i];
      }
    }
    if (!there) return;
    const int g = head - m.Hq - (value ? m.Hkv : 0);
    uint16_t* to = head < m.Hq
                       ? m.q + ((int64_t)row * m.Hq + head) * m.D
                       : value ? m.v : m.k;
    if (head >= m.Hq && to != nullptr) to += ((int64_t)row * m.Hkv + g) * m.D;
    const int64_t page = m.shift >= 0 ? slot >> m.shift : slot / m.bs;
    const int64_t place =
        ((page * m.Hkv + g) * m.bs + (slot - page * m.bs)) * m.D;
#pragma unroll
    for (int j = 0; j < NI; ++j) {
      const int at = (second || j == 1 ? half : 0) + d;
      if (to != nullptr) st_bf16x4(to + at, o[j]);
      if (head >= m.Hq && slot >= 0)
        write_cache4<F8>(value ? m.vc : m.kc, place + at, o[j]);
    }
  }
}

using OptT = c10::optional<torch::Tensor>;

// Everything goes by raw addresses: packed, of one GPU and on these boundaries.
void check(const torch::Tensor& t, const torch::Tensor& x,
           torch::ScalarType type, int to) {
  TORCH_CHECK(t.is_cuda() && t.device() == x.device() && t.is_contiguous() &&
              t.scalar_type() == type && (uintptr_t)t.data_ptr() % to == 0,
              "packed operands on one GPU");
}

LayerRows rows_of(const torch::Tensor& x, const torch::Tensor& w,
                  const OptT& squares, double eps,
                  torch::ScalarType type = torch::kBFloat16,
                  int most = MOST_ROWS) {
  check(x, x, type, 16);
  check(w, x, type, 16);
  TORCH_CHECK(x.dim() == 2 && w.dim() == 2 && x.size(1) == w.size(1));
  LayerRows m{};
  m.x = (const char*)x.data_ptr();
  m.w = (const char*)w.data_ptr();
  m.M = x.size(0);
  m.N = w.size(0);
  m.K = x.size(1);
  m.eps = (float)eps;
  TORCH_CHECK(m.M >= 1 && x.size(0) <= most && m.K > 0 &&
              x.size(1) * x.element_size() % 512 == 0 &&
              x.size(1) <= 1 << 24 && m.N > 0 && w.size(0) <= 1 << 24,
              "a few rows of whole chunks");
  if (squares.has_value()) {
    check(*squares, x, torch::kFloat32, 16);
    TORCH_CHECK(squares->dim() == 2 && squares->size(0) == m.M &&
                squares->size(1) % 4 == 0 && squares->size(1) <= MOST_PARTS);
    m.squares = squares->data_ptr<float>();
    m.parts = squares->size(1);
  }
  return m;
}

// Tiles of 32 rows of w read x half as often, which is worth as much from 5 rows
// on; few columns would leave CUs idle by them (us of 1, 8 and 16 rows by 16 and
// by 32: 6144 x 4096 11.8 and 12.1, 13.5 and 12.2, 15.7 and 13.2; 4096 x 14336 23
// and 37). Of the gated product a wave has 32 columns of either factor, in chunks of
// 256 bytes that begin apart: 41.2, 42.8 and 45.7 us of 2 x 14336 x 4096, with 16 in
// chunks of 512 41.3, 43.8 and 46.4.
template <Form FORM, bool F8 = false, bool F8X = false>
void run(const LayerRows& m) {
#define HELIX_LR(MR, NI, CHUNK)                                              \
  hipLaunchKernelGGL((layer_rows_kernel<MR, NI, CHUNK, FORM, F8, F8X>),      \
                     dim3(m.N / (FORM == GLU ? 8 * NI : 16 * NI)), dim3(NT), \
                     0, at::hip::getCurrentHIPStream(), m)
  constexpr int NI = FORM == GLU ? 4 : 1, MORE = FORM == QKV ? 2 : NI;
  constexpr int CHUNK = FORM == GLU ? 256 : 512;
  if (m.M <= 4) HELIX_LR(4, NI, CHUNK);
  else if (m.M <= 8) HELIX_LR(8, MORE, CHUNK);
  else if (m.M <= 16) HELIX_LR(16, MORE, CHUNK);
  else if constexpr (FORM == QKV) HELIX_LR(32, 2, 256);
#undef HELIX_LR
}

}  // namespace

// residual += x w^T; rows leave times norm, with their sums of squares
// [M, N / 16], which are of the sums before they were rounded.
std::vector<torch::Tensor> layer_rows_join(torch::Tensor x, torch::Tensor w,
                                           torch::Tensor residual,
                                           torch::Tensor norm) {
  const c10::DeviceGuard on(x.device());
  LayerRows m = rows_of(x, w, c10::nullopt, 0);
  check(residual, x, torch::kBFloat16, 8);
  check(norm, x, torch::kBFloat16, 8);
  TORCH_CHECK(m.N % 64 == 0 && m.N / 16 <= MOST_PARTS &&
              residual.dim() == 2 && residual.size(0) == m.M &&
              residual.size(1) == m.N && norm.numel() == m.N);
  torch::Tensor out = torch::empty_like(residual);
  torch::Tensor squares = torch::empty({m.M, m.N / 16},
                                       x.options().dtype(torch::kFloat32));
  m.residual = (uint16_t*)residual.data_ptr();
  m.norm = (const uint16_t*)norm.data_ptr();
  m.out = (uint16_t*)out.data_ptr();
  m.squares_out = squares.data_ptr<float>();
  run<JOIN>(m);
  return {out, squares};
}

// silu(x w[:N]^T f) * (x w[N:]^T f), f one over the root of a row's mean square
torch::Tensor layer_rows_glu(torch::Tensor x, torch::Tensor w, OptT squares,
                             double eps) {
  const c10::DeviceGuard on(x.device());
  LayerRows m = rows_of(x, w, squares, eps);
  TORCH_CHECK(m.N % 64 == 0);
  m.N /= 2;
  torch::Tensor out = torch::empty({m.M, m.N}, x.options());
  m.out = (uint16_t*)out.data_ptr();
  run<GLU>(m);
  return out;
}

// Heads of x w^T f + bias, turned, to q (and k, v) and the pages of slots. x and w
// are bf16, or e4m3 with scales of their rows; squares of up to 16 rows of bf16.
void layer_rows_qkv(torch::Tensor x, torch::Tensor w, OptT bias, OptT squares,
                    double eps, torch::Tensor positions, torch::Tensor cos_sin,
                    torch::Tensor q, OptT k, OptT v, OptT k_cache,
                    OptT v_cache, OptT slots, int64_t num_q, int64_t num_kv,
                    int64_t head_dim, OptT x_scale, OptT w_scale) {
  const c10::DeviceGuard on(x.device());
  const bool f8x = x_scale.has_value();
  LayerRows m = rows_of(x, w, squares, eps,
                        f8x ? torch::kUInt8 : torch::kBFloat16, MOST_ROWS_QKV);
  TORCH_CHECK(w_scale.has_value() == f8x &&
              (m.squares == nullptr || (!f8x && m.M <= MOST_ROWS)));
  if (f8x) {
    check(*x_scale, x, torch::kFloat32, 4);
    check(*w_scale, x, torch::kFloat32, 4);
    TORCH_CHECK(x_scale->numel() == m.M && w_scale->numel() == m.N);
    m.xs = x_scale->data_ptr<float>();
    m.ws = w_scale->data_ptr<float>();
  }
  TORCH_CHECK(num_q > 0 && num_kv > 0 && head_dim > 0 && head_dim % 32 == 0 &&
              (num_q + 2 * num_kv) * head_dim == m.N);
  m.Hq = num_q;
  m.Hkv = num_kv;
  m.D = head_dim;
  if (bias.has_value()) {
    check(*bias, x, torch::kBFloat16, 2);
    TORCH_CHECK(bias->numel() == m.N);
    m.bias = (const uint16_t*)bias->data_ptr();
  }
  check(positions, x, torch::kInt64, 8);
  check(cos_sin, x, torch::kFloat32, 4);
  TORCH_CHECK(positions.numel() == m.M && cos_sin.dim() == 2 &&
              cos_sin.size(1) == m.D);
  m.positions = positions.data_ptr<int64_t>();
  m.cs = cos_sin.data_ptr<float>();
  check(q, x, torch::kBFloat16, 8);
  TORCH_CHECK(q.numel() == m.M * num_q * head_dim);
  m.q = (uint16_t*)q.data_ptr();
  TORCH_CHECK(k.has_value() == v.has_value());
  if (k.has_value()) {
    for (const auto& t : {*k, *v}) {
      check(t, x, torch::kBFloat16, 8);
      TORCH_CHECK(t.numel() == m.M * num_kv * head_dim);
    }
    m.k = (uint16_t*)k->data_ptr();
    m.v = (uint16_t*)v->data_ptr();
  }
  m.bs = 1;
  bool f8 = false;
  TORCH_CHECK(k_cache.has_value() == v_cache.has_value());
  if (k_cache.has_value()) {
    f8 = k_cache->scalar_type() == torch::kUInt8;
    for (const auto& t : {*k_cache, *v_cache}) {
      check(t, x, f8 ? torch::kUInt8 : torch::kBFloat16, 8);
      TORCH_CHECK(t.dim() == 4 && t.sizes() == k_cache->sizes() &&
                  t.size(1) == num_kv && t.size(3) == head_dim);
    }
    TORCH_CHECK(slots.has_value());
    check(*slots, x, torch::kInt64, 8);
    TORCH_CHECK(slots->numel() == m.M);
    m.bs = k_cache->size(2);
    m.kc = k_cache->data_ptr();
    m.vc = v_cache->data_ptr();
    m.slots = slots->data_ptr<int64_t>();
  }
  m.shift = (m.bs & (m.bs - 1)) == 0 ? __builtin_ctz(m.bs) : -1;
  if (f8x) {
    if (f8) run<QKV, true, true>(m);
    else run<QKV, false, true>(m);
  } else if (f8) {
    run<QKV, true>(m);
  } else {
    run<QKV>(m);
  }
}
