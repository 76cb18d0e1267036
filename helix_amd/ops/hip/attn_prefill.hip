// Flash-attention prefill (varlen, causal/bidirectional, GQA) for CDNA4.
//
// Replaces the prefill attention the reference delegates to vLLM. Bound by
// instruction issue: of a wave's 2500 cycles per tile the matrix cores have
// 1020 and the vector ALU 1250 (half of it exponentials), and counters show
// that the two hardly overlap, neither within a wave (the next scores computed
// beside the exponentials changed nothing) nor between the two waves of a SIMD
// (nor did their priorities).
//
//  - A workgroup has 128 queries of one head, each of its 4 waves 32 of them.
//    Scores are computed transposed (key x query): a lane has one query, its
//    statistics cost two lane swaps, and 8 neighbouring keys of its weights
//    are an operand of the value product as they lie.
//  - Tiles of 64 keys and values go straight to LDS, the next one while the
//    last is worked on, with one barrier a tile. Rows lie as in memory; their
//    16-byte pieces are stored crosswise, so that keys leave LDS as operands
//    and values through the transposing load without bank conflicts.
//  - All tiles of a (sequence, head) run on one XCD, the latest, which see
//    the most keys, first.
//
// The kernel before had 64 queries, stored values transposed element by
// element and passed weights through LDS. 32 heads on 8 of 128, us before ->
// now (TFLOP/s now): 1 x 8192 2551 -> 645 (850), 8 x 2048 1918 -> 413 (665),
// 31 of 400..620 440 -> 188 (384), 1500 behind 5001 with a window of 4096
// 466 -> 173 (582). 12 heads of 64, 64 texts of 20..500: 178 -> 68. Workgroups
// of 64 queries (2 waves) take 1.1 to 1.8 times as long from 100 queries on,
// and no less time below. The distance from 64 bits is what it was.
//
// MFMA fragment layouts (gfx950, f32_16x16x32_bf16), hi = lane / 16,
// lo = lane % 16: A[lo][8 hi + i], B[8 hi + i][lo], D[4 hi + r][lo].
#include "hybrid/tile.h"
#include <torch/extension.h>
#include <ATen/hip/HIPContext.h>

using namespace helix;

namespace {

constexpr int NT = 256, NW = NT / WAVE;
constexpr int QT = NW * 32;                   // queries of a workgroup
constexpr int KT = 64;                        // keys of a tile
constexpr float LOG2E = 1.4426950408889634f;
constexpr float NEG = -1e30f;
// instruction classes of the scheduling hints
constexpr int MFMA = 0x008, DS_READ = 0x100;

struct Prefill {
  const int* cu_q;             // [B + 1] query rows
  const int* cu_k;             // [B + 1] key rows (>= query rows)
  int64_t q_stride, k_stride, v_stride;       // of a row, in elements
  int Hq, G, q_tiles, seqs, window;
  bool flip;                   // negative scale: of negated queries
  float mul;                   // |scale| * log2(e)
};

__device__ __forceinline__ float max_over_groups(float v) {
  const unsigned u = __float_as_uint(v);
  const auto a = __builtin_amdgcn_permlane32_swap(u, u, false, false);
  const float x = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
  const unsigned w = __float_as_uint(x);
  const auto b = __builtin_amdgcn_permlane16_swap(w, w, false, false);
  return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}

// Four rows of one column from LDS: the 16 lanes of a quarter wave name 4
// rows x 16 columns, 4 columns each (lane j: row j / 4, columns 4 (j % 4)..),
// and get a column each.
__device__ __forceinline__ u16x4 ld_tr4(const uint16_t* p) {
  typedef __attribute__((ext_vector_type(4))) int16_t i16x4;
  return __builtin_bit_cast(u16x4, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
      (__attribute__((address_space(3))) i16x4*)p));
}

// Piece p of row r lies at p ^ cross(r): the 16 rows 8 a + 4 s + b (a, b < 4)
// of a score operand, and the 16 of a value operand, meet every bank equally.
template <int D>
__device__ __forceinline__ int cross(int r) {
  return D == 128 ? (r & 3) | (r >> 1 & 12) : (r >> 1 & 1) | (r >> 2 & 6);
}

template <int D, bool CAUSAL>
__global__ __launch_bounds__(NT, 2) void attn_prefill_kernel(
    uint16_t* __restrict__ out, const uint16_t* __restrict__ q,
    const uint16_t* __restrict__ k, const uint16_t* __restrict__ v,
    Prefill m) {
  constexpr int NK = D / 32, NV = D / 16, PR = D / 8;
  constexpr int LOADS = KT * PR / NT;
  __shared__ __attribute__((aligned(16))) uint16_t kl[2][KT * D];
  __shared__ __attribute__((aligned(16))) uint16_t vl[2][KT * D];
  const int xcd = blockIdx.x & 7, at = blockIdx.x >> 3;
  const int total = m.seqs * m.Hq, chunk = cdiv(total, 8);
  const int sh = xcd * chunk + at / m.q_tiles;
  if (at / m.q_tiles >= chunk || sh >= total) return;
  const int b = sh / m.Hq, h = sh % m.Hq, g = h / m.G;
  const int q0 = (m.q_tiles - 1 - at % m.q_tiles) * QT;
  const int row0 = m.cu_q[b], qlen = m.cu_q[b + 1] - row0;
  if (q0 >= qlen) return;
  const int key0 = m.cu_k[b], klen = m.cu_k[b + 1] - key0;
  const int ctx = klen - qlen;                // cached tokens before

  const int tid = threadIdx.x, wid = tid / WAVE, lane = tid & (WAVE - 1);
  const int lo = lane & 15, hi = lane >> 4;
  u16x8 qf[2][NK];
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const int qi = min(q0 + wid * 32 + u * 16 + lo, qlen - 1);
    const uint16_t* qr = q + (row0 + qi) * m.q_stride + h * D + hi * 8;
#pragma unroll
    for (int c = 0; c < NK; ++c) {
      qf[u][c] = ld_u16x8(qr + c * 32);
      if (m.flip) qf[u][c] ^= (uint16_t)0x8000;
    }
  }

  const uint16_t* kb = k + key0 * m.k_stride + g * D;
  const uint16_t* vb = v + key0 * m.v_stride + g * D;
  // This lane's pieces of a tile: where they lie is the same in every tile but
  // a partial one, whose rows past the end repeat the last and are masked.
  int ko[LOADS], vo[LOADS];
  auto places = [&](int rows, int64_t stride, int* o) {
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
      const int e = (i * NW + wid) * WAVE + lane, r = e / PR;
      o[i] = (min(r, rows - 1) * (int)stride + (e % PR ^ cross<D>(r)) * 8) * 2;
    }
  };
  auto fetch = [&](const uint16_t* base, int64_t stride, int* o, int t,
                   uint16_t* lds) {
    if (t + KT > klen) places(klen - t, stride, o);
    const char* from = (const char*)(base + t * stride);
#pragma unroll
    for (int i = 0; i < LOADS; ++i)
      __builtin_amdgcn_global_load_lds(
          (const __attribute__((address_space(1))) uint32_t*)(from + o[i]),
          (__attribute__((address_space(3))) uint32_t*)(
              lds + (i * NW + wid) * WAVE * 8),
          16, 0, 0);
  };
  places(KT, m.k_stride, ko);
  places(KT, m.v_stride, vo);
  // where this lane reads, within 16 rows of keys and 4 of values
  int ka[NK], va[NV];
  const int kr = (lo >> 2) * 8 + (lo & 3), vr = hi * 8 + (lo >> 2);
#pragma unroll
  for (int c = 0; c < NK; ++c)
    ka[c] = kr * D + ((c * 4 + hi) ^ cross<D>(kr)) * 8;
#pragma unroll
  for (int d = 0; d < NV; ++d)
    va[d] = vr * D + ((d * 2 + (lo >> 1 & 1)) ^ cross<D>(vr)) * 8 +
            (lo & 1) * 4;

  floatx4 acc[NV][2];
  float m_run[2] = {NEG, NEG}, l[2] = {0.f, 0.f};
#pragma unroll
  for (int d = 0; d < NV; ++d) acc[d][0] = acc[d][1] = floatx4{0, 0, 0, 0};
  const int last = CAUSAL ? min(klen, ctx + q0 + QT) : klen;
  const int qa = ctx + q0 + wid * 32, qz = qa + 31;       // of this wave
  const bool windowed = CAUSAL && m.window > 0;
  int t = windowed ? max(0, ctx + q0 - m.window + 1) / KT * KT : 0;

  // scores of 64 keys: [32 keys][half][query tile]
  auto product = [&](const uint16_t* keys, floatx4 (*s)[2][2]) {
#pragma unroll
    for (int w = 0; w < 2; ++w)
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        s[w][j][0] = s[w][j][1] = floatx4{0, 0, 0, 0};
#pragma unroll
        for (int c = 0; c < NK; ++c) {
          const u16x8 a = ld_u16x8(keys + (w * 32 + j * 4) * D + ka[c]);
          s[w][j][0] = mfma16(a, qf[0][c], s[w][j][0]);
          s[w][j][1] = mfma16(a, qf[1][c], s[w][j][1]);
        }
      }
  };
  if (t < last) {
    fetch(kb, m.k_stride, ko, t, kl[0]);
    fetch(vb, m.v_stride, vo, t, vl[0]);
  }
  for (int buf = 0; t < last; t += KT, buf ^= 1) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (t + KT < last) {
      fetch(kb, m.k_stride, ko, t + KT, kl[buf ^ 1]);
      fetch(vb, m.v_stride, vo, t + KT, vl[buf ^ 1]);
    }
    if (CAUSAL && t > qz) continue;
    floatx4 s[2][2][2];
    product(kl[buf], s);
    // operands leave LDS a group ahead of their products
    __builtin_amdgcn_sched_group_barrier(DS_READ, 2 * NK, 0);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      __builtin_amdgcn_sched_group_barrier(MFMA, 2 * NK, 0);
      __builtin_amdgcn_sched_group_barrier(DS_READ, NK, 0);
    }
    __builtin_amdgcn_sched_group_barrier(MFMA, 4 * NK, 0);

    const bool edge = (CAUSAL && t + KT - 1 > qa) || t + KT > klen ||
                      (windowed && t <= qz - m.window);
    if (edge) {
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const int qi = qa + u * 16 + lo;
        const int low = windowed ? qi - m.window : -1;
        const int top = CAUSAL ? min(qi, klen - 1) : klen - 1;
#pragma unroll
        for (int w = 0; w < 2; ++w)
#pragma unroll
          for (int i = 0; i < 8; ++i) {
            const int key = t + w * 32 + hi * 8 + i;
            if (key > top || key <= low) s[w][i >> 2][u][i & 3] = NEG;
          }
      }
    }
    float mx[2], base[2];
    bool stay = true;
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      mx[u] = m_run[u];
#pragma unroll
      for (int w = 0; w < 2; ++w)
#pragma unroll
        for (int i = 0; i < 8; ++i)
          mx[u] = fmaxf(mx[u], s[w][i >> 2][u][i & 3]);
      mx[u] = max_over_groups(mx[u]);
      stay = stay && mx[u] == m_run[u];
    }
    if (!__all(stay)) {
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const float corr = __builtin_amdgcn_exp2f((m_run[u] - mx[u]) * m.mul);
        l[u] *= corr;
        m_run[u] = mx[u];
#pragma unroll
        for (int d = 0; d < NV; ++d)
#pragma unroll
          for (int i = 0; i < 4; ++i) acc[d][u][i] *= corr;
      }
    }
    // a query that has seen no key yet keeps weights of exactly zero
#pragma unroll
    for (int u = 0; u < 2; ++u)
      base[u] = m_run[u] <= NEG ? 0.f : m_run[u] * m.mul;
    u16x8 pf[2][2];
    auto weights = [&]() {
#pragma unroll
      for (int w = 0; w < 2; ++w)
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          float p[8];
#pragma unroll
          for (int i = 0; i < 8; ++i) {
            p[i] = __builtin_amdgcn_exp2f(
                fmaf(s[w][i >> 2][u][i & 3], m.mul, -base[u]));
            l[u] += p[i];
          }
          pf[w][u] = pack8(p);
        }
    };
    weights();
#pragma unroll
    for (int w = 0; w < 2; ++w)
#pragma unroll
      for (int d = 0; d < NV; ++d) {
        const uint16_t* at = vl[buf] + w * 32 * D + va[d];
        const u16x4 x = ld_tr4(at), y = ld_tr4(at + 4 * D);
        const u16x8 a = {x[0], x[1], x[2], x[3], y[0], y[1], y[2], y[3]};
        acc[d][0] = mfma16(a, pf[w][0], acc[d][0]);
        acc[d][1] = mfma16(a, pf[w][1], acc[d][1]);
      }
    __builtin_amdgcn_sched_group_barrier(DS_READ, 8, 0);
#pragma unroll
    for (int i = 0; i < 2 * NV - 4; ++i) {
      __builtin_amdgcn_sched_group_barrier(MFMA, 2, 0);
      __builtin_amdgcn_sched_group_barrier(DS_READ, 2, 0);
    }
    __builtin_amdgcn_sched_group_barrier(MFMA, 8, 0);
  }

#pragma unroll
  for (int u = 0; u < 2; ++u) {
    l[u] += __shfl_xor(l[u], 16, WAVE);
    l[u] += __shfl_xor(l[u], 32, WAVE);
    const float f = 1.f / fmaxf(l[u], 1e-20f);
    const int qi = q0 + wid * 32 + u * 16 + lo;
    if (qi >= qlen) continue;
    uint16_t* dst = out + ((int64_t)(row0 + qi) * m.Hq + h) * D + hi * 4;
#pragma unroll
    for (int d = 0; d < NV; ++d) {
      const float x[4] = {acc[d][u][0] * f, acc[d][u][1] * f,
                          acc[d][u][2] * f, acc[d][u][3] * f};
      st_bf16x4(dst + d * 16, x);
    }
  }
}

// Rows of [T, H, D] with their heads side by side, 16-byte aligned, anywhere;
// other layouts are copied. Places within a tile are 32-bit byte offsets.
torch::Tensor rows(const torch::Tensor& t) {
  const bool fits = t.stride(2) == 1 && t.stride(1) == t.size(2) &&
                    t.stride(0) % 8 == 0 && t.stride(0) > 0 &&
                    t.stride(0) < (1 << 23);
  const torch::Tensor r = fits ? t : t.contiguous();
  return (uintptr_t)r.data_ptr() % 16 == 0 ? r : r.clone();
}

}  // namespace

void attn_prefill(torch::Tensor out, torch::Tensor q, torch::Tensor k,
                  torch::Tensor v, torch::Tensor cu_seqlens,
                  torch::Tensor cu_seqlens_k, int64_t max_seqlen,
                  double scale, bool causal, int64_t window) {
  const int Hq = q.size(1);
  const int D = q.size(2);
  const int Hkv = k.size(1);
  const int B = cu_seqlens.size(0) - 1;
  TORCH_CHECK(cu_seqlens.scalar_type() == torch::kInt32 &&
              cu_seqlens_k.scalar_type() == torch::kInt32);
  TORCH_CHECK(D == 64 || D == 128, "head_dim must be 64 or 128");
  TORCH_CHECK(Hkv > 0 && Hq % Hkv == 0 && v.size(1) == Hkv &&
              k.size(2) == D && v.size(2) == D && v.size(0) == k.size(0));
  TORCH_CHECK(out.is_contiguous() && out.sizes() == q.sizes());
  if (B <= 0 || max_seqlen <= 0 || q.numel() == 0) return;
  q = rows(q);
  k = rows(k);
  v = rows(v);
  Prefill m{};
  m.cu_q = cu_seqlens.data_ptr<int>();
  m.cu_k = cu_seqlens_k.data_ptr<int>();
  m.q_stride = q.stride(0);
  m.k_stride = k.stride(0);
  m.v_stride = v.stride(0);
  m.Hq = Hq;
  m.G = Hq / Hkv;
  m.q_tiles = cdiv((int)max_seqlen, QT);
  m.seqs = B;
  m.window = (int)window;
  m.flip = scale < 0;
  m.mul = (float)std::abs(scale) * LOG2E;
  const dim3 grid(8 * cdiv(B * Hq, 8) * m.q_tiles);
  auto stream = at::hip::getCurrentHIPStream();
#define LAUNCH(DH, C)                                                        \
  hipLaunchKernelGGL((attn_prefill_kernel<DH, C>), grid, dim3(NT), 0,        \
                     stream, (uint16_t*)out.data_ptr(),                      \
                     (const uint16_t*)q.data_ptr(),                          \
                     (const uint16_t*)k.data_ptr(),                          \
                     (const uint16_t*)v.data_ptr(), m)
  if (causal) {
    if (D == 128) LAUNCH(128, true); else LAUNCH(64, true);
  } else {
    if (D == 128) LAUNCH(128, false); else LAUNCH(64, false);
  }
#undef LAUNCH
}
