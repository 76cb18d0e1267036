// Flash-attention prefill (varlen, causal/bidirectional, GQA) for CDNA4.
//
// Replaces the prefill attention the reference delegates to vLLM. Bound by
// instruction issue and, at long contexts, by power: a wave takes 1876 cycles a
// tile, its products 1020 and its 200 vector instructions 1050 (one in 5), and
// the clock is at 1.75 GHz (on zeros 1 x 8192 takes 403 us instead of 562). LDS
// is busy for a quarter. A third wave on a SIMD (tiles of 32 keys), the next
// scores computed beside the exponentials and two halves of waves a phase apart
// change nothing or cost.
//
//  - A workgroup has 128 queries of one head, each of its 4 waves 32 of them,
//    in products of 32x32. Scores are computed transposed (key x query): a lane
//    has one query, its statistics cost one lane swap, and 8 neighbouring keys
//    of its weights are an operand of the value product as they lie.
//  - Tiles of 64 keys and values go straight to LDS, the next one while the
//    last is worked on, with one barrier a tile. Rows lie as in memory; their
//    16-byte pieces are stored crosswise, so that keys leave LDS as operands
//    and values through the transposing load without bank conflicts.
//  - The loop has a body for each of the two buffers, and places in memory are
//    unsigned 32-bit offsets from a scalar base: no addresses are computed in
//    it.
//  - The heads that share keys run on one XCD, the latest queries, which see the
//    most keys, first. Such groups go round the XCDs: with each XCD's sequences in
//    a row, the one with the longest took 1.2 to 1.3 times the mean of them. Waves
//    past the last query only load. us alone, before -> now: 64 texts 52 -> 49, 31
//    of 400..620 154 -> 146, 2000 and 5000 467 -> 262, 1 x 8192 560 -> 528; in steps
//    between products, where the clock is lower, the second takes 164, the last 561.
//    Some sizes lose by the order: 3 x 600 22.7 -> 23.8.
//
// 32 heads on 8 of 128, us of the first kernel (64 queries, values transposed
// element by element) -> products of 16x16 with addresses computed per tile
// (340 vector instructions) -> with the next tile's loads waited for by reads of
// LDS -> as now but for the heads' order (TFLOP/s; the last two on one card): 1 x
// 8192 2551 -> 645 ->
// 579 -> 568 (968), 8 x 2048 1918 -> 413 -> 364 -> 341 (806), 31 of 400..620
// 440 -> 188 -> 168 -> 154 (467), 1500 behind 5001 with a window of 4096 466 ->
// 173 -> 136 -> 130 (773). 12 heads of 64, 64 texts of 20..500: 178 -> 68 -> 52
// -> 49.6; 16 heads, 8 x 288: 12.5 -> 10.6. Workgroups of 64 queries
// (2 waves) took 1.1 to 1.8 times as long from 100 queries on, and no less time
// below. The distance from 64 bits is what it was.
//
// MFMA fragment layouts (gfx950, f32_32x32x16_bf16), hi = lane / 32,
// lo = lane % 32: A[lo][8 hi + i], B[8 hi + i][lo],
// D[8 (r / 4) + 4 hi + r % 4][lo].
#pragma once
#include "hybrid/tile.h"
#include <torch/extension.h>
#include <ATen/hip/HIPContext.h>
#include <cfloat>

namespace helix {
namespace prefill {
namespace {

constexpr int NT = 256, NW = NT / WAVE;
constexpr int QT = NW * 32;                   // queries of a workgroup
constexpr int KT = 64;                        // keys of a tile
constexpr float LOG2E = 1.4426950408889634f;
// Before the first key: below every score but those of no weight.
constexpr float LOWEST = -FLT_MAX;
// A weight is 2^(score mul - maximum mul), in one operation: what is rounded
// off maximum mul is in all weights alike and falls out, until it exceeds the
// exponents (from 2^31 on, 2^6 before). Scores that differ at all are then 2^7
// apart and only the largest counts, for any factor as large; a power of two
// rounds nothing off.
constexpr float FAR = 0x1p31f;
// instruction classes of the scheduling hints
constexpr int MFMA = 0x008, DS_READ = 0x100;

struct Prefill {
  const int* cu_q;             // [B + 1] query rows
  const int* cu_k;             // [B + 1] key rows (>= query rows)
  int64_t q_stride, k_stride, v_stride;       // of a row, in elements
  int Hq, G, groups, q_tiles, seqs, window;   // groups: of G heads
  bool flip;                   // negative scale: of negated queries
  bool spread;                 // groups of heads go round the XCDs
  int whole;                   // spread: rounds in which each XCD has a group
  int in_round;                // workgroups of a round
  float mul, far_mul;          // |scale| * log2(e); a power of two above it
};

typedef __attribute__((ext_vector_type(16))) float floatx16;

__device__ __forceinline__ floatx16 mfma32(u16x8 a, u16x8 b, floatx16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(
      __builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0,
      0);
}

__device__ __forceinline__ float max_over_halves(float v) {
  const unsigned u = __float_as_uint(v);
  const auto a = __builtin_amdgcn_permlane32_swap(u, u, false, false);
  return fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
}

// Four rows of one column from LDS: the 16 lanes of a quarter wave name 4
// rows x 16 columns, 4 columns each (lane j: row j / 4, columns 4 (j % 4)..),
// and get a column each.
__device__ __forceinline__ u16x4 ld_tr4(const uint16_t* p) {
  typedef __attribute__((ext_vector_type(4))) int16_t i16x4;
  return __builtin_bit_cast(u16x4, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
      (__attribute__((address_space(3))) i16x4*)p));
}

// 64 lanes' 16 bytes at base + offset to 1024 bytes of LDS. As a builtin the
// compiler lets every transposing read wait for all such loads, the next tile's
// among them; here the barrier of a tile alone does, after its own wait.
__device__ __forceinline__ void direct_load(const char* base, unsigned offset,
                                            uint16_t* lds) {
#ifdef __HIP_DEVICE_COMPILE__
  const unsigned to = (unsigned)(uintptr_t)(
      __attribute__((address_space(3))) uint16_t*)lds;
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\t"
               "global_load_lds_dwordx4 %0, %1"
               ::"v"(offset), "s"(base), "s"(to) : "memory", "m0");
#endif
}

// Piece p of row r lies at p ^ cross(r): 16 rows of a score operand, and 4
// rows of 4 pieces of a value operand, meet every bank equally.
template <int D>
__device__ __forceinline__ int cross(int r) {
  return D == 128 ? (r & 3) << 2 | (r >> 2 & 3)
                  : (r >> 1 & 1) << 2 | (r >> 2 & 3);
}

// Bytes of LDS that a workgroup takes.
constexpr int lds_of(int D) { return 4 * KT * D * 2; }

// A workgroup's XCD, tile of queries (latest first), head within its group and the
// group's number among those of this XCD. Not spread: heads are groups of their own.
struct Place {
  int xcd, head, tile, round;
};
// By a number within a round and the round's, or by one number, which is a division
// more.
__device__ __forceinline__ Place place_of(const Prefill& m, int block,
                                          int round) {
  const int in = block >> 3;
  if (!m.spread || m.G == 1) return {block & 7, 0, in, round};
  const int tile = in / m.G;
  return {block & 7, in - tile * m.G, tile, round};
}
__device__ __forceinline__ Place place_of(const Prefill& m, int block) {
  const int round = block / m.in_round;
  return place_of(m, block - round * m.in_round, round);
}

// tiles: lds_of(D) bytes
template <int D, bool CAUSAL>
__device__ __forceinline__ void queries(uint16_t* __restrict__ out,
                                        const uint16_t* __restrict__ q,
                                        const uint16_t* __restrict__ k,
                                        const uint16_t* __restrict__ v,
                                        Prefill m, Place at, uint16_t* tiles) {
  constexpr int NK = D / 16, NV = D / 32, PR = D / 8;
  constexpr int LOADS = KT * PR / NT;
  uint16_t* const kl[2] = {tiles, tiles + KT * D};
  uint16_t* const vl[2] = {tiles + 2 * KT * D, tiles + 3 * KT * D};
  int b, g, h;
  if (m.spread && at.round < m.whole) {
    const int group = at.round * 8 + at.xcd;
    b = group / m.groups;
    g = group - b * m.groups;
    h = g * m.G + at.head;
  } else {
    // heads one by one: of all groups, or of those that are too few for a round
    const int from = m.spread ? m.whole * 8 * m.G : 0;
    const int left = m.seqs * m.Hq - from, chunk = cdiv(left, 8);
    const int in = m.spread ? at.head : at.round, item = at.xcd * chunk + in;
    if (in >= chunk || item >= left) return;
    const int sh = from + item;
    b = sh / m.Hq;
    h = sh - b * m.Hq;
    g = h / m.G;
  }
  const int q0 = (m.q_tiles - 1 - at.tile) * QT;
  const int row0 = m.cu_q[b], qlen = m.cu_q[b + 1] - row0;
  if (q0 >= qlen) return;
  const int key0 = m.cu_k[b], klen = m.cu_k[b + 1] - key0;
  const int ctx = klen - qlen;                // cached tokens before

  const int tid = threadIdx.x, lane = tid & (WAVE - 1);
  const int wid = __builtin_amdgcn_readfirstlane(tid / WAVE);
  const int lo = lane & 31, hi = lane >> 5;
  // a wave without queries only loads; which of the four that is goes round, or
  // one SIMD would have all of them
  const int qw = q0 + (wid + at.head + at.round & 3) * 32;
  const bool idle = qw >= qlen;
  u16x8 qf[NK];
  const int qi = qw + lo;                     // of this lane
  {
    const uint16_t* qr =
        q + (row0 + min(qi, qlen - 1)) * m.q_stride + h * D + hi * 8;
#pragma unroll
    for (int c = 0; c < NK; ++c) {
      qf[c] = ld_u16x8(qr + c * 16);
      if (m.flip) qf[c] ^= (uint16_t)0x8000;
    }
  }

  const uint16_t* kb = k + key0 * m.k_stride + g * D;
  const uint16_t* vb = v + key0 * m.v_stride + g * D;
  // This lane's pieces of a tile: where they lie is the same in every tile but
  // a partial one, whose rows past the end repeat the last and are masked.
  unsigned ko[LOADS], vo[LOADS];
  auto places = [&](int rows, int64_t stride, unsigned* o) {
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
      const int e = (i * NW + wid) * WAVE + lane, r = e / PR;
      o[i] = (min(r, rows - 1) * (int)stride + (e % PR ^ cross<D>(r)) * 8) * 2;
      asm volatile("" : "+v"(o[i]));         // kept, not computed again
    }
  };
  auto fetch = [&](const uint16_t* base, int64_t stride, unsigned* o, int t,
                   uint16_t* lds) {
    if (t + KT > klen) places(klen - t, stride, o);
    const char* from = (const char*)(base + t * stride);
#pragma unroll
    for (int i = 0; i < LOADS; ++i)
      direct_load(from, o[i], lds + (i * NW + wid) * WAVE * 8);
  };
  places(KT, m.k_stride, ko);
  places(KT, m.v_stride, vo);
  // Where this lane reads. Keys: row 8 a + 4 h + b of a score operand is key
  // 16 (a / 2) + 8 h + 4 (a % 2) + b of its 32, so that a lane's scores 8 i..
  // are the neighbouring keys 16 i + 8 hi.., an operand of the value product.
  // Values: columns 32 d.. of keys 8 hi.. and of the 4 behind them.
  int ka[NK], va[NV][2];
  const int kr = (lo >> 4) * 16 + (lo >> 2 & 1) * 8 + (lo >> 3 & 1) * 4 +
                 (lo & 3);
#pragma unroll
  for (int c = 0; c < NK; ++c)
    ka[c] = kr * D + ((c * 2 + hi) ^ cross<D>(kr)) * 8;
#pragma unroll
  for (int d = 0; d < NV; ++d)
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int r = hi * 8 + j * 4 + (lo >> 2 & 3);
      va[d][j] = r * D +
                 ((d * 4 + (lo >> 4) * 2 + (lo >> 1 & 1)) ^ cross<D>(r)) * 8 +
                 (lo & 1) * 4;
    }

  floatx16 acc[NV];
  float m_run = LOWEST, l = 0.f, mul = m.mul;
#pragma unroll
  for (int d = 0; d < NV; ++d) acc[d] = floatx16{};
  const int last = CAUSAL ? min(klen, ctx + q0 + QT) : klen;
  const int qa = ctx + qw, qz = qa + 31;      // of this wave
  const bool windowed = CAUSAL && m.window > 0;
  int t = windowed ? max(0, ctx + q0 - m.window + 1) / KT * KT : 0;

  if (t < last) {
    fetch(kb, m.k_stride, ko, t, kl[0]);
    fetch(vb, m.v_stride, vo, t, vl[0]);
  }
  auto step = [&](auto half) {
    constexpr int buf = decltype(half)::value;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (t + KT < last) {
      fetch(kb, m.k_stride, ko, t + KT, kl[buf ^ 1]);
      fetch(vb, m.v_stride, vo, t + KT, vl[buf ^ 1]);
    }
    if (idle || (CAUSAL && t > qz)) return;
    floatx16 s[KT / 32];
#pragma unroll
    for (int w = 0; w < KT / 32; ++w) s[w] = floatx16{};
#pragma unroll
    for (int c = 0; c < NK; ++c)
#pragma unroll
      for (int w = 0; w < KT / 32; ++w)
        s[w] = mfma32(ld_u16x8(kl[buf] + w * 32 * D + ka[c]), qf[c], s[w]);
    // operands leave LDS a group ahead of their products
    __builtin_amdgcn_sched_group_barrier(DS_READ, 4, 0);
#pragma unroll
    for (int i = 0; i < NK - 2; ++i) {
      __builtin_amdgcn_sched_group_barrier(MFMA, 2, 0);
      __builtin_amdgcn_sched_group_barrier(DS_READ, 2, 0);
    }
    __builtin_amdgcn_sched_group_barrier(MFMA, 4, 0);

    // heads of 64 have as much to do here as in products: the other wave's
    // products go first (8 x 288 11.6 -> 10.5 us; heads of 128 lose 1 to 2%)
    if (D == 64) __builtin_amdgcn_s_setprio(0);
    const bool edge = (CAUSAL && t + KT - 1 > qa) || t + KT > klen ||
                      (windowed && t <= qz - m.window);
    if (edge) {
      const int at = ctx + qi;
      const int low = windowed ? at - m.window : -1;
      const int top = CAUSAL ? min(at, klen - 1) : klen - 1;
#pragma unroll
      for (int w = 0; w < KT / 32; ++w)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const int key = t + w * 32 + (i >> 3) * 16 + hi * 8 + (i & 7);
          if (key > top || key <= low) s[w][i] = -INFINITY;
        }
    }
    float mx = m_run;
#pragma unroll
    for (int w = 0; w < KT / 32; ++w)
#pragma unroll
      for (int i = 0; i < 16; ++i) mx = fmaxf(mx, s[w][i]);
    mx = max_over_halves(mx);
    if (!__all(mx == m_run)) {
      const float corr = __builtin_amdgcn_exp2f((m_run - mx) * m.mul);
      l *= corr;
      m_run = mx;
      mul = fabsf(mx * m.mul) < FAR ? m.mul : m.far_mul;
#pragma unroll
      for (int d = 0; d < NV; ++d)
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[d][i] *= corr;
    }
    // a query that has seen no key yet keeps weights of exactly zero
    const float base = m_run <= LOWEST ? 0.f : m_run * mul;
    u16x8 pf[KT / 16];
#pragma unroll
    for (int k = 0; k < KT / 16; ++k) {
      float p[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        p[i] = __builtin_amdgcn_exp2f(
            fmaf(s[k >> 1][(k & 1) * 8 + i], mul, -base));
        l += p[i];
      }
      pf[k] = pack8(p);
    }
    if (D == 64) __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int k = 0; k < KT / 16; ++k)
#pragma unroll
      for (int d = 0; d < NV; ++d) {
        const u16x4 x = ld_tr4(vl[buf] + k * 16 * D + va[d][0]);
        const u16x4 y = ld_tr4(vl[buf] + k * 16 * D + va[d][1]);
        const u16x8 a = {x[0], x[1], x[2], x[3], y[0], y[1], y[2], y[3]};
        acc[d] = mfma32(a, pf[k], acc[d]);
      }
    __builtin_amdgcn_sched_group_barrier(DS_READ, 4, 0);
#pragma unroll
    for (int i = 0; i < KT / 16 * NV - 2; ++i) {
      __builtin_amdgcn_sched_group_barrier(MFMA, 1, 0);
      __builtin_amdgcn_sched_group_barrier(DS_READ, 2, 0);
    }
    __builtin_amdgcn_sched_group_barrier(MFMA, 2, 0);
  };
  while (t < last) {
    step(std::integral_constant<int, 0>());
    if ((t += KT) >= last) break;
    step(std::integral_constant<int, 1>());
    t += KT;
  }

  l += __shfl_xor(l, 32, WAVE);
  if (qi >= qlen) return;
  // zeros where a query sees no key; scores of -inf alone are no number
  const int top = CAUSAL ? min(ctx + qi, klen - 1) : klen - 1;
  const bool sees = top >= (windowed ? max(0, ctx + qi - m.window + 1) : 0);
  const float f = sees ? 1.f / l : 0.f;
  uint16_t* dst = out + ((int64_t)(row0 + qi) * m.Hq + h) * D + hi * 4;
#pragma unroll
  for (int d = 0; d < NV; ++d)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float x[4] = {acc[d][i * 4] * f, acc[d][i * 4 + 1] * f,
                          acc[d][i * 4 + 2] * f, acc[d][i * 4 + 3] * f};
      st_bf16x4(dst + d * 32 + i * 8, x);
    }
}

// Rows of [T, H, D] with their heads side by side, 16-byte aligned, anywhere;
// other layouts are copied. Places within a tile are 32-bit byte offsets.
inline torch::Tensor rows(const torch::Tensor& t) {
  const bool fits = t.stride(2) == 1 && t.stride(1) == t.size(2) &&
                    t.stride(0) % 8 == 0 && t.stride(0) > 0 &&
                    t.stride(0) < (1 << 23);
  const torch::Tensor r = fits ? t : t.contiguous();
  return (uintptr_t)r.data_ptr() % 16 == 0 ? r : r.clone();
}

// Work of a call and its workgroups, checked (none: blocks is 0). q, k and v are copied
// where the kernel would not read them as they lie.
struct Plan {
  Prefill m{};
  int rounds = 0;
  int blocks() const { return m.in_round * rounds; }
};

inline Plan plan(torch::Tensor out, torch::Tensor& q, torch::Tensor& k,
                 torch::Tensor& v, torch::Tensor cu_seqlens,
                 torch::Tensor cu_seqlens_k, int64_t max_seqlen, double scale,
                 int64_t window) {
  Plan p;
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
  for (const auto& t : {out, q, k, v})
    TORCH_CHECK(t.scalar_type() == torch::kBFloat16, "rows are bf16");
  TORCH_CHECK(cu_seqlens.is_contiguous() && cu_seqlens_k.is_contiguous() &&
              cu_seqlens_k.numel() >= B + 1, "a boundary more than sequences");
  for (const auto& t : {out, q, k, v, cu_seqlens, cu_seqlens_k})
    TORCH_CHECK(t.is_cuda() && t.device() == q.device(),
                "everything on one GPU");
  if (B <= 0 || max_seqlen <= 0 || q.numel() == 0) return p;
  Prefill& m = p.m;
  m.mul = (float)std::abs(scale) * LOG2E;
  if (m.mul == 0.f) {          // masks are set on scores before they are scaled
    q = at::zeros_like(q);
    m.mul = LOG2E;
  }
  m.far_mul = (float)std::ldexp(1.0, std::ilogb(m.mul) + 1);
  q = rows(q);
  k = rows(k);
  v = rows(v);
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
  // Groups of heads that share keys go round the XCDs, and each sees some of every
  // sequence, whatever their lengths; a few that leave XCDs without one are cut
  // into heads, and so are those left over by whole rounds: the XCDs that had one
  // of them more took that much longer (28 heads on 4, 9 x 128 12.4 us, 10.0
  // now; 8 on 1, 41 x 600 65.6 and 62.8; 24 on 3, 17 x 600 77.8 and 75.5).
  m.groups = Hkv;
  const int groups = B * Hkv;
  m.spread = groups % 8 == 0 || groups >= 32;
  m.whole = groups / 8;
  m.in_round = 8 * m.q_tiles * (m.spread ? m.G : 1);
  p.rounds = cdiv(m.spread ? groups : B * Hq, 8);
  return p;
}

}  // namespace
}  // namespace prefill
}  // namespace helix
