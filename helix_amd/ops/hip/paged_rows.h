// Paged-attention decode (single query token per sequence) for CDNA4.
//
// Replaces the decode attention the reference delegates to vLLM. Bound by the
// cache: every key and value is read once for the G = Hq / Hkv query heads
// that share it.
//
//  - A wave works alone on tiles of 32 keys and passes nothing through LDS
//    until the waves of a workgroup put their results together, so no barrier
//    stands between loads. Keys go straight from their pages into MFMA
//    operands (scores key x query); they are permuted so that lane group hi
//    ends up with the scores of the 8 keys whose values it loads itself. The
//    query columns repeat every four lanes.
//  - From four heads on the value product runs on matrix instructions without
//    rounding the weights: a lane of each four has a head's weight in one of three
//    bf16 parts that add up to its 24 bits, so the 16 rows of an operand are four
//    heads in all parts, and a sum's are added at the end. Values meet them as
//    columns of 8 keys, which takes an instruction for every two. Up to two heads
//    the product runs in fp32, a weight of another head a quad broadcast away.
//    In fp32 it was most of a tile's instructions and kept e4m3 and eight heads
//    from the rate of the memory; us before and now: 64 heads on 8, 16 of
//    100..6000 53 and 49, e4m3 45 and 39, heads of 64 33 and 28, e4m3 28 and 23;
//    32 on 8 of 128, 61 of 1000..4096 118.8 and 117.0, e4m3 75.7 and 72.0, 512 of
//    513..640 e4m3 115.6 and 112.4. Distance from 64 bits the same (1.66e-3, the
//    rounding of results, of which 1 in 4000 differs).
//  - The next tile's keys are under way during softmax and value product, its
//    values during the next scores; page numbers are read a tile earlier.
//  - Work is cut by the lengths themselves, on the device, because a captured
//    graph only knows its bucket: all (sequence, head) pairs share TARGET
//    workgroups in proportion to their tokens, in units of 128. Sequences in
//    one piece are written at once, others are merged by a second launch. Short
//    or many rows are not cut at all (see `whole`).
//
// Before, a partition was a share of the bucket, its two waves met at three
// barriers per 128 tokens and the value product waited for the softmax of all
// heads. Measured with 32 heads on 8, 16-token pages in random order, merge
// included (us before -> now, TB/s now):
//   1 row of 777            22.5 -> 10.0      (launches and latency)
//   8 of 300..6000, window  89 -> 25          3.5
//   61 of 1000..4096        345 -> 117        5.3
//   512 of 513..640         279 -> 193        6.3
//   24 of 4000..16000, fp8  487 -> 99         5.0
// Values by ordinary loads: 133 us for the 61, 226 for the 512; keys by
// streaming loads as well: 128 and 218.
// The 512 take the same where every pass reads another of six caches of 1.2 GB, so
// theirs is the rate of the memory. TARGET of 512 to 2048 is within 5% of each
// other; the results' distance from 64 bits is what it was (their rounding to
// bf16).
#pragma once
#include "common.h"
#include <torch/extension.h>
#include <ATen/hip/HIPContext.h>
#include <cfloat>

namespace helix {
namespace paged {
namespace {

constexpr int NT = 256, NW = NT / WAVE;
constexpr int KT = 32;                        // keys of a tile
constexpr int UNIT = KT * NW;                 // tokens that work is cut in
constexpr int TARGET = 1024;                  // workgroups: 4 on each CU
constexpr float LOG2E = 1.4426950408889634f;
// Before the first key: below every score but those of no weight.
constexpr float LOWEST = -FLT_MAX;

struct Rows {
  const int* bt;               // [B, max_blocks]
  const int* lens;             // [B]
  uint16_t* out;               // [B, Hq, D]
  float* part;                 // [B, Hq, max_parts, D]
  float* ml;                   // [B, Hq, max_parts, 2]
  int B, Hkv, bs, shift, max_blocks, max_parts, window, limit;
  bool split, heads_first;     // whose neighbours are heads, not rows or pieces
  float mul;                   // scale * log2(e)
};

__device__ __forceinline__ float max_over_groups(float v) {
  const unsigned u = __float_as_uint(v);
  const auto a = __builtin_amdgcn_permlane32_swap(u, u, false, false);
  const float x = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
  const unsigned w = __float_as_uint(x);
  const auto b = __builtin_amdgcn_permlane16_swap(w, w, false, false);
  return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}
__device__ __forceinline__ float sum_over_groups(float v) {
  const unsigned u = __float_as_uint(v);
  const auto a = __builtin_amdgcn_permlane32_swap(u, u, false, false);
  const float x = __uint_as_float(a[0]) + __uint_as_float(a[1]);
  const unsigned w = __float_as_uint(x);
  const auto b = __builtin_amdgcn_permlane16_swap(w, w, false, false);
  return __uint_as_float(b[0]) + __uint_as_float(b[1]);
}

// Lane j of every four, in all four.
template <int J>
__device__ __forceinline__ float quad(float v) {
  return __int_as_float(__builtin_amdgcn_mov_dpp(
      __float_as_int(v), J * 0x55, 0xf, 0xf, true));
}
template <int J>
__device__ __forceinline__ float of_head(const float* v) {
  return quad<(J & 3)>(v[J >> 2]);
}

// Tokens that sequence b's query sees are [first, len); units are whole.
// No more than the caller's bound, which the grid is sized by.
__device__ __forceinline__ int len_of(const Rows& m, int b) {
  return min(m.lens[b], m.limit);
}
__device__ __forceinline__ int first_key(const Rows& m, int len) {
  return m.window > 0 ? max(0, len - m.window) : 0;
}
__device__ __forceinline__ int units_of(const Rows& m, int b) {
  if (b >= m.B) return 0;
  const int len = len_of(m, b);
  return len > 0 ? cdiv(len - first_key(m, len) / KT * KT, UNIT) : 0;
}

// Units of a workgroup such that all pieces come to about TARGET.
__device__ __forceinline__ int piece_for(const Rows& m, int units) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) units += __shfl_xor(units, off, WAVE);
  return max(1, cdiv(units * m.Hkv, TARGET));
}
// Pieces of a sequence (one, if it is empty: its zeros have to be written).
__device__ __forceinline__ int pieces_of(const Rows& m, int units, int c) {
  return min(max(1, cdiv(units, c)), m.max_parts);
}

// Number `left` of the pieces of 64 sequences, `mine` of them this lane's.
__device__ __forceinline__ bool find_in(int mine, int& left, int& at, int& p,
                                        int& n) {
  const int lane = threadIdx.x & (WAVE - 1);
  int upto = mine;
#pragma unroll
  for (int off = 1; off < WAVE; off <<= 1) {
    const int v = __shfl_up(upto, off, WAVE);
    if (lane >= off) upto += v;
  }
  const int total = __shfl(upto, WAVE - 1, WAVE);
  if (left >= total) {
    left -= total;
    return false;
  }
  at = __ffsll((unsigned long long)__ballot(left < upto)) - 1;
  n = __shfl(mine, at, WAVE);
  p = left - (__shfl(upto, at, WAVE) - n);
  return true;
}

// Sequence and piece number of workgroup `block`; false where none is left.
__device__ __forceinline__ bool find(const Rows& m, int block, int& seq, int& p,
                                     int& n) {
  seq = block;
  p = 0;
  n = 1;
  if (!m.split) return true;
  const int lane = threadIdx.x & (WAVE - 1);
  int left = block;
  if (m.B <= WAVE) {                          // each length is read once
    const int u = units_of(m, lane), c = piece_for(m, u);
    return find_in(lane < m.B ? pieces_of(m, u, c) : 0, left, seq, p, n);
  }
  int u = 0;
  for (int b = lane; b < m.B; b += WAVE) u += units_of(m, b);
  const int c = piece_for(m, u);
  for (int b0 = 0; b0 < m.B; b0 += WAVE) {
    const int b = b0 + lane;
    if (find_in(b < m.B ? pieces_of(m, units_of(m, b), c) : 0, left, seq, p,
                n)) {
      seq += b0;
      return true;
    }
  }
  return false;
}

// A key row's or value row's elements of this lane as they lie in memory.
template <int BYTES> struct Raw;
template <> struct Raw<4> { typedef uint32_t T; };
template <> struct Raw<8> { typedef u32x2 T; };
template <> struct Raw<16> { typedef u32x4 T; };
template <typename R>
__device__ __forceinline__ uint32_t word_of(const R& row, int i) {
  if constexpr (sizeof(R) == 4)
    return row;
  else
    return row[i];
}

template <bool F8, int DPL>
__device__ __forceinline__ void widen(const void* raw, float* v) {
  const uint32_t* w = (const uint32_t*)raw;
  if constexpr (F8) {
#pragma unroll
    for (int i = 0; i < DPL / 4; ++i) {
      const auto a = __builtin_amdgcn_cvt_pk_f32_fp8(w[i], false);
      const auto b = __builtin_amdgcn_cvt_pk_f32_fp8(w[i], true);
      v[4 * i] = a[0];
      v[4 * i + 1] = a[1];
      v[4 * i + 2] = b[0];
      v[4 * i + 3] = b[1];
    }
  } else {
#pragma unroll
    for (int i = 0; i < DPL / 2; ++i) {
      v[2 * i] = __uint_as_float(w[i] << 16);
      v[2 * i + 1] = __uint_as_float(w[i] & 0xffff0000u);
    }
  }
}

// 8 e4m3 values as bf16 (exact).
__device__ __forceinline__ bf16x8 widen8(uint32_t a, uint32_t b) {
  const auto p = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(a, 1.f, false);
  const auto q = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(a, 1.f, true);
  const auto r = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(b, 1.f, false);
  const auto s = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(b, 1.f, true);
  return bf16x8{p[0], p[1], q[0], q[1], r[0], r[1], s[0], s[1]};
}

// The part of the wave's work that every head adds for itself.
template <int G, int J, int DPL>
__device__ __forceinline__ void add_values(float (*acc)[DPL], const float* pg,
                                           const float* v) {
  if constexpr (J < G) {
    const float w = G == 1 ? pg[0] : of_head<J>(pg);
#pragma unroll
    for (int d = 0; d < DPL; ++d) acc[J][d] += w * v[d];
    add_values<G, J + 1, DPL>(acc, pg, v);
  }
}
template <int G, int J, int DPL>
__device__ __forceinline__ void rescale(float (*acc)[DPL], const float* c) {
  if constexpr (J < G) {
    const float w = G == 1 ? c[0] : of_head<J>(c);
#pragma unroll
    for (int d = 0; d < DPL; ++d) acc[J][d] *= w;
    rescale<G, J + 1, DPL>(acc, c);
  }
}

// Weights as three bf16 that add up to all their 24 bits: a lane's part is what the
// parts before it leave.
__device__ __forceinline__ float part_of(float w, bool second, bool third) {
  auto lower = [](float v) {
    return v - __uint_as_float(__float_as_uint(v) & 0xffff0000u);
  };
  const float a = lower(w);
  w = second ? a : w;
  const float b = lower(a);
  return third ? b : w;
}
// The upper (lower) halves of two words.
__device__ __forceinline__ uint32_t uppers(uint32_t a, uint32_t b) {
  return __builtin_amdgcn_perm(b, a, 0x07060302);
}
__device__ __forceinline__ uint32_t lowers(uint32_t a, uint32_t b) {
  return __builtin_amdgcn_perm(b, a, 0x05040100);
}
// Values 2 c and 2 c + 1 of a row.
template <bool F8, typename R>
__device__ __forceinline__ uint32_t two_values(const R& row, int c) {
  if constexpr (F8) {
    const uint32_t w = word_of(row, c >> 1);
    return __builtin_bit_cast(
        uint32_t, (c & 1) ? __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w, 1.f, true)
                          : __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w, 1.f, false));
  } else {
    return word_of(row, c);
  }
}

// What fits the registers without spilling.
constexpr int waves_per_simd(int D, int G) {
  return D == 128 ? (G > 4 ? 2 : 3) : (G > 4 ? 3 : 4);
}

// The waves' results.
template <int D, int G>
struct Shared {
  float sh[NW][G][D];
  float st[2][NW][G];
};

// Work of a workgroup: `block` of those of KV head g. The heads of an uncut row
// follow each other, so that a long row's lie on different XCDs (32 heads on 8, one of
// 1000 beside 63 of 100 27.8 us before and 18.9, 256 of 20..1000 104.4 and 99.6).
// PAGE8: pages are a power of two of at least 8 tokens, so the 8 keys of a
// lane group lie in one page.
template <int D, int G, bool F8, bool PAGE8>
__device__ __forceinline__ void rows(const uint16_t* __restrict__ q,
                                     const void* __restrict__ kc,
                                     const void* __restrict__ vc,
                                     Rows m, int block, int g,
                                     Shared<D, G>& lds) {
  constexpr int NC = D / 32;                  // inner steps of the scores
  constexpr int DPL = D / 16;                 // value dimensions of a lane
  constexpr int QS = G > 4 ? G / 4 : 1;       // sets of query columns
  constexpr int EB = F8 ? 1 : 2;              // bytes of a cached element
  // keys: a lane's 16 bytes of a row hold one step in bf16, two in e4m3
  constexpr int KL = F8 ? NC / 2 : NC;
  typedef typename Raw<DPL * EB>::T VRaw;
  auto& sh = lds.sh;
  auto& st = lds.st;

  const int lane = threadIdx.x & (WAVE - 1);
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
  const int lo = lane & 15, hi = lane >> 4;
  int seq, part, parts;
  if (!find(m, block, seq, part, parts)) return;
  // The same in all lanes: scalar registers, so that a wave more fits a SIMD. Not
  // for up to four heads of bf16, which have waves enough and lose by more (32
  // heads of 64 on 8, 16 of 100..6000 24 us and 26; 16 on 16 of 128, 1 of 900
  // 13.4 and 15.7; e4m3 of the first 20.5 and 19.4).
  if constexpr (F8 || G > 4) {
    seq = __builtin_amdgcn_readfirstlane(seq);
    part = __builtin_amdgcn_readfirstlane(part);
    parts = __builtin_amdgcn_readfirstlane(parts);
  }
  const int Hq = m.Hkv * G;
  const int len = len_of(m, seq), first = first_key(m, len);
  const int tile0 = first / KT, tiles = max(0, cdiv(len, KT) - tile0);
  const int per = cdiv(tiles, parts);
  const int t_end = tile0 + min(tiles, (part + 1) * per);
  int t = tile0 + part * per + wid;

  // Queries: the inner dimension is numbered as keys are loaded
  bf16x8 qf[QS][NC];
#pragma unroll
  for (int s = 0; s < QS; ++s)
#pragma unroll
    for (int j = 0; j < NC; ++j) {
      const int h = g * G + s * 4 + (lo & (G < 4 ? G - 1 : 3));
      const int d = F8 ? (j >> 1) * 64 + hi * 16 + (j & 1) * 8
                       : j * 32 + hi * 8;
      qf[s][j] = *reinterpret_cast<const bf16x8*>(
          q + ((int64_t)seq * Hq + h) * D + d);
    }

  const int* bt = m.bt + (int64_t)seq * m.max_blocks;
  const int last = len - 1;
  // the table is read from the window's first key on: a tile begins up to 31
  // before it, where pages may have been given back
  auto page = [&](int key) {
    key = max(min(key, last), first);
    return bt[PAGE8 ? key >> m.shift : key / m.bs];
  };
  // Byte offset of a key's row. With PAGE8 the rows of a lane group follow
  // each other; those past the end are there as well, and masked.
  auto row_at = [&](int pg, int key) {
    if constexpr (!PAGE8) key = min(key, last);
    const int off = PAGE8 ? key & (m.bs - 1) : key % m.bs;
    return (((int64_t)pg * m.Hkv + g) * m.bs + off) * (D * EB);
  };
  // operand row lo of half s is key 8 (lo / 4) + 4 s + lo % 4
  const int key_k = (lo >> 2) * 8 + (lo & 3), key_v = hi * 8;
  constexpr int KG = PAGE8 ? 1 : 2, VG = PAGE8 ? 1 : 8;
  int kp[KG], vp[VG];
  auto pages = [&](int tile) {
#pragma unroll
    for (int i = 0; i < KG; ++i) kp[i] = page(tile * KT + key_k + 4 * i);
#pragma unroll
    for (int i = 0; i < VG; ++i) vp[i] = page(tile * KT + key_v + i);
  };
  u32x4 kr[2][KL];
  VRaw vr[8];
  auto load_k = [&](int tile) {
    const char* row[2];
#pragma unroll
    for (int s = 0; s < 2; ++s)
      row[s] = s < KG ? (const char*)kc + hi * 16 +
                            row_at(kp[s % KG], tile * KT + key_k + 4 * s)
                      : row[0] + 4 * D * EB;
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int j = 0; j < KL; ++j)
        kr[s][j] = *reinterpret_cast<const u32x4*>(row[s] + j * 64);
  };
  auto load_v = [&](int tile) {
    const char* row[VG];
#pragma unroll
    for (int i = 0; i < VG; ++i)
      row[i] = (const char*)vc + row_at(vp[i], tile * KT + key_v + i) +
               lo * DPL * EB;
    // read once, by whole lines: they need not stay in the caches (keys come
    // by half lines and do)
#pragma unroll
    for (int i = 0; i < 8; ++i)
      vr[i] = __builtin_nontemporal_load(reinterpret_cast<const VRaw*>(
          row[i % VG] + (i / VG) * D * EB));
  };

  // from four heads on by matrix instructions: rows are 4 heads in each of the
  // weights' parts, columns the dimensions lo DPL + d
  constexpr bool MMA = G >= 4;
  float acc[MMA ? 1 : G][DPL], m_run[QS], l[QS];
  floatx4 sum[QS][MMA ? DPL : 1];
#pragma unroll
  for (int d = 0; d < DPL; ++d) {
#pragma unroll
    for (int j = 0; j < (MMA ? 1 : G); ++j) acc[j][d] = 0.f;
    if constexpr (MMA)
#pragma unroll
      for (int s = 0; s < QS; ++s) sum[s][d] = floatx4{0, 0, 0, 0};
  }
  const bool second = lo >= 4, third = lo >= 8;
#pragma unroll
  for (int s = 0; s < QS; ++s) {
    m_run[s] = LOWEST;
    l[s] = 0.f;
  }
  if (t < t_end) {
    pages(t);
    load_k(t);
    load_v(t);
    pages(min(t + NW, t_end - 1));
  }
  for (; t < t_end; t += NW) {
    const bool more = t + NW < t_end;
    floatx4 x[QS][2];
#pragma unroll
    for (int s = 0; s < QS; ++s)
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        x[s][u] = floatx4{0, 0, 0, 0};
#pragma unroll
        for (int j = 0; j < NC; ++j) {
          bf16x8 k;
          if constexpr (F8) {
            const u32x4 r = kr[u][j >> 1];
            k = (j & 1) ? widen8(r[2], r[3]) : widen8(r[0], r[1]);
          } else {
            k = __builtin_bit_cast(bf16x8, kr[u][j]);
          }
          x[s][u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(k, qf[s][j],
                                                            x[s][u], 0, 0, 0);
        }
      }
    load_k(more ? t + NW : t);
    __builtin_amdgcn_sched_barrier(0);
    const int key0 = t * KT + key_v;
    const bool edge = t * KT < first || (t + 1) * KT > len;
    float p[8][QS], corr[QS];
    bool keep = true;
#pragma unroll
    for (int s = 0; s < QS; ++s) {
      float mx = m_run[s];
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        float v = x[s][i >> 2][i & 3] * m.mul;
        if (edge && (key0 + i < first || key0 + i >= len)) v = -INFINITY;
        p[i][s] = v;
        mx = fmaxf(mx, v);
      }
      mx = max_over_groups(mx);
      corr[s] = __builtin_amdgcn_exp2f(m_run[s] - mx);
      keep = keep && mx == m_run[s];
      m_run[s] = mx;
      l[s] *= corr[s];
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        p[i][s] = __builtin_amdgcn_exp2f(p[i][s] - mx);
        l[s] += p[i][s];
      }
    }
    // nothing that lies past the end may meet even a weight of zero
    if (edge) {
#pragma unroll
      for (int i = 0; i < 8; ++i)
        vr[i] = key0 + i < first || key0 + i >= len ? VRaw(0) : vr[i];
    }
    if constexpr (MMA) {
      if (!__all(keep)) {
#pragma unroll
        for (int s = 0; s < QS; ++s) {
          const floatx4 c = {quad<0>(corr[s]), quad<1>(corr[s]),
                             quad<2>(corr[s]), quad<3>(corr[s])};
#pragma unroll
          for (int d = 0; d < DPL; ++d)
#pragma unroll
            for (int r = 0; r < 4; ++r) sum[s][d][r] *= c[r];
        }
      }
      u32x4 w[QS];
#pragma unroll
      for (int s = 0; s < QS; ++s)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          w[s][i] = uppers(
              __float_as_uint(part_of(p[2 * i][s], second, third)),
              __float_as_uint(part_of(p[2 * i + 1][s], second, third)));
#pragma unroll
      for (int c = 0; c < DPL / 2; ++c) {
        uint32_t two[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) two[i] = two_values<F8>(vr[i], c);
        u32x4 even, odd;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          even[i] = lowers(two[2 * i], two[2 * i + 1]);
          odd[i] = uppers(two[2 * i], two[2 * i + 1]);
        }
#pragma unroll
        for (int s = 0; s < QS; ++s) {
          const bf16x8 ws = __builtin_bit_cast(bf16x8, w[s]);
          sum[s][2 * c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              ws, __builtin_bit_cast(bf16x8, even), sum[s][2 * c], 0, 0, 0);
          sum[s][2 * c + 1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              ws, __builtin_bit_cast(bf16x8, odd), sum[s][2 * c + 1], 0, 0, 0);
        }
        // else all values are widened at once and registers run out
        __builtin_amdgcn_sched_barrier(0);
      }
    } else {
      if (!__all(keep)) rescale<G, 0, DPL>(acc, corr);
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        float v[DPL];
        widen<F8, DPL>(&vr[i], v);
        add_values<G, 0, DPL>(acc, p[i], v);
        // else all values are widened at once and registers run out
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    load_v(more ? t + NW : t);
    pages(min(t + 2 * NW, t_end - 1));
  }

  // the lane groups, then the waves together
#pragma unroll
  for (int s = 0; s < QS; ++s) {
    l[s] = sum_over_groups(l[s]);
    if (lane < min(4, G)) {
      st[0][wid][s * 4 + lane] = m_run[s];
      st[1][wid][s * 4 + lane] = l[s];
    }
  }
#pragma unroll
  for (int j = 0; j < G; ++j)
#pragma unroll
    for (int d = 0; d < DPL; ++d) {
      if constexpr (MMA) {
        // the parts; infinite values count by the first, as a later one may be 0
        const float first = sum[j >> 2][d][j & 3];
        const float all = sum_over_groups(hi < 3 ? first : 0.f);
        if (hi == 0)
          sh[wid][j][lo * DPL + d] = fabsf(first) <= FLT_MAX ? all : first;
      } else {
        const float v = sum_over_groups(acc[j][d]);
        if (hi == (j & 3)) sh[wid][j][lo * DPL + d] = v;
      }
    }
  __syncthreads();
  for (int i = threadIdx.x; i < G * D; i += NT) {
    const int j = i / D, d = i % D;
    float top = LOWEST, sum = 0.f, o = 0.f;
#pragma unroll
    for (int w = 0; w < NW; ++w) top = fmaxf(top, st[0][w][j]);
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      const float f = __builtin_amdgcn_exp2f(st[0][w][j] - top);
      sum += f * st[1][w][j];
      o += f * sh[w][j][d];
    }
    const int64_t row = (int64_t)seq * Hq + g * G + j;
    if (parts == 1) {
      // zeros where there are no keys; scores of -inf alone are no number
      m.out[row * D + d] = f32_to_bf16(len > 0 ? o / sum : 0.f);
    } else {
      const int64_t at = row * m.max_parts + part;
      m.part[at * D + d] = o;
      if (d == 0) {
        m.ml[at * 2] = top;
        m.ml[at * 2 + 1] = sum;
      }
    }
  }
}

// Pieces of a sequence into one: a workgroup has a query head, each of its
// D / 4 lanes four dimensions of every eighth (D = 64: sixteenth) piece.
template <int D>
__global__ __launch_bounds__(NT) void paged_merge_kernel(Rows m, int Hq) {
  constexpr int LANES = D / 4, ROWS = NT / LANES;
  __shared__ f32x4 os[ROWS][LANES];
  __shared__ float ls[ROWS];
  const int seq = blockIdx.x, tid = threadIdx.x;
  int u = 0;
  for (int b = tid & (WAVE - 1); b < m.B; b += WAVE) u += units_of(m, b);
  const int parts = pieces_of(m, units_of(m, seq), piece_for(m, u));
  if (parts == 1) return;
  const int64_t row = (int64_t)seq * Hq + blockIdx.y;
  const float2* ml = (const float2*)m.ml + row * m.max_parts;
  const float* part = m.part + row * m.max_parts * D + tid % LANES * 4;
  float top = LOWEST;
  for (int p = tid & (WAVE - 1); p < parts; p += WAVE)
    top = fmaxf(top, ml[p].x);
  top = wave_reduce_max(top);
  f32x4 o = {0, 0, 0, 0};
  float sum = 0.f;
#pragma unroll 4
  for (int p = tid / LANES; p < parts; p += ROWS) {
    const float2 v = ml[p];
    const f32x4 x = *reinterpret_cast<const f32x4*>(part + (int64_t)p * D);
    const float f = __builtin_amdgcn_exp2f(v.x - top);
    sum += f * v.y;
#pragma unroll
    for (int i = 0; i < 4; ++i) o[i] += f * x[i];
  }
  os[tid / LANES][tid % LANES] = o;
  if (tid % LANES == 0) ls[tid / LANES] = sum;
  __syncthreads();
  if (tid >= D) return;
  float s = 0.f, r = 0.f;
#pragma unroll
  for (int i = 0; i < ROWS; ++i) {
    s += ls[i];
    r += os[i][tid / 4][tid % 4];
  }
  m.out[row * D + tid] = f32_to_bf16(r / s);
}

// Work of a call and the workgroups it takes, checked (no rows: m.B is 0). q is
// copied where it does not begin on 16 bytes.
struct Plan {
  Rows m{};
  int pieces, Hq, D, G;                       // pieces: workgroups of a KV head
  bool f8;
};

inline Plan plan(torch::Tensor out, torch::Tensor& q, torch::Tensor k_cache,
                 torch::Tensor v_cache, torch::Tensor block_tables,
                 torch::Tensor seq_lens, double scale, torch::Tensor tmp_out,
                 torch::Tensor tmp_ml, int64_t max_len_hint, int64_t window) {
  Plan p;
  const int B = q.size(0);
  const int Hq = q.size(1);
  const int D = q.size(2);
  const int Hkv = k_cache.size(1);
  const int G = Hq / Hkv;
  TORCH_CHECK(D == 64 || D == 128, "head_dim must be 64 or 128");
  TORCH_CHECK(G <= 8 && Hq % Hkv == 0);
  TORCH_CHECK(G == 1 || G == 2 || G == 4 || G == 8, "G must be 1/2/4/8");
  TORCH_CHECK(block_tables.scalar_type() == torch::kInt32);
  TORCH_CHECK(seq_lens.scalar_type() == torch::kInt32);
  p.Hq = Hq;
  p.D = D;
  p.G = G;
  p.f8 = k_cache.scalar_type() == torch::kUInt8;
  if (B == 0) return p;
  // everything below goes by raw addresses
  TORCH_CHECK(q.is_contiguous() && q.scalar_type() == torch::kBFloat16,
              "q is packed bf16");
  TORCH_CHECK(out.is_contiguous() && out.scalar_type() == q.scalar_type() &&
              out.sizes() == q.sizes(), "out is packed bf16 of q's shape");
  TORCH_CHECK((k_cache.scalar_type() == torch::kBFloat16 ||
               k_cache.scalar_type() == torch::kUInt8) &&
              v_cache.scalar_type() == k_cache.scalar_type() &&
              k_cache.is_contiguous() && v_cache.is_contiguous() &&
              v_cache.sizes() == k_cache.sizes() && k_cache.size(3) == D,
              "caches are packed pages of q's head_dim, bf16 or e4m3");
  TORCH_CHECK(block_tables.is_contiguous() && block_tables.size(0) >= B &&
              seq_lens.is_contiguous() && seq_lens.numel() >= B,
              "a length and a row of the table for every sequence");
  if ((uintptr_t)q.data_ptr() % 16 != 0) q = q.clone();

  Rows& m = p.m;
  m.bt = block_tables.data_ptr<int>();
  m.lens = seq_lens.data_ptr<int>();
  m.out = (uint16_t*)out.data_ptr();
  m.part = tmp_out.data_ptr<float>();
  m.ml = tmp_ml.data_ptr<float>();
  m.B = B;
  m.Hkv = Hkv;
  m.bs = k_cache.size(2);
  m.shift = (m.bs & (m.bs - 1)) == 0 ? __builtin_ctz(m.bs) : -1;
  m.max_blocks = block_tables.size(1);
  m.max_parts = tmp_out.size(2);
  m.window = (int)window;
  // nor more than the table has pages for
  m.limit = (int)std::min<int64_t>(
      cdiv((int)max_len_hint, UNIT) * UNIT, (int64_t)m.max_blocks * m.bs);
  m.mul = (float)scale * LOG2E;
  // A row in one workgroup needs no search for its piece and no second launch, but
  // takes as long as its length, and the chip waits for the longest. Cut only where
  // that is the longer of the two; the graph knows rows and bound, not lengths. us
  // cut and uncut, 32 heads on 8 of 128, lengths up to the bound evenly spread:
  //   512 and below: 1 row of 512 10.1 and 10.1, of 300 10.0 and 8.4; 16 rows 13.3
  //     and 10.4, 64 28.0 and 17.3. With 8 heads of 128 a row's own time is longer:
  //     1 row of 512 13.0 and 14.4, 8 13.6 and 14.6, but 16 16.7 and 14.7.
  //   1024: 8 rows 13.3 and 16.1, 16 17.0 and 16.4, 32 22.8 and 18.2, 128 61.3 and
  //     53.5 (e4m3 40.1 and 28.5). The least good are single long rows: one of 1000
  //     beside 47 of 100 16.9 and 18.9.
  //   2048: 16 heads on 8, 128 rows 103 and 108, 256 198 and 187; one of 2036 beside
  //     255 of 100 46 and 37.
  const int most = cdiv((int)(window > 0 ? std::min(max_len_hint, window + KT)
                                         : max_len_hint), UNIT);
  const int64_t rows = (int64_t)B * Hkv;
  const bool cuts = m.max_parts > 1 && most > 1 &&
                    !(rows >= 2 * TARGET && most <= 8);
  const bool whole = (most <= 4 && (rows >= 128 || G * D < 1024)) ||
                     (most <= 8 && rows >= 128) ||
                     (most <= 16 && rows >= 2 * TARGET);
  m.split = cuts && !whole;
  m.heads_first = !m.split && B < 1 << 16;    // a grid has no more along y
  // a workspace is looked at whether or not these rows would be cut
  const int64_t pieces = (int64_t)B * Hq * m.max_parts;
  TORCH_CHECK(!cuts || (tmp_out.is_contiguous() && tmp_ml.is_contiguous() &&
                        tmp_out.numel() >= pieces * D &&
                        tmp_ml.numel() >= pieces * 2),
              "a workspace of [B, Hq, parts, D] and [B, Hq, parts, 2]");
  for (const auto& t : {q, out, k_cache, v_cache, block_tables, seq_lens,
                        tmp_out, tmp_ml})
    TORCH_CHECK(t.is_cuda() && t.device() == q.device(),
                "everything on one GPU");
  // a workgroup without a piece costs its search, so no more than can be
  p.pieces = m.split ? std::min(B * most, B + TARGET / Hkv + 1) : B;
  return p;
}

// Pieces of sequences into one, where there are any.
inline void merge(const Plan& p, hipStream_t stream) {
  if (!p.m.split) return;
  const dim3 grid(p.m.B, p.Hq);
  if (p.D == 128)
    hipLaunchKernelGGL(paged_merge_kernel<128>, grid, dim3(NT), 0, stream, p.m,
                       p.Hq);
  else
    hipLaunchKernelGGL(paged_merge_kernel<64>, grid, dim3(NT), 0, stream, p.m,
                       p.Hq);
}

}  // namespace
}  // namespace paged
}  // namespace helix
