// Products of bf16 matrices, x[M,K] @ w[N,K]^T with fp32 sums, by persistent
// workgroups whose loads never pause. gemm_bf16.hip and gemm_gated.hip choose
// the tile and launch.
//
// Bound by the matrix cores, and for large products by the power they draw (the
// clock falls to 1.7 to 1.9 GHz). A workgroup has one wave a SIMD, 2 x 2 of
// them, each with 16 MI x 16 NI sums in accumulation registers:
//
//  - Tiles of 64 of the inner dimension go straight to LDS, as many steps ahead
//    as 160 KB hold. Rows are 128 bytes, so a load takes whole cache lines
//    (with 32 of the inner dimension at a time 8192 x 4096 x 4096 took 204 us,
//    with 64 185). 16-byte piece p of row r lies at p ^ r / 2 % 8: operands
//    leave LDS without bank conflicts.
//  - A step has two halves of 32. While one is multiplied, the operands of the
//    next one come from LDS and a later step's loads are ordered, one of them at
//    a time between two products: what stands together holds the matrix cores
//    up (2423 cycles a step of 256 x 256 with a read, a load and then four
//    products, 2286 one by one; the products alone take 2048). One barrier a
//    step.
//  - Loads go on from tile to tile: the next tile's first steps arrive during
//    the last ones of this tile and while its results are stored, and nobody
//    waits for the stores (before, 5.5 us of 1 x 768 steps of 256 x 256 were
//    first loads, 7.5 the stores). Rows of w are put into LDS in such an order
//    that a lane has 8 neighbouring columns: 16-byte stores.
//  - With one tile of rows nobody else reads a tile's w, and tiles of columns
//    may begin at different places of the inner dimension (ring_turn).
//
// us by the kernels that were here before -> now, weights in the caches; the
// former had 256 x 256 by two halves of waves a phase apart, and 128 x 128 with
// one barrier and all loads drained each step (tile now; TFLOP/s):
//   16600 x 2304 x 768    90 -> 60   (224 x 256;  983)
//   16600 x 768 x 768     34 -> 23   (224 x 256;  840)
//   16600 x 3072 x 768   113 -> 74   (224 x 256; 1056)
//   16600 x 768 x 3072    80 -> 62   (224 x 256; 1254)
//   2304 x 3072 x 1024    23 -> 19   (160 x 192;  756)
//   2304 x 4096 x 1024    32 -> 21   (160 x 256;  901)
//   2304 x 1024 x 1024  12.5 -> 10.1 (160 x 64;   477)
//   2304 x 1024 x 4096    34 -> 26   (160 x 64;   749)
//   8192 x 4096 x 4096   225 -> 189  (256 x 256; 1456)
//   8192 x 8192 x 8192   879 -> 696  (256 x 256; 1581)
// Steps of 32 and 3 to 5 buffers of them, reads of LDS early in a half, loads
// closer together gave nothing or cost.
#pragma once
#include "gelu.h"
#include "hybrid/tile.h"
#include <ATen/hip/HIPContext.h>
#include <torch/extension.h>
#include <cmath>

namespace helix {
namespace {

// Of the result. ANY: rows of any number of columns, on any boundary.
enum RingForm { ROWS, GATED, SUMS, ANY };

constexpr int RING_STRIP = 8;                 // tiles of columns, see item_of
constexpr int RING_LDS = 160 * 1024;
constexpr int RING_STEP = 64;                 // of the inner dimension

// Quotients of a fixed number below 2^31, by the method of Granlund and
// Montgomery (Division by invariant integers using multiplication): d <=
// 2^shift, mul the rounded up rest of 2^(32 + shift) / d above 2^32.
struct Divide {
  uint32_t mul, shift;
  Divide() = default;
  explicit Divide(uint32_t d) : shift(0) {
    while ((1ull << shift) < d) ++shift;
    mul = (uint32_t)((((1ull << shift) - d) << 32) / d + 1);
  }
  __device__ __forceinline__ int operator()(uint32_t n) const {
    return (__umulhi(n, mul) + n) >> shift;
  }
};

// x, w, bias on 16-byte boundaries; out as well and N % 8 == 0, sums N % 4 == 0.
// ANY: neither bias nor out has to be, and N is whatever it is.
// GATED: w has N rows of the gate and N of the other factor.
struct Ring {
  const uint16_t *x, *w, *bias;               // bias may be null
  uint16_t* out;
  float* sums;                                // [stretch][M][N]
  int M, N, K, m_tiles, n_tiles, tiles, total, stretch, gelu;
  int ld, up;                  // columns of a row of out; GATED: rows of w from
                               // a gate to its other factor (0: N)
  int group, strip_shift;      // tiles of rows; of group * RING_STRIP tiles
  int unit;                    // ANY: columns that are stored at a time
  int turn;                    // see ring_turn
  Divide by_tiles, by_group;
};

struct RingItem {
  int m0, n0, split, k0, k1;
};

// Where loads are along the inner dimension: from k0 + turn to k1, then from k0.
// After the last item they stay at its start: descriptors are empty by then, and
// what lies past the end of one is checked by a load's own offset, not by this
// scalar one on top of it.
struct RingAt {
  int k, end, ahead, from, wrap;              // from and wrap: what is behind end
  __host__ __device__ __forceinline__ void open(int k0, int k1, int turn) {
    k = k0 + turn;
    end = k1;
    ahead = RING_STEP;
    from = k0;
    wrap = turn;
  }
  __host__ __device__ __forceinline__ void close() {
    k = ahead = 0;
    end = 0x7fffffff;
  }
  // Whether all of the item is ordered.
  __host__ __device__ __forceinline__ bool step() {
    if ((k += ahead) < end) return false;
    if (wrap == 0) return true;
    k = from;
    end = from + wrap;
    wrap = 0;
    return false;
  }
};

// A thread's 16-byte pieces of ROWS_ rows of 64, as offsets in bytes.
template <int N_ROWS>
struct RingUnit {
  int off[N_ROWS / 32];
  template <typename F>
  __device__ __forceinline__ RingUnit(int K, F row) {
#pragma unroll
    for (int i = 0; i < N_ROWS / 32; ++i) {
      const int e = i * 256 + threadIdx.x, r = e / 8;
      off[i] = (int)((row(r) * K + ((e % 8) ^ (r >> 1 & 7)) * 8) * 2);
    }
  }
};

#ifdef __HIP_DEVICE_COMPILE__
// 64 lanes' pieces to 1024 bytes of LDS. What lies past the end of the
// descriptor is zero and not read.
__device__ __forceinline__ void ring_load(const uint16_t* base, int bytes,
                                          int off, int k, uint16_t* lds) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(
      __builtin_amdgcn_make_buffer_rsrc((void*)base, 0, bytes, 0x00020000),
      (__attribute__((address_space(3))) void*)lds, 16, off, k * 2, 0, 0);
}

// Dropped past the end of the descriptor, but issued all the same.
__device__ __forceinline__ void ring_store(void* base, int bytes, int off,
                                           u32x4 v) {
  __builtin_amdgcn_raw_buffer_store_b128(
      v, __builtin_amdgcn_make_buffer_rsrc(base, 0, bytes, 0x00020000), off, 0,
      0);
}

// The same for the first `left` of 8 columns, `unit` at a time: 4 or 2 of them
// have to lie on boundaries of their own size.
__device__ __forceinline__ void ring_store_some(void* base, int bytes, int off,
                                                u32x4 v, int left, int unit) {
  constexpr int NONE = 0x7fffff00;
  const auto to = __builtin_amdgcn_make_buffer_rsrc(base, 0, bytes, 0x00020000);
  if (unit == 4) {
#pragma unroll
    for (int q = 0; q < 2; ++q)
      __builtin_amdgcn_raw_buffer_store_b64(
          u32x2{v[2 * q], v[2 * q + 1]}, to, 4 * q < left ? off + 8 * q : NONE,
          0, 0);
  } else if (unit == 2) {
#pragma unroll
    for (int q = 0; q < 4; ++q)
      __builtin_amdgcn_raw_buffer_store_b32(
          v[q], to, 2 * q < left ? off + 4 * q : NONE, 0, 0);
  } else {
#pragma unroll
    for (int q = 0; q < 8; ++q)
      __builtin_amdgcn_raw_buffer_store_b16(
          (uint16_t)(v[q / 2] >> (q & 1) * 16), to,
          q < left ? off + 2 * q : NONE, 0, 0);
  }
}

// c (+)= a b in place. As a builtin the sums wander from register to register,
// at two moves a product. A product reads its sums four or more products after
// it wrote them.
template <bool FIRST>
__device__ __forceinline__ void ring_mma(floatx4& c, u16x8 a, u16x8 b) {
  if constexpr (FIRST)
    asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, 0"
                 : "=a"(c) : "v"(a), "v"(b));
  else
    asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0"
                 : "+a"(c) : "v"(a), "v"(b));
}

// All but the last VM memory operations and all reads of LDS are through, here
// and in the other waves.
template <int VM>
__device__ __forceinline__ void ring_wait() {
  constexpr int V = VM > 63 ? 63 : VM;        // the counter's range
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt((V & 15) | 7 << 4 | (V >> 4) << 14);
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}
#endif

template <int MI, int NI, RingForm FORM>
__global__ __launch_bounds__(256, 1) void gemm_ring_kernel(Ring m) {
#ifdef __HIP_DEVICE_COMPILE__
  constexpr int BM = 32 * MI, BN = 32 * NI, BK = RING_STEP;
  constexpr int AU = BM * BK, BU = BN * BK;
  // steps of w in LDS, and one more of x: x is ordered in the first half of a
  // step, into what the step before has read, w in the second half, into what
  // this step has read by then; both for NB steps later
  constexpr int NB = (RING_LDS / 2 - AU) / (AU + BU), NA = NB + 1;
  constexpr int OUT_N = FORM == GATED ? BN / 2 : BN;
  // loads ordered since those of the next step, when half of a step is done
  constexpr int ALLOW = (NB - 1) * MI + (NB - 2) * NI;
  constexpr int STORES = MI * NI / (FORM == SUMS ? 1 : FORM == GATED ? 4 : 2);
  static_assert(NB >= 2 && NI % (FORM == GATED ? 4 : 2) == 0, "tile");
  extern __shared__ __attribute__((aligned(16))) uint16_t lds[];
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
  const int lane = threadIdx.x & (WAVE - 1);
  const int lo = lane & 15, hi = lane >> 4, wr = wid / 2, wc = wid % 2;

  // Workgroups of an XCD have neighbouring items of a round, also of the last
  // one, which may not have one for each: 4 x 8 tiles, whose rows and columns
  // its L2 keeps. Four such blocks, or eight, stand above each other in a strip
  // and the others' blocks beside them, so that a round reads little of either
  // matrix (8192 x 28672 x 4096: 1317 us with blocks in one row, 1286 with
  // four of them above each other, 1270 with eight; 8192 x 4096 x 14336: 617,
  // 615 and 629).
  auto item_of = [&](int round, RingItem& p)
      __attribute__((always_inline)) -> bool {
    const int all = gridDim.x, n = min(all, m.total - round * all);
    if ((int)blockIdx.x >= n) return false;
    const int at = round * all + xcd_chunk(blockIdx.x, n);
    p.split = m.by_tiles(at);
    int in = at - p.split * m.tiles;
    const int group = m.by_group(in);
    in -= group * m.group * m.n_tiles;
    const int high = min(m.group, m.m_tiles - group * m.group);
    const int strip = high == m.group ? in >> m.strip_shift
                                      : in / (high * RING_STRIP);
    in -= strip * high * RING_STRIP;
    const int wide = min(RING_STRIP, m.n_tiles - strip * RING_STRIP);
    const int block = wide == RING_STRIP ? in >> 5 : in / (4 * wide);
    in -= block * 4 * wide;
    const int rows = min(4, high - block * 4);
    const int col = rows == 4 ? in >> 2 : in / rows;
    p.m0 = (group * m.group + block * 4 + in - col * rows) * BM;
    p.n0 = (strip * RING_STRIP + col) * OUT_N;
    p.k0 = p.split * m.stretch;
    p.k1 = min(m.K, p.k0 + m.stretch);
    return true;
  };

  const RingUnit<BM> xu(m.K, [](int r) -> int64_t { return r; });
  // row 16 s + 4 a + b of 32 in LDS is column 8 a + 4 s + b, so that two
  // neighbouring products leave 8 columns to a lane
  const RingUnit<BN> wu(m.K, [&](int r) -> int64_t {
    const int n = (r & ~31) | (r & 12) << 1 | (r & 16) >> 2 | (r & 3);
    if constexpr (FORM == GATED) {            // half of a wave's from either
      const int wave = n / (16 * NI), c = n % (16 * NI);
      return wave * 8 * NI + (c < 8 * NI ? c : (int64_t)m.up + c - 8 * NI);
    }
    return n;
  });

  // where loads are, NB steps ahead; empty descriptors after the last item
  const uint16_t *x_at = m.x, *w_at = m.w;
  int x_bytes = 0, w_bytes = 0, load_round = 0;
  RingAt order;
  auto order_from = [&](const RingItem& p, bool on)
      __attribute__((always_inline)) {
    x_bytes = w_bytes = 0;
    order.close();
    if (!on) return;
    x_at = m.x + (int64_t)p.m0 * m.K;
    w_at = m.w + (int64_t)p.n0 * m.K;
    x_bytes = min(BM, m.M - p.m0) * m.K * 2;
    w_bytes = FORM == GATED ? (m.up + m.N - p.n0) * m.K * 2
                            : min(BN, m.N - p.n0) * m.K * 2;
    order.open(p.k0, p.k1,
               (p.n0 / OUT_N & m.turn) * RING_STEP);
  };
  RingItem cur, next;
  if (!item_of(0, cur)) return;
  order_from(cur, true);
  auto advance = [&]() __attribute__((always_inline)) {
    if (!order.step()) return;
    const bool more = item_of(++load_round, next);
    order_from(next, more);
  };

  uint16_t* const xs = lds;
  uint16_t* const ws = lds + NA * AU;
  const int mine = wid * WAVE * 8;
  const int p0 = (hi ^ (lo >> 1 & 7)) * 8, p1 = ((4 + hi) ^ (lo >> 1 & 7)) * 8;
  const uint16_t* const xl = xs + (wr * MI * 16 + lo) * BK;
  const uint16_t* const wl = ws + (wc * NI * 16 + lo) * BK;
  floatx4 acc[NI][MI];
  // products of xa and wa; meanwhile xb and wb are read and a unit is ordered
  auto half = [&](auto first, auto of_w, u16x8 (&xa)[MI], u16x8 (&wa)[NI],
                  u16x8 (&xb)[MI], u16x8 (&wb)[NI], const uint16_t* xr,
                  const uint16_t* wr_, uint16_t* to)
      __attribute__((always_inline)) {
    constexpr bool W = decltype(of_w)::value;
    constexpr int Q = MI * NI, R = MI + NI, L = W ? NI : MI;
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      // to and fro: one operand is that of the product before (1% of large
      // products, by the power it saves)
      const int j = q / MI, i = j & 1 ? MI - 1 - q % MI : q % MI;
      ring_mma<decltype(first)::value>(acc[j][i], wa[j], xa[i]);
#pragma unroll
      for (int r = 0; r < R; ++r)             // in three quarters of the half
        if (r * 3 * Q / (4 * R) == q) {
          if (r < MI) xb[r < MI ? r : 0] = ld_u16x8(xr + r * 16 * BK);
          else wb[r < MI ? 0 : r - MI] = ld_u16x8(wr_ + (r - MI) * 16 * BK);
        }
#pragma unroll
      for (int l = 0; l < L; ++l)
        if (l * Q / L + Q / L / 4 == q) {
          if (W) ring_load(w_at, w_bytes, wu.off[W ? l : 0], order.k,
                           to + l * 2048);
          else ring_load(x_at, x_bytes, xu.off[W ? 0 : l], order.k,
                           to + l * 2048);
        }
      __builtin_amdgcn_sched_barrier(0);
    }
  };
#pragma unroll
  for (int s = 0; s < NB; ++s) {
#pragma unroll
    for (int i = 0; i < MI; ++i)
      ring_load(x_at, x_bytes, xu.off[i], order.k,
                xs + s * AU + mine + i * 2048);
#pragma unroll
    for (int i = 0; i < NI; ++i)
      ring_load(w_at, w_bytes, wu.off[i], order.k,
                ws + s * BU + mine + i * 2048);
    advance();
  }
  ring_wait<(NB - 1) * (MI + NI)>();
  u16x8 xa[MI], wa[NI], xb[MI], wb[NI], bias[NI / 2];
#pragma unroll
  for (int i = 0; i < MI; ++i) xa[i] = ld_u16x8(xl + i * 16 * BK + p0);
#pragma unroll
  for (int j = 0; j < NI; ++j) wa[j] = ld_u16x8(wl + j * 16 * BK + p0);
  // places in LDS: of this step's x and w, and of the x that is ordered
  int sx = 0, sw = 0, so = NB;
  // steps whose operands were ordered before the last tile's stores, for which
  // nobody has to wait then
  int stores_open = 0;
  auto step = [&](auto first) __attribute__((always_inline)) {
    half(first, std::false_type{}, xa, wa, xb, wb, xl + sx * AU + p1,
         wl + sw * BU + p1, xs + so * AU + mine);
    if (stores_open > 0) {
      --stores_open;
      ring_wait<ALLOW + STORES>();
    } else {
      ring_wait<ALLOW>();
    }
    __builtin_amdgcn_sched_barrier(0);
    const int free_w = sw;
    so = sx;
    sx = sx + 1 == NA ? 0 : sx + 1;
    sw = sw + 1 == NB ? 0 : sw + 1;
    if constexpr (decltype(first)::value && FORM == ANY) {
#pragma unroll
      for (int j = 0; j < NI / 2; ++j)
#pragma unroll
        for (int q = 0; q < 8; ++q)
          bias[j][q] = m.bias == nullptr
                           ? 0
                           : m.bias[min(cur.n0 + wc * 16 * NI + j * 32 +
                                        hi * 8 + q, m.N - 1)];
    }
    if constexpr (decltype(first)::value && FORM == ROWS) {
      // more operations in flight than the waits count: they wait for more
#pragma unroll
      for (int j = 0; j < NI / 2; ++j)
        bias[j] = m.bias == nullptr ? u16x8{0, 0, 0, 0, 0, 0, 0, 0}
                                    : ld_u16x8(m.bias + min(
                      cur.n0 + wc * 16 * NI + j * 32 + hi * 8, m.N - 8));
    }
    half(std::false_type{}, std::true_type{}, xb, wb, xa, wa,
         xl + sx * AU + p0, wl + sw * BU + p0, ws + free_w * BU + mine);
    advance();
  };
  for (int round = 1;; ++round) {
    step(std::true_type{});
    for (int n = (cur.k1 - cur.k0) / BK; --n > 0;) step(std::false_type{});
    // the last products reach their registers before these are read
    asm volatile("s_nop 15\n\ts_nop 15");
#pragma unroll
    for (int j = 0; j < NI; ++j)
#pragma unroll
      for (int i = 0; i < MI; ++i) asm volatile("" : "+a"(acc[j][i]));
    // lane: 8 columns from 8 hi of 32, rows lo of 16. All stores are issued,
    // also those that are dropped: stores_open counts on them.
    constexpr int NONE = 0x7fffff00;          // past the end of any tile
    constexpr int SIZE = FORM == SUMS ? 4 : 2;
    const int row = wr * 16 * MI + lo, down = 16 * m.ld * SIZE;
    const int bytes = ((min(BM, m.M - cur.m0) - 1) * m.ld + m.N) * SIZE;
    const int64_t at = ((int64_t)cur.split * m.M + cur.m0) * m.ld;
#pragma unroll
    for (int j = 0; j < NI / (FORM == GATED ? 4 : 2); ++j) {
      const int c = cur.n0 + wc * (OUT_N / 2) + j * 32 + hi * 8;
      const int o = (row * m.ld + c) * SIZE;
#pragma unroll
      for (int i = 0; i < MI; ++i) {
        if constexpr (FORM == SUMS) {
          ring_store(m.sums + at, bytes, c < m.N ? o + i * down : NONE,
                     __builtin_bit_cast(u32x4, acc[2 * j][i]));
          ring_store(m.sums + at, bytes, c + 4 < m.N ? o + i * down + 16 : NONE,
                     __builtin_bit_cast(u32x4, acc[2 * j + 1][i]));
        } else {
          float v[8];
#pragma unroll
          for (int q = 0; q < 8; ++q) {
            v[q] = acc[2 * j + q / 4][i][q % 4];
            if constexpr (FORM == GATED)
              v[q] = silu_f32(v[q]) *
                     acc[NI / 2 + 2 * j + q / 4][i][q % 4];
            else
              v[q] += bf16_to_f32(bias[j][q]);
          }
          if (FORM != GATED && m.gelu)
#pragma unroll
            for (int q = 0; q < 8; ++q) v[q] = gelu_tanh_f32(v[q]);
          const u32x4 packed = __builtin_bit_cast(u32x4, pack8(v));
          if constexpr (FORM == ANY)
            ring_store_some(m.out + at, bytes, o + i * down, packed, m.N - c,
                            m.unit);
          else
            ring_store(m.out + at, bytes, c < m.N ? o + i * down : NONE, packed);
        }
      }
    }
    if (!item_of(round, cur)) break;
    stores_open = NB - 1;
  }
  // LDS goes to another workgroup when no load is on its way to it
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
#endif
}

// What the kernel's offsets of 32 bits reach.
bool ring_fits(const Ring& m, RingForm form) {
  return m.K % 64 == 0 && m.K <= 1 << 21 && m.N <= 1 << 20 &&
         (form == ANY || m.N % (form == SUMS ? 4 : 8) == 0) &&
         (form != GATED || (int64_t)4 * m.N * m.K < INT32_MAX);
}

// Tiles of 32 mi x 32 ni, and us of a step of one with every CU at work.
struct RingTile {
  int mi, ni;
  double step;
};
constexpr RingTile RING_TILES[] = {
    {1, 4, 0.315}, {2, 2, 0.231}, {2, 4, 0.334}, {3, 4, 0.401}, {4, 2, 0.320},
    {4, 4, 0.500}, {4, 8, 0.808}, {5, 2, 0.353}, {5, 4, 0.539}, {5, 6, 0.740},
    {5, 8, 1.010}, {6, 4, 0.616}, {6, 6, 0.891}, {7, 8, 1.216}, {8, 8, 1.300}};

// Whether a kernel of that tile is in a list of pairs.
template <int N>
bool ring_has(const int (&pairs)[N][2], const RingTile& t) {
  for (const auto& p : pairs)
    if (p[0] == t.mi && p[1] == t.ni) return true;
  return false;
}

// us of a product by as many workgroups as there are CUs: rounds of items, and
// what w and sums take to read and write, part of it at the same time. Fitted to
// 11000 times of 318 sizes (17 to 16000 rows, 768 to 28672 columns, 768 to 14336
// deep, 1 to 8 stretches, weights from memory). Against the best tile of each
// size what it picks takes 0.4% longer as rows (at worst 15%), 0.2% gated (4%)
// and, with the reader of the stretches, 1.6% as sums (at worst 35%, 48 x 768 x
// 768). The end of a gated tile with its SiLU as corrected (gelu.h) is 0.055, with
// an exact division 0.064: 47 of 2900 sizes go by other tiles than with 0.035, which
// is what the uncorrected one took, 1.7% faster in the mean (0.90 to 1.15). An item
// takes less while other CUs are idle; few workgroups do not reach the rate of the
// memory.
struct RingCost {
  double busy, fed;
  double least() const { return 3.3 + std::max(busy, fed); }
  double us() const {
    return 3.3 + std::pow(std::pow(busy, 1.8) + std::pow(fed, 1.8), 1 / 1.8);
  }
};
RingCost ring_cost(const Ring& m, RingForm form, const RingTile& t,
                   int stretches, int cus) {
  const int64_t items = (int64_t)cdiv(m.M, 32 * t.mi) *
                        cdiv(m.N, (form == GATED ? 16 : 32) * t.ni) * stretches;
  const double end = form == SUMS ? 0.073 : form == GATED ? 0.055
                     : m.gelu ? 0.11 : 0.038;
  const double item = cdiv(m.K / RING_STEP, stretches) * t.step +
                      end * t.mi * t.ni + 0.27;
  const double rest = (double)(items % cus) / cus;
  RingCost c;
  c.busy = item * ((double)(items / cus) +
                   (rest > 0 ? 0.72 + 0.28 * rest : 0));
  c.fed = (form == GATED ? 4. : 2.) * m.N * m.K / 9e6 /
              std::sqrt(std::min(1., (double)items / cus)) +
          (form == SUMS ? 4. * stretches * m.M * m.N / 4.1e6 : 0.);
  return c;
}

// Tile and stretches, and their time with what it takes to read the stretches:
// their bytes at 4.5 TB/s.
struct RingPlan {
  RingTile tile{};
  int stretches = 1;
  double us = 1e30;
  int weighed = 0;                            // times that were worked out
};

// The tile of a list, and the number of stretches, that take least time, if that
// is below `below`. A host that is behind pays for every call, so a time is only
// worked out where its larger part leaves a chance: 4 of 12 times and 1 of 72 at
// 2304 x 3072 x 1024. All of them took 7 us a product.
template <int N>
RingPlan ring_plan(const Ring& m, RingForm form, const int (&tiles)[N][2],
                   int from, int to, int cus, double below = 1e30) {
  RingPlan best;
  best.us = below;
  for (const RingTile& t : RING_TILES) {
    if (!ring_has(tiles, t)) continue;
    for (int n = from; n <= to; ++n) {
      const double reader = form == SUMS ? 4. * n * m.M * m.N / 4.5e6 : 0.;
      const RingCost c = ring_cost(m, form, t, n, cus);
      if (c.least() + reader >= best.us) continue;
      ++best.weighed;
      const double us = c.us() + reader;
      if (us < best.us) best.tile = t, best.stretches = n, best.us = us;
    }
  }
  return best;
}

// A product in two launches: the first has rounds of large tiles that leave no CU
// idle, the second what is left, in tiles of its own choice; cut behind that many
// rows or columns. Where one launch ends with a round of few tiles that takes
// three quarters of a full one, the second takes less and its start, 3 us. Other
// tiles than the two largest and fewer rounds than all full ones gain nothing more
// by the estimates. us in one launch and cut: 660 of 2 x 14336 x 4096 gated 157 and
// 129, 1537 295 and 268, 5188 848 and 829; 8540 of 4096 x 14336 759 and 700, 5537 of
// 4096 x 4096 154 and 136, 3330 of 6144 x 4096 140 and 128, 12476 of 4096 x 1024 99
// and 95. Over 90 sizes that it takes at a gain of 2% or more, 4.5% in the mean;
// what ring_cut_below asks for leaves out those that lost (8065 of 2304 x 768 31 and
// 34, 4788 of 4096 x 1024 41 and 44).
constexpr double ring_cut_below(double us, double part) {
  return us * (1 - part) - 2.5;
}
struct RingCut {
  bool rows = false;
  int at = 0;
  RingTile first{}, rest{};
  double us = 1e30;
};

template <int N>
RingCut ring_cut(const Ring& m, RingForm form, const int (&tiles)[N][2], int cus,
                 double below) {
  RingCut best;
  best.us = below;
  for (const RingTile& t : RING_TILES) {
    if (t.mi < 7 || t.ni < 8 || !ring_has(tiles, t)) continue;
    const int rows = 32 * t.mi, columns = (form == GATED ? 16 : 32) * t.ni;
    const int64_t down = cdiv(m.M, rows), right = cdiv(m.N, columns);
    const int64_t full = down * right / cus * cus;
    for (const bool by_rows : {true, false}) {
      const int64_t at = by_rows ? full / right * rows : full / down * columns;
      if (at <= 0 || at >= (by_rows ? m.M : m.N)) continue;
      Ring a = m, b = m;
      (by_rows ? a.M : a.N) = (int)at;
      (by_rows ? b.M : b.N) -= (int)at;
      const double us = ring_cost(a, form, t, 1, cus).us();
      if (us >= best.us) continue;
      const RingPlan rest = ring_plan(b, form, tiles, 1, 1, cus, best.us - us);
      if (rest.tile.mi != 0)
        best = RingCut{by_rows, (int)at, t, rest.tile, us + rest.us};
    }
  }
  return best;
}

// The two parts of a product.
void ring_parts(const Ring& m, const RingCut& cut, Ring& a, Ring& b) {
  a = b = m;
  if (cut.rows) {
    a.M = cut.at;
    b.M -= cut.at;
    b.x += (int64_t)cut.at * m.K;
    b.out += (int64_t)cut.at * m.ld;
  } else {
    a.N = cut.at;
    b.N -= cut.at;
    b.w += (int64_t)cut.at * m.K;
    b.out += cut.at;
    if (m.bias != nullptr) b.bias += cut.at;
  }
}

// Mask of a tile of columns' number: at which step of an inner dimension that is
// not cut it begins. Rows of w a multiple of 8 KB apart lie on the same channels, and
// workgroups that start together would all read those; but where several tiles of
// rows share a tile of w, or x does not stay in an XCD's L2, going through it in
// step is worth more. us in step and apart, weights from memory: 24 rows of 2 x
// 14336 x 4096 51.7 and 44.4, 61 51.3 and 45.7, 96 of 28672 x 4096 54 and 44, 128 of
// 128256 x 4096 247 and 189, 61 of 2 x 28672 x 8192 167 and 161; 512 of 2 x 14336 x
// 4096 97 and 111; 37 of 2 x 8192 x 2048 19.1 and 19.8, 64 of 2 x 10240 x 5120 52
// and 54. In stretches 61 of 4096 x 14336 24.9 and 25.7.
int ring_turn(const Ring& m) {
  constexpr int UNIT = 4096;
  return m.m_tiles == 1 && m.K % UNIT == 0 && m.stretch >= m.K
             ? UNIT / RING_STEP - 1 : 0;
}

int ring_cus() {
  int device, cus;
  TORCH_CHECK(hipGetDevice(&device) == hipSuccess &&
              hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount,
                                    device) == hipSuccess && cus > 0);
  return cus;
}

bool ring_allow(const void* kernel) {
  TORCH_CHECK(hipFuncSetAttribute(
                  kernel, hipFuncAttributeMaxDynamicSharedMemorySize,
                  RING_LDS) == hipSuccess, "LDS size refused");
  return true;
}

template <int MI, int NI, RingForm FORM>
void ring_run(Ring m, int stretches, int cus) {
  const void* kernel = (const void*)gemm_ring_kernel<MI, NI, FORM>;
  static const bool once = ring_allow(kernel);
  (void)once;
  if (m.ld == 0) m.ld = m.N;
  if (m.up == 0) m.up = m.N;
  m.m_tiles = cdiv(m.M, 32 * MI);
  m.n_tiles = cdiv(m.N, (FORM == GATED ? 16 : 32) * NI);
  const int64_t total = (int64_t)m.m_tiles * m.n_tiles * stretches;
  TORCH_CHECK(total < 1 << 30, "a product of too many tiles");
  m.tiles = m.m_tiles * m.n_tiles;
  m.total = (int)total;
  m.by_tiles = Divide(m.tiles);
  m.turn = ring_turn(m);
  // eight blocks of 4 tiles of rows where w is too large for the memory-side
  // cache beside the rest
  m.group = (int64_t)m.N * (FORM == GATED ? 2 : 1) * m.K >= 64 << 20 ? 32 : 16;
  m.strip_shift = m.group == 32 ? 8 : 7;
  m.by_group = Divide(m.group * m.n_tiles);
  void* args[] = {&m};
  const hipError_t err = hipLaunchKernel(
      kernel, dim3(std::min(cus, m.total)), dim3(256), args, RING_LDS,
      at::hip::getCurrentHIPStream());
  TORCH_CHECK(err == hipSuccess, hipGetErrorString(err));
}

}  // namespace
}  // namespace helix
