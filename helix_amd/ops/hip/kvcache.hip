// Paged KV cache: scatter this step's K/V rows into their cache slots, gather
// a context's rows from them.
//
// Cache layout (chosen for the decode kernel's per-token contiguous reads):
//   k_cache, v_cache: [num_blocks, Hkv, block_size, D] bf16
// slot_mapping[t] = block_idx * block_size + offset   (int64, -1 = skip)
#include "common.h"
#include <torch/extension.h>
#include <ATen/hip/HIPContext.h>

using namespace helix;

namespace {

// 8 e4m3 bytes, lowest first (exact)
__device__ __forceinline__ u16x8 bf16_of_e4m3(uint64_t x) {
  const unsigned a = (unsigned)x, b = (unsigned)(x >> 32);
  const auto p = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(a, 1.f, false);
  const auto q = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(a, 1.f, true);
  const auto r = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(b, 1.f, false);
  const auto s = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(b, 1.f, true);
  return __builtin_bit_cast(
      u16x8, u32x4{__builtin_bit_cast(unsigned, p),
                   __builtin_bit_cast(unsigned, q),
                   __builtin_bit_cast(unsigned, r),
                   __builtin_bit_cast(unsigned, s)});
}

// EB = element bytes (2 = bf16 cache, 1 = fp8/e4m3 cache: inputs are
// already-quantized byte views with identical [T, Hkv, D] geometry).
template <int EB>
__global__ void reshape_and_cache_kernel(
    const uint8_t* __restrict__ k, const uint8_t* __restrict__ v,
    uint8_t* __restrict__ k_cache, uint8_t* __restrict__ v_cache,
    const int64_t* __restrict__ slot_mapping, int Hkv, int D, int block_size) {
  const int t = blockIdx.x;
  const int64_t slot = slot_mapping[t];
  if (slot < 0) return;
  const int64_t block = slot / block_size;
  const int off = slot % block_size;
  const int row_bytes = Hkv * D * EB;
  const int nvec = row_bytes / 16;

  for (int idx = threadIdx.x; idx < nvec; idx += blockDim.x) {
    const int b16 = idx * 16;               // byte offset within the row
    const int h = b16 / (D * EB);
    const int d = b16 % (D * EB);
    const int64_t src = (int64_t)t * row_bytes + b16;
    const int64_t dst =
        (((block * Hkv + h) * (int64_t)block_size + off) * D) * EB + d;
    *reinterpret_cast<u8x16*>(k_cache + dst) =
        *reinterpret_cast<const u8x16*>(k + src);
    *reinterpret_cast<u8x16*>(v_cache + dst) =
        *reinterpret_cast<const u8x16*>(v + src);
  }
}

constexpr int GATHER = 256;    // threads of a gathering workgroup

// Row t of the results is the row at offset off[t] of page blk[t], of every
// head; e4m3 bytes become bf16. Bound by memory: keys and values in one launch,
// 8 elements a lane, neighbouring lanes on neighbouring addresses on both
// sides, a row's place looked up once for both. us by torch's indexing (and
// conversion) -> here, 8 heads of 128: 6501 rows 54.6 -> 10.1 (5.2 TB/s), of
// e4m3 82.6 -> 8.0; 30000 rows 221 -> 40.5 (6.1 TB/s), of e4m3 329 -> 29.2;
// 600 rows 11.2 -> 3.1. Places outside the cache give zeros.
template <bool F8>
__global__ __launch_bounds__(GATHER) void gather_kernel(
    uint16_t* __restrict__ k, uint16_t* __restrict__ v,
    const uint8_t* __restrict__ k_cache, const uint8_t* __restrict__ v_cache,
    const int64_t* __restrict__ blk, const int64_t* __restrict__ off, int T,
    int Hkv, int D, int64_t blocks, int block_size, int rows) {
  constexpr int EB = F8 ? 1 : 2;
  const int per_head = D / 8, per_row = Hkv * per_head;
  const int t0 = blockIdx.x * rows;
  for (int e = threadIdx.x; e < rows * per_row; e += GATHER) {
    const int t = t0 + e / per_row, at = e % per_row;
    if (t >= T) return;
    const int64_t page = blk[t], place = off[t];
    const bool in = page >= 0 && page < blocks && place >= 0 &&
                    place < block_size;
    const int64_t from =
        (((page * Hkv + at / per_head) * block_size + place) * D +
         at % per_head * 8) * EB;
    u16x8 a{}, b{};
    if (in) {
      if (F8) {
        a = bf16_of_e4m3(*reinterpret_cast<const uint64_t*>(k_cache + from));
        b = bf16_of_e4m3(*reinterpret_cast<const uint64_t*>(v_cache + from));
      } else {
        a = *reinterpret_cast<const u16x8*>(k_cache + from);
        b = *reinterpret_cast<const u16x8*>(v_cache + from);
      }
    }
    const int64_t to = ((int64_t)t * per_row + at) * 8;
    *reinterpret_cast<u16x8*>(k + to) = a;
    *reinterpret_cast<u16x8*>(v + to) = b;
  }
}

}  // namespace

void reshape_and_cache(torch::Tensor k, torch::Tensor v,
                       torch::Tensor k_cache, torch::Tensor v_cache,
                       torch::Tensor slot_mapping) {
  const int T = slot_mapping.size(0);
  const int Hkv = k_cache.size(1);
  const int block_size = k_cache.size(2);
  const int D = k_cache.size(3);
  TORCH_CHECK(D % 16 == 0);
  TORCH_CHECK(slot_mapping.scalar_type() == torch::kInt64);
  const bool kv8 = k_cache.scalar_type() == torch::kUInt8;
  TORCH_CHECK(!kv8 || k.scalar_type() == torch::kUInt8,
              "fp8 cache takes pre-quantized uint8 K/V views");
  auto stream = at::hip::getCurrentHIPStream();
  const int eb = kv8 ? 1 : 2;
  const int threads = std::min(256, Hkv * D * eb / 16);
  if (kv8) {
    hipLaunchKernelGGL(reshape_and_cache_kernel<1>, dim3(T), dim3(threads),
                       0, stream, (const uint8_t*)k.data_ptr(),
                       (const uint8_t*)v.data_ptr(),
                       (uint8_t*)k_cache.data_ptr(),
                       (uint8_t*)v_cache.data_ptr(),
                       slot_mapping.data_ptr<int64_t>(), Hkv, D, block_size);
  } else {
    hipLaunchKernelGGL(reshape_and_cache_kernel<2>, dim3(T), dim3(threads),
                       0, stream, (const uint8_t*)k.data_ptr(),
                       (const uint8_t*)v.data_ptr(),
                       (uint8_t*)k_cache.data_ptr(),
                       (uint8_t*)v_cache.data_ptr(),
                       slot_mapping.data_ptr<int64_t>(), Hkv, D, block_size);
  }
}

void gather_kv(torch::Tensor k, torch::Tensor v, torch::Tensor k_cache,
               torch::Tensor v_cache, torch::Tensor blk, torch::Tensor off) {
  const int64_t T = blk.numel();
  const int Hkv = k_cache.size(1), block_size = k_cache.size(2);
  const int D = k_cache.size(3);
  const bool f8 = k_cache.scalar_type() == torch::kUInt8;
  TORCH_CHECK(D % 8 == 0 && T < (1LL << 31) - GATHER);
  TORCH_CHECK(f8 || k_cache.scalar_type() == torch::kBFloat16);
  TORCH_CHECK(k_cache.is_contiguous() && v_cache.is_contiguous() &&
              v_cache.sizes() == k_cache.sizes() &&
              v_cache.scalar_type() == k_cache.scalar_type());
  TORCH_CHECK(blk.scalar_type() == torch::kInt64 && blk.is_contiguous() &&
              off.scalar_type() == torch::kInt64 && off.is_contiguous() &&
              off.numel() == T);
  for (const auto& t : {k, v, k_cache, v_cache, blk, off})
    TORCH_CHECK(t.is_cuda() && t.device() == k.device(),
                "everything on one GPU");
  TORCH_CHECK(k.is_contiguous() && v.is_contiguous() &&
              k.scalar_type() == torch::kBFloat16 &&
              v.scalar_type() == torch::kBFloat16 &&
              k.numel() == T * Hkv * D && v.numel() == k.numel());
  if (k.numel() == 0) return;
  // a workgroup has whole rows, 2 pieces a lane at 8 x 128
  const int rows = std::max(1, 2 * GATHER * 8 / (Hkv * D));
  const dim3 grid((T + rows - 1) / rows);
  auto stream = at::hip::getCurrentHIPStream();
#define GATHER_ROWS(F8)                                                      \
  hipLaunchKernelGGL(gather_kernel<F8>, grid, dim3(GATHER), 0, stream,       \
                     (uint16_t*)k.data_ptr(), (uint16_t*)v.data_ptr(),       \
                     (const uint8_t*)k_cache.data_ptr(),                     \
                     (const uint8_t*)v_cache.data_ptr(),                     \
                     blk.data_ptr<int64_t>(), off.data_ptr<int64_t>(),       \
                     (int)T, Hkv, D, k_cache.size(0), block_size, rows)
  if (f8) GATHER_ROWS(true); else GATHER_ROWS(false);
#undef GATHER_ROWS
}
