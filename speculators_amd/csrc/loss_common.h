// Row streaming helpers shared by the vocabulary-loss kernels (gfx950): 8-element chunk
// loads / stores of bf16 or fp32 rows with 16-byte non-temporal accesses.
#pragma once

#include <type_traits>

#include "spx_common.h"
#include "../../include/spx.h"

namespace spx {

constexpr int kLossThreads = 256;
constexpr int kLossWaves = kLossThreads / 64;

// ---- 8-element chunk loads -------------------------------------------------
// VEC: the row base is 16-byte aligned and the chunk is complete.
template <typename T>
__device__ __forceinline__ void load8_vec(const T* p, float v[8]);

// streaming accesses bypass the cache hierarchy's allocate-on-access policy: every row is
// read (and every gradient row written) exactly once per launch
#define SPX_LOSS_NT 1
__device__ __forceinline__ u32x4 ld16(const void* p) {
#if SPX_LOSS_NT
  return __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(p));
#else
  return *reinterpret_cast<const u32x4*>(p);
#endif
}
__device__ __forceinline__ void st16(void* p, u32x4 v) {
#if SPX_LOSS_NT
  __builtin_nontemporal_store(v, reinterpret_cast<u32x4*>(p));
#else
  *reinterpret_cast<u32x4*>(p) = v;
#endif
}
template <>
__device__ __forceinline__ void load8_vec<uint16_t>(const uint16_t* p, float v[8]) {
  u32x4 raw = ld16(p);
  v[0] = bf16_lo(raw.x); v[1] = bf16_hi(raw.x);
  v[2] = bf16_lo(raw.y); v[3] = bf16_hi(raw.y);
  v[4] = bf16_lo(raw.z); v[5] = bf16_hi(raw.z);
  v[6] = bf16_lo(raw.w); v[7] = bf16_hi(raw.w);
}
template <>
__device__ __forceinline__ void load8_vec<float>(const float* p, float v[8]) {
  f32x4 a = *reinterpret_cast<const f32x4*>(p);
  f32x4 b = *reinterpret_cast<const f32x4*>(p + 4);
  v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
  v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
}

__device__ __forceinline__ float load1(const uint16_t* p) { return bf16_bits_to_f32(*p); }
__device__ __forceinline__ float load1(const float* p) { return *p; }

template <typename T>
__device__ __forceinline__ void load8_guard(const T* p, int64_t base, int64_t n, float v[8]) {
#pragma unroll
  for (int i = 0; i < 8; ++i) v[i] = (base + i < n) ? load1(p + base + i) : kNegBig;
}

template <typename T, bool VEC>
__device__ __forceinline__ void load8(const T* row, int64_t base, int64_t n, float v[8]) {
  if (VEC && base + 8 <= n) load8_vec<T>(row + base, v);
  else load8_guard<T>(row, base, n, v);
}

template <typename T>
__device__ __forceinline__ void store8_vec(T* p, const float v[8]);
template <>
__device__ __forceinline__ void store8_vec<uint16_t>(uint16_t* p, const float v[8]) {
  u32x4 raw;
  raw.x = pack_bf16x2(v[0], v[1]); raw.y = pack_bf16x2(v[2], v[3]);
  raw.z = pack_bf16x2(v[4], v[5]); raw.w = pack_bf16x2(v[6], v[7]);
  st16(p, raw);
}
template <>
__device__ __forceinline__ void store8_vec<float>(float* p, const float v[8]) {
  f32x4 a = {v[0], v[1], v[2], v[3]}, b = {v[4], v[5], v[6], v[7]};
  *reinterpret_cast<f32x4*>(p) = a;
  *reinterpret_cast<f32x4*>(p + 4) = b;
}
__device__ __forceinline__ void store1(uint16_t* p, float v) { *p = (uint16_t)f32_to_bf16_bits(v); }
__device__ __forceinline__ void store1(float* p, float v) { *p = v; }

template <typename T, bool VEC>
__device__ __forceinline__ void store8(T* row, int64_t base, int64_t n, const float v[8]) {
  if (VEC && base + 8 <= n) store8_vec<T>(row + base, v);
  else {
#pragma unroll
    for (int i = 0; i < 8; ++i)
      if (base + i < n) store1(row + base + i, v[i]);
  }
}

__host__ __device__ __forceinline__ bool ptr_aligned16(const void* p) {
  return (reinterpret_cast<uintptr_t>(p) & 15) == 0;
}

// ---- reductions over a wave ----
// op over the 64 lanes, every lane gets the result: moves inside the sixteen lanes of a row, then swaps of rows, where a
// shuffle would be a trip through LDS (six of them a value: kl, 4096 rows x 7 steps 748 -> 719 us)
template <typename T, typename Op>
__device__ __forceinline__ T wave_all(T v, Op op) {
  static_assert(sizeof(T) == 4, "one register");
  auto moved = [](T x, auto ctrl) __attribute__((always_inline)) {
    const int i = __builtin_bit_cast(int, x);
    return __builtin_bit_cast(T, __builtin_amdgcn_update_dpp(i, i, decltype(ctrl)::value, 0xf, 0xf, true));
  };
  v = op(v, moved(v, std::integral_constant<int, 0xb1>{}));   // quad_perm 1 0 3 2
  v = op(v, moved(v, std::integral_constant<int, 0x4e>{}));   // quad_perm 2 3 0 1
  v = op(v, moved(v, std::integral_constant<int, 0x141>{}));  // row_half_mirror
  v = op(v, moved(v, std::integral_constant<int, 0x140>{}));  // row_mirror
  uint32_t u = __builtin_bit_cast(uint32_t, v);
  const auto rows = __builtin_amdgcn_permlane16_swap(u, u, false, false);
  v = op(__builtin_bit_cast(T, (uint32_t)rows[0]), __builtin_bit_cast(T, (uint32_t)rows[1]));
  u = __builtin_bit_cast(uint32_t, v);
  const auto halves = __builtin_amdgcn_permlane32_swap(u, u, false, false);
  return op(__builtin_bit_cast(T, (uint32_t)halves[0]), __builtin_bit_cast(T, (uint32_t)halves[1]));
}

// ---- mask element access ---------------------------------------------------
__device__ __forceinline__ float mask_value(const void* p, int kind, int64_t i) {
  switch (kind) {
    case SPX_KIND_U8: return (float)reinterpret_cast<const uint8_t*>(p)[i];
    case SPX_KIND_I32: return (float)reinterpret_cast<const int32_t*>(p)[i];
    case SPX_KIND_I64: return (float)reinterpret_cast<const int64_t*>(p)[i];
    case SPX_KIND_F32: return reinterpret_cast<const float*>(p)[i];
    default: return bf16_bits_to_f32(reinterpret_cast<const uint16_t*>(p)[i]);
  }
}

// row_map[r] = number of live rows before r if live(r), else -1; *count = number of live rows; row_of (may be null) = the live
// rows.  One workgroup of 1024 threads, rows in order.
template <typename Live>
__device__ __forceinline__ void pack_row_map(Live live_at, int rows, int32_t* __restrict__ row_map,
                                             int32_t* __restrict__ count, int32_t* __restrict__ row_of = nullptr) {
  __shared__ int wave_tot[16];
  __shared__ int base_s;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  if (tid == 0) base_s = 0;
  __syncthreads();
  for (int r0 = 0; r0 < rows; r0 += 1024) {
    const int r = r0 + tid;
    const bool live = r < rows && live_at(r);
    const unsigned long long m = __ballot(live);
    const int before = __popcll(m & ((1ull << lane) - 1ull));
    if (lane == 0) wave_tot[wave] = __popcll(m);
    __syncthreads();
    int off = base_s;
    for (int w = 0; w < wave; ++w) off += wave_tot[w];
    if (r < rows) row_map[r] = live ? off + before : -1;
    if (live && row_of) row_of[off + before] = r;
    __syncthreads();
    if (tid == 0) {
      int t = 0;
      for (int w = 0; w < 16; ++w) t += wave_tot[w];
      base_s += t;
    }
    __syncthreads();
  }
  if (tid == 0) *count = base_s;
}

}  // namespace spx
