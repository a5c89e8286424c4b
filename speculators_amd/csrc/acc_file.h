// 64 accumulators of v_mfma_f32_16x16x32_bf16 that live in the accumulation registers a0 .. a255 by name, accumulator I in
// a[4 I .. 4 I + 3], out of the compiler's sight.  For a kernel that reads its accumulators while other operands are live: the
// compiler brings accumulators that it knows into vector registers all at once, wherever the first of them is read, and spills
// what does not fit (400 bytes a lane in the kernel this was made for).
// Such a kernel uses `claim()` once, which counts the registers as used, and must leave the compiler no reason to use them itself:
// tests/test_kernel_isa.py checks on the compiled code that nothing else does.  Products and reads are volatile statements and
// stay in the order of the source; behind the last product of an accumulator come `wait()` or 16 other products before its read.
//
// With -DSPX_MFMA_BUILTIN=1 (the cross-check build, see mfma16) the accumulators are ordinary values.
#pragma once

#include <type_traits>
#include <utility>

#include "spx_common.h"

namespace spx {

// f(0), f(1), .. f(N - 1) with constants
template <int... I, typename F>
__device__ __forceinline__ void each_of(std::integer_sequence<int, I...>, F&& f) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <int N, typename F>
__device__ __forceinline__ void each(F&& f) {
  each_of(std::make_integer_sequence<int, N>{}, f);
}

struct AccFile {
#if SPX_MFMA_BUILTIN
  f32x4 v[64];
  __device__ __forceinline__ void claim() {}
  __device__ __forceinline__ void wait() {}
  // (FRESH: the first product of an accumulator)
  template <int I, bool FRESH>
  __device__ __forceinline__ void product(bf16x8 a, bf16x8 b) {
    v[I] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, FRESH ? f32x4{0.f, 0.f, 0.f, 0.f} : v[I], 0, 0, 0);
  }
  template <int I>
  __device__ __forceinline__ f32x4 read() { return v[I]; }
#else
  __device__ __forceinline__ void claim() { asm volatile("" ::: "a0", "a255"); }
  __device__ __forceinline__ void wait() { asm volatile("s_nop 15\n\ts_nop 15" ::: "memory"); }
  template <int I, bool FRESH>
  __device__ __forceinline__ void product(bf16x8 a, bf16x8 b) {
    if constexpr (FRESH)
      asm volatile("v_mfma_f32_16x16x32_bf16 a[%0:%1], %2, %3, 0" ::"n"(4 * I), "n"(4 * I + 3), "v"(a), "v"(b));
    else
      asm volatile("v_mfma_f32_16x16x32_bf16 a[%0:%1], %2, %3, a[%0:%1]" ::"n"(4 * I), "n"(4 * I + 3), "v"(a), "v"(b));
  }
  template <int I>
  __device__ __forceinline__ f32x4 read() {
    f32x4 r;
    float x, y, z, w;
    asm volatile("v_accvgpr_read_b32 %0, a[%4]\n\tv_accvgpr_read_b32 %1, a[%5]\n\tv_accvgpr_read_b32 %2, a[%6]\n\t"
                 "v_accvgpr_read_b32 %3, a[%7]"
                 : "=v"(x), "=v"(y), "=v"(z), "=v"(w)
                 : "n"(4 * I), "n"(4 * I + 1), "n"(4 * I + 2), "n"(4 * I + 3));
    r[0] = x; r[1] = y; r[2] = z; r[3] = w;
    return r;
  }
#endif
};

}  // namespace spx
