// Cross-entropy of full-vocabulary logits against integer labels with an
// ignore index (the multi-token-prediction loss), for gfx950.  One workgroup
// streams one logits row once with 16-byte non-temporal loads and keeps the
// online soft-max statistics in registers: loss = logsumexp(x) - x[label].
// Ignored rows are not read at all.  HBM-bound: algorithmic traffic is one row
// read (forward), one row read + one row written (backward).
//
// Exponentials run in the base-2 domain (v_exp_f32 is 2^x).

#include "loss_common.h"
#include "../../include/spx.h"

namespace spx {

struct CeStats {
  float m, z;       // running max of x * log2(e), sum of 2^(x' - m)
  float best; int idx;  // arg-max value (unscaled) / first index
};

__device__ __forceinline__ void ce_merge(CeStats& a, float bm, float bz, float bb, int bi) {
  const float m = fmaxf(a.m, bm);
  a.z = a.z * fast_exp2(a.m - m) + bz * fast_exp2(bm - m);
  a.m = m;
  if (bb > a.best || (bb == a.best && bi < a.idx)) { a.best = bb; a.idx = bi; }
}

// Chunks a thread requests before it uses the first.  Rows of 151936, 70 % live: 32760 forward 1050 -> 1016 us, gradient of the packed
// rows 2740 -> 2728; 1997 85 -> 77 and 192 -> 178; 510 54 -> 24 and 73 -> 49.
constexpr int kCeAhead = 4;

template <typename T, bool VEC, bool ARGMAX>
__global__ __launch_bounds__(kLossThreads) void label_ce_fwd_kernel(
    const T* __restrict__ logits, int64_t ld, const int64_t* __restrict__ labels, int64_t vocab,
    int64_t ignore_index, float* __restrict__ loss, float* __restrict__ lse_out,
    int32_t* __restrict__ argmax_out) {
  __shared__ float sm[kLossWaves], sz[kLossWaves], sb[kLossWaves];
  __shared__ int si[kLossWaves];
  const int64_t r = blockIdx.x;
  const int64_t label = labels[r];
  const bool ignored = label == ignore_index;
  if (ignored && !ARGMAX) {  // uniform over the workgroup
    if (threadIdx.x == 0) { loss[r] = 0.f; lse_out[r] = 0.f; }
    return;
  }
  const T* row = logits + r * ld;
  const int tid = threadIdx.x;
  const int64_t nchunks = (vocab + 7) >> 3;

  CeStats s;
  s.m = kNegBig; s.z = 0.f; s.best = -INFINITY; s.idx = 0x7fffffff;
  auto take = [&](int64_t base, const float (&x)[8]) __attribute__((always_inline)) {
    float cm = x[0];
#pragma unroll
    for (int i = 1; i < 8; ++i) cm = fmaxf(cm, x[i]);
    if (ARGMAX && cm > s.best) {
      // first index inside the chunk that attains the chunk maximum
      int k = 7;
#pragma unroll
      for (int i = 6; i >= 0; --i) k = (x[i] == cm) ? i : k;
      s.best = cm; s.idx = (int)base + k;
    }
    const float cm2 = cm * kLog2e;
    if (cm2 > s.m) {  // the running maximum moved: rescale the sum
      s.z *= fast_exp2(s.m - cm2);
      s.m = cm2;
    }
    float zz = 0.f;
#pragma unroll
    for (int i = 0; i < 8; ++i) zz += fast_exp2(fmaf(x[i], kLog2e, -s.m));
    s.z += zz;
  };
  int64_t c = tid;
  if constexpr (VEC && !ARGMAX) {  // (with the arg-max the compares bound it)
    for (; c + (kCeAhead - 1) * kLossThreads < (vocab >> 3); c += kCeAhead * kLossThreads) {
      float x[kCeAhead][8];
#pragma unroll
      for (int u = 0; u < kCeAhead; ++u) load8_vec<T>(row + ((c + u * kLossThreads) << 3), x[u]);
#pragma unroll
      for (int u = 0; u < kCeAhead; ++u) take((c + u * kLossThreads) << 3, x[u]);
    }
  }
  for (; c < nchunks; c += kLossThreads) {
    float x[8];
    load8<T, VEC>(row, c << 3, vocab, x);
    take(c << 3, x);
  }
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1)
    ce_merge(s, __shfl_xor(s.m, m, 64), __shfl_xor(s.z, m, 64), __shfl_xor(s.best, m, 64),
             __shfl_xor(s.idx, m, 64));
  if ((tid & 63) == 0) { sm[tid >> 6] = s.m; sz[tid >> 6] = s.z; sb[tid >> 6] = s.best; si[tid >> 6] = s.idx; }
  __syncthreads();
  if (tid == 0) {
#pragma unroll
    for (int w = 1; w < kLossWaves; ++w) ce_merge(s, sm[w], sz[w], sb[w], si[w]);
    const float lse = (s.m + fast_log2(s.z)) * kLn2;
    float l = 0.f;
    if (!ignored) {
      // a label outside [0, vocab) that is not the ignore index has no defined loss
      l = (label >= 0 && label < vocab) ? lse - load1(row + label) : __builtin_nanf("");
    }
    loss[r] = l;
    lse_out[r] = lse;
    if (ARGMAX) argmax_out[r] = s.idx < vocab ? s.idx : 0;  // (no value above -infinity: 0, as torch has it)
  }
}

// dlogits[r, j] = g[r] * (softmax(x[r])[j] - [j == label[r]]); rows with g == 0 or an ignored
// label are written as zeros without reading the logits.  With a row map the gradient of row r
// goes to row row_map[r] of the output and rows mapped to -1 are not written at all (the live
// rows packed to the front: the product that consumes them skips the dead ones).
template <typename T, bool VEC>
__global__ __launch_bounds__(kLossThreads) void label_ce_bwd_kernel(
    const T* __restrict__ logits, int64_t ld, const int64_t* __restrict__ labels,
    const float* __restrict__ lse, const float* __restrict__ grad_rows, int64_t vocab,
    int64_t ignore_index, T* __restrict__ dlogits, int64_t ld_out, const int32_t* __restrict__ row_map) {
  const int64_t r = blockIdx.x;
  const int64_t label = labels[r];
  const float g = grad_rows[r];
  const T* row = logits + r * ld;
  int64_t dst = r;
  if (row_map) {
    dst = row_map[r];
    if (dst < 0) return;
  }
  T* out = dlogits + dst * ld_out;
  const int tid = threadIdx.x;
  const int64_t nchunks = (vocab + 7) >> 3;
  if (g == 0.f || label == ignore_index) {
    const float z[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    for (int64_t c = tid; c < nchunks; c += kLossThreads) store8<T, VEC>(out, c << 3, vocab, z);
    return;
  }
  const float l2 = lse[r] * kLog2e;
  auto grad = [&](int64_t base, const float (&x)[8], float (&d)[8]) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float p = fast_exp2(fmaf(x[i], kLog2e, -l2));
      d[i] = g * (p - ((base + i == label) ? 1.f : 0.f));
    }
  };
  int64_t c = tid;
  if constexpr (VEC) {
    for (; c + (kCeAhead - 1) * kLossThreads < (vocab >> 3); c += kCeAhead * kLossThreads) {
      float x[kCeAhead][8], d[8];
#pragma unroll
      for (int u = 0; u < kCeAhead; ++u) load8_vec<T>(row + ((c + u * kLossThreads) << 3), x[u]);
#pragma unroll
      for (int u = 0; u < kCeAhead; ++u) {
        const int64_t base = (c + u * kLossThreads) << 3;
        grad(base, x[u], d);
        store8_vec<T>(out + base, d);
      }
    }
  }
  for (; c < nchunks; c += kLossThreads) {
    float x[8], d[8];
    load8<T, VEC>(row, c << 3, vocab, x);
    grad(c << 3, x, d);
    store8<T, VEC>(out, c << 3, vocab, d);
  }
}

// loss[r] = lse[r] - x[r, label[r]] for rows whose log-sum-exp is already known (the statistics
// epilogue of the head product, spx_gemm_bf16_nt_stats): one element of the row is read instead of
// the row.  Ignored rows: loss 0; a label outside [0, vocab) that is not the ignore index: NaN,
// as in label_ce_fwd_kernel.
template <typename T>
__global__ __launch_bounds__(256) void label_ce_pick_kernel(const T* __restrict__ logits, int64_t ld,
                                                            const int64_t* __restrict__ labels, int64_t rows,
                                                            int64_t vocab, int64_t ignore_index,
                                                            const float* __restrict__ lse,
                                                            float* __restrict__ loss) {
  const int64_t r = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (r >= rows) return;
  const int64_t label = labels[r];
  float l = 0.f;
  if (label != ignore_index)
    l = (label >= 0 && label < vocab) ? lse[r] - load1(logits + r * ld + label) : __builtin_nanf("");
  loss[r] = l;
}

// ---- forward and logits gradient in one read -------------------------------------------------------
// Rows that carry a gradient are known before the loss is (labels), and the gradient but for the weight of its row: one
// workgroup of 1024 threads holds a whole row of up to 155648 columns in registers (19 chunks of 16 bytes a thread), reduces
// it, and goes over the registers a second time for softmax(x) - onehot(label), the gradient of a row of weight ONE, packed to
// the front; the input-gradient product, which is linear in it, applies the weights (spx_gemm_bf16_rows_graded).  A
// workgroup walks its rows, and behind every stored chunk it requests that chunk of its next row: loads and stores of two
// rows are under way while one is reduced.  22930 live of 32760 rows of 151936, us: a forward and a backward pass (two
// reads and a write) 3773, so 2725 (5.15 TB/s); 1400 of 1997 267 / 176, 350 of 510 78 / 53; 1400 of 2000 rows of 65536 112 / 78.
constexpr int kOneThreads = 1024, kOneWaves = kOneThreads / 64, kOneChunks = 19;

// row_map and row_of (the live rows in their order), and a loss of zero for the others
__global__ __launch_bounds__(1024) void label_rows_kernel(const int64_t* __restrict__ labels, int64_t ignore_index, int rows,
                                                          int32_t* __restrict__ row_map, int32_t* __restrict__ count,
                                                          int32_t* __restrict__ row_of, float* __restrict__ loss) {
  pack_row_map([&](int r) {
    const bool live = labels[r] != ignore_index;
    if (!live) loss[r] = 0.f;
    return live;
  }, rows, row_map, count, row_of);
}

__global__ __launch_bounds__(kOneThreads) __attribute__((amdgpu_waves_per_eu(4, 4))) void label_ce_fwd_grad_kernel(
    const uint16_t* __restrict__ logits, int64_t ld, const int64_t* __restrict__ labels, int vocab,
    const int32_t* __restrict__ row_of, const int32_t* __restrict__ count, float* __restrict__ loss,
    uint16_t* __restrict__ grad, int64_t ld_grad) {
  __shared__ float sm[2][kOneWaves], sz[2][kOneWaves];
  const int n = *count, tid = threadIdx.x, nchunks = vocab >> 3;
  int slot = blockIdx.x;
  if (slot >= n) return;
  int r = row_of[slot];
  const uint16_t* row = logits + (int64_t)r * ld;
  u32x4 xr[kOneChunks];
#pragma unroll
  for (int j = 0; j < kOneChunks; ++j) {
    const int c = tid + j * kOneThreads;
    if (c < nchunks) xr[j] = ld16(row + ((int64_t)c << 3));
  }
  auto unpack = [](u32x4 raw, float (&v)[8]) __attribute__((always_inline)) {
    v[0] = bf16_lo(raw.x); v[1] = bf16_hi(raw.x); v[2] = bf16_lo(raw.y); v[3] = bf16_hi(raw.y);
    v[4] = bf16_lo(raw.z); v[5] = bf16_hi(raw.z); v[6] = bf16_lo(raw.w); v[7] = bf16_hi(raw.w);
  };
  for (int turn = 0;; turn ^= 1) {
    const int64_t label = labels[r];
    const bool inside = label >= 0 && label < vocab;
    const float xt = tid == 0 && inside ? load1(row + label) : __builtin_nanf("");
    const int next = slot + (int)gridDim.x;
    const bool more = next < n;
    const int nr = more ? row_of[next] : 0;
    // (places of chunks worked out where they are needed: kept over the rows they would be spilled, and a reload waits for
    // every load in front of it)
    int lane0 = tid;
    asm volatile("" : "+v"(lane0));
    float m = kNegBig, z = 0.f;
#pragma unroll
    for (int j = 0; j < kOneChunks; ++j) {
      if (lane0 + j * kOneThreads >= nchunks) continue;
      float x[8];
      unpack(xr[j], x);
      float cx = x[0];
#pragma unroll
      for (int i = 1; i < 8; ++i) cx = fmaxf(cx, x[i]);
      const float cs = cx * kLog2e;
      if (cs > m) {  // the running maximum moved: rescale the sum
        z *= fast_exp2(m - cs);
        m = cs;
      }
#pragma unroll
      for (int i = 0; i < 8; ++i) z += fast_exp2(fmaf(x[i], kLog2e, -m));
    }
    const float wm = wave_all(m, [](float a, float b) { return fmaxf(a, b); });
    z = wave_all(z * fast_exp2(m - wm), [](float a, float b) { return a + b; });
    if ((tid & 63) == 0) { sm[turn][tid >> 6] = wm; sz[turn][tid >> 6] = z; }
    __syncthreads();
    m = sm[turn][0];
#pragma unroll
    for (int w = 1; w < kOneWaves; ++w) m = fmaxf(m, sm[turn][w]);
    z = 0.f;
#pragma unroll
    for (int w = 0; w < kOneWaves; ++w) z += sz[turn][w] * fast_exp2(sm[turn][w] - m);
    const float l2 = m + fast_log2(z);
    // (a label outside [0, vocab) that is not the ignore index has no defined loss)
    if (tid == 0) loss[r] = l2 * kLn2 - xt;
    uint16_t* const out = grad + (int64_t)slot * ld_grad;
    const uint16_t* const nrow = logits + (int64_t)nr * ld;
    asm volatile("" : "+v"(lane0));
#pragma unroll
    for (int j = 0; j < kOneChunks; ++j)  // (the packed chunks are what stays in registers between the passes)
      asm volatile("" : "+v"(xr[j].x), "+v"(xr[j].y), "+v"(xr[j].z), "+v"(xr[j].w));
#pragma unroll
    for (int j = 0; j < kOneChunks; ++j) {
      const int c = lane0 + j * kOneThreads;
      if (c >= nchunks) continue;
      const uint32_t base = (uint32_t)c << 3;
      float x[8], d[8];
      unpack(xr[j], x);
#pragma unroll
      for (int i = 0; i < 8; ++i) d[i] = fast_exp2(fmaf(x[i], kLog2e, -l2));
      if (inside && c == (int)(label >> 3)) {
#pragma unroll
        for (int i = 0; i < 8; ++i) d[i] -= i == (int)(label & 7) ? 1.f : 0.f;
      }
      store8_vec<uint16_t>(out + base, d);
      if (more) xr[j] = ld16(nrow + base);
      __builtin_amdgcn_sched_barrier(0);  // (one chunk's unpacked values at a time)
    }
    if (!more) return;
    slot = next;
    r = nr;
    row = nrow;
  }
}

}  // namespace spx

using namespace spx;

static int label_ce_checks(const char* fn, const void* logits, int64_t ld, const void* labels,
                           int64_t rows, int64_t vocab, int dtype) {
  if (!(rows > 0 && rows < (1ll << 31))) return fail_arg(fn, "rows out of range");
  if (!(vocab > 0 && vocab < (1ll << 31))) return fail_arg(fn, "vocab out of range");
  if (!(logits && labels)) return fail_arg(fn, "null buffer");
  if (ld < vocab) return fail_arg(fn, "leading dimension smaller than vocab");
  if (!(dtype == SPX_DTYPE_BF16 || dtype == SPX_DTYPE_F32)) return fail_arg(fn, "dtype must be bf16 or fp32");
  return SPX_OK;
}

extern "C" int spx_label_ce_fwd(const void* logits, int64_t ld_logits, const int64_t* labels,
                                int64_t rows, int64_t vocab, int dtype, int64_t ignore_index,
                                float* loss, float* lse, int32_t* argmax, void* stream) {
  if (int rc = label_ce_checks(__func__, logits, ld_logits, labels, rows, vocab, dtype)) return rc;
  SPX_REQUIRE(loss && lse, "null output");
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  const int esz = dtype == SPX_DTYPE_BF16 ? 2 : 4;
  const bool vec = ptr_aligned16(logits) && (ld_logits * esz) % 16 == 0;
  const dim3 grid((unsigned)rows), block(kLossThreads);
#define SPX_LAUNCH(T, V)                                                                          \
  if (argmax)                                                                                     \
    hipLaunchKernelGGL((label_ce_fwd_kernel<T, V, true>), grid, block, 0, st,                     \
                       reinterpret_cast<const T*>(logits), ld_logits, labels, vocab, ignore_index, \
                       loss, lse, argmax);                                                        \
  else                                                                                            \
    hipLaunchKernelGGL((label_ce_fwd_kernel<T, V, false>), grid, block, 0, st,                    \
                       reinterpret_cast<const T*>(logits), ld_logits, labels, vocab, ignore_index, \
                       loss, lse, argmax)
  if (dtype == SPX_DTYPE_BF16) { if (vec) { SPX_LAUNCH(uint16_t, true); } else { SPX_LAUNCH(uint16_t, false); } }
  else { if (vec) { SPX_LAUNCH(float, true); } else { SPX_LAUNCH(float, false); } }
#undef SPX_LAUNCH
  return check_launch(__func__);
}

extern "C" int spx_label_ce_from_lse(const void* logits, int64_t ld_logits, const int64_t* labels,
                                     int64_t rows, int64_t vocab, int dtype, int64_t ignore_index,
                                     const float* lse, float* loss, void* stream) {
  if (int rc = label_ce_checks(__func__, logits, ld_logits, labels, rows, vocab, dtype)) return rc;
  SPX_REQUIRE(loss && lse, "null buffer");
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  const dim3 grid((unsigned)((rows + 255) / 256)), block(256);
  if (dtype == SPX_DTYPE_BF16)
    hipLaunchKernelGGL(label_ce_pick_kernel<uint16_t>, grid, block, 0, st,
                       reinterpret_cast<const uint16_t*>(logits), ld_logits, labels, rows, vocab, ignore_index,
                       lse, loss);
  else
    hipLaunchKernelGGL(label_ce_pick_kernel<float>, grid, block, 0, st, reinterpret_cast<const float*>(logits),
                       ld_logits, labels, rows, vocab, ignore_index, lse, loss);
  return check_launch(__func__);
}

static int label_ce_bwd_impl(const char* fn, const void* logits, int64_t ld_logits, const int64_t* labels,
                             const float* lse, const float* grad_rows, int64_t rows, int64_t vocab,
                             int dtype, int64_t ignore_index, void* dlogits, int64_t ld_out,
                             const int32_t* row_map, void* stream) {
  if (int rc = label_ce_checks(fn, logits, ld_logits, labels, rows, vocab, dtype)) return rc;
  if (!(lse && grad_rows && dlogits)) return fail_arg(fn, "null buffer");
  if (ld_out < vocab) return fail_arg(fn, "leading dimension of the gradient smaller than vocab");
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  const int esz = dtype == SPX_DTYPE_BF16 ? 2 : 4;
  const bool vec = ptr_aligned16(logits) && ptr_aligned16(dlogits) && (ld_logits * esz) % 16 == 0 &&
                   (ld_out * esz) % 16 == 0;
  const dim3 grid((unsigned)rows), block(kLossThreads);
#define SPX_LAUNCH(T, V)                                                                       \
  hipLaunchKernelGGL((label_ce_bwd_kernel<T, V>), grid, block, 0, st,                          \
                     reinterpret_cast<const T*>(logits), ld_logits, labels, lse, grad_rows, vocab, \
                     ignore_index, reinterpret_cast<T*>(dlogits), ld_out, row_map)
  if (dtype == SPX_DTYPE_BF16) { if (vec) SPX_LAUNCH(uint16_t, true); else SPX_LAUNCH(uint16_t, false); }
  else { if (vec) SPX_LAUNCH(float, true); else SPX_LAUNCH(float, false); }
#undef SPX_LAUNCH
  return check_launch(fn);
}

extern "C" int spx_label_ce_bwd(const void* logits, int64_t ld_logits, const int64_t* labels,
                                const float* lse, const float* grad_rows, int64_t rows,
                                int64_t vocab, int dtype, int64_t ignore_index, void* dlogits,
                                int64_t ld_out, void* stream) {
  return label_ce_bwd_impl(__func__, logits, ld_logits, labels, lse, grad_rows, rows, vocab, dtype,
                           ignore_index, dlogits, ld_out, nullptr, stream);
}

extern "C" int spx_label_ce_bwd_packed(const void* logits, int64_t ld_logits, const int64_t* labels,
                                       const float* lse, const float* grad_rows, int64_t rows,
                                       int64_t vocab, int dtype, int64_t ignore_index,
                                       const int32_t* row_map, void* dlogits, int64_t ld_out,
                                       void* stream) {
  if (!row_map) return fail_arg(__func__, "null row map");
  return label_ce_bwd_impl(__func__, logits, ld_logits, labels, lse, grad_rows, rows, vocab, dtype,
                           ignore_index, dlogits, ld_out, row_map, stream);
}

extern "C" int spx_label_ce_fwd_grad(const void* logits, int64_t ld_logits, const int64_t* labels, int64_t rows, int64_t vocab,
                                     int64_t ignore_index, float* loss, int32_t* row_map, int32_t* count, int32_t* row_of,
                                     void* grad_logits, int64_t ld_grad, void* stream) {
  if (int rc = label_ce_checks(__func__, logits, ld_logits, labels, rows, vocab, SPX_DTYPE_BF16)) return rc;
  SPX_REQUIRE(vocab % 8 == 0 && vocab <= (int64_t)kOneThreads * kOneChunks * 8, "vocab must be a multiple of 8, at most 155648");
  SPX_REQUIRE(loss && row_map && count && row_of && grad_logits, "null output");
  SPX_REQUIRE(ld_grad >= vocab && ld_grad % 8 == 0 && ld_logits % 8 == 0 && ptr_aligned16(logits) && ptr_aligned16(grad_logits),
              "rows must be 16-byte aligned, strides at least vocab");
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  hipLaunchKernelGGL(label_rows_kernel, dim3(1), dim3(1024), 0, st, labels, ignore_index, (int)rows, row_map, count, row_of,
                     loss);
  if (int rc = check_launch(__func__)) return rc;
  // a workgroup fills a compute unit
  hipLaunchKernelGGL(label_ce_fwd_grad_kernel, dim3((unsigned)(rows < 256 ? rows : 256)), dim3(kOneThreads), 0, st,
                     reinterpret_cast<const uint16_t*>(logits), ld_logits, labels, (int)vocab, row_of, count, loss,
                     reinterpret_cast<uint16_t*>(grad_logits), ld_grad);
  return check_launch(__func__);
}
