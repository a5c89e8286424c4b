// Row movement around the expert products of a sparse MoE block for gfx950 (HBM-bound, bf16 rows,
// 16-byte accesses).  The (token, slot) pairs of the router's top-k choice are sorted by expert on
// the host side of the library (a permutation, no arithmetic); these kernels move rows between the
// token order [T, H] and the sorted order [T * k, H]:
//   gather   sorted[p]  = scale[p] * x[src_row[p]]                      (scale optional)
//   combine  out[t]     = sum_j weight[t, j] * sorted[pos[t, j]]        (weight optional)
//   dot      d[t, j]    = <a[t], sorted[pos[t, j]]>                     (gradient of the router scores)
// Sums run in fp32 in the order j = 0 .. k-1 and are rounded once.

#include "spx_common.h"
#include "../../include/spx.h"

namespace spx {
namespace moe {

__device__ __forceinline__ void unpack8(u32x4 raw, float v[8]) {
  v[0] = bf16_lo(raw.x); v[1] = bf16_hi(raw.x);
  v[2] = bf16_lo(raw.y); v[3] = bf16_hi(raw.y);
  v[4] = bf16_lo(raw.z); v[5] = bf16_hi(raw.z);
  v[6] = bf16_lo(raw.w); v[7] = bf16_hi(raw.w);
}
__device__ __forceinline__ u32x4 pack8(const float v[8]) {
  u32x4 r;
  r.x = pack_bf16x2(v[0], v[1]); r.y = pack_bf16x2(v[2], v[3]);
  r.z = pack_bf16x2(v[4], v[5]); r.w = pack_bf16x2(v[6], v[7]);
  return r;
}

// one thread: 8 consecutive columns of one sorted row
__global__ __launch_bounds__(256) void gather_rows_kernel(const uint16_t* __restrict__ x, int64_t ld_x,
                                                          const int32_t* __restrict__ src_row,
                                                          const float* __restrict__ scale,
                                                          uint16_t* __restrict__ out, int64_t ld_out,
                                                          int64_t rows, int64_t src_rows, int h8) {
  const int64_t item = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (item >= rows * h8) return;
  const int64_t p = item / h8;
  const int c = (int)(item % h8) * 8;
  const int64_t r = src_row[p];
  u32x4 raw = {0u, 0u, 0u, 0u};
  if (r >= 0 && r < src_rows) raw = *reinterpret_cast<const u32x4*>(x + r * ld_x + c);
  if (scale) {
    float v[8];
    unpack8(raw, v);
    const float s = scale[p];
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] *= s;
    raw = pack8(v);
  }
  *reinterpret_cast<u32x4*>(out + p * ld_out + c) = raw;
}

// one thread: 8 consecutive columns of one token row, the k sorted rows added in slot order
__global__ __launch_bounds__(256) void combine_rows_kernel(const uint16_t* __restrict__ sorted, int64_t ld_s,
                                                           const int32_t* __restrict__ pos,
                                                           const float* __restrict__ weight,
                                                           uint16_t* __restrict__ out, int64_t ld_out,
                                                           int64_t tokens, int k, int64_t sorted_rows, int h8) {
  const int64_t item = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (item >= tokens * h8) return;
  const int64_t t = item / h8;
  const int c = (int)(item % h8) * 8;
  float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  for (int j = 0; j < k; ++j) {
    const int64_t p = pos[t * k + j];
    if (p < 0 || p >= sorted_rows) continue;
    float v[8];
    unpack8(*reinterpret_cast<const u32x4*>(sorted + p * ld_s + c), v);
    const float w = weight ? weight[t * k + j] : 1.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) acc[e] += w * v[e];
  }
  *reinterpret_cast<u32x4*>(out + t * ld_out + c) = pack8(acc);
}

// one wave per (token, slot)
__global__ __launch_bounds__(256) void pair_dot_kernel(const uint16_t* __restrict__ a, int64_t ld_a,
                                                       const uint16_t* __restrict__ sorted, int64_t ld_s,
                                                       const int32_t* __restrict__ pos, float* __restrict__ out,
                                                       int64_t pairs, int k, int64_t sorted_rows, int h8) {
  const int64_t pair = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (pair >= pairs) return;
  const int lane = threadIdx.x & 63;
  const int64_t t = pair / k;
  const int64_t p = pos[pair];
  float sum = 0.f;
  if (p >= 0 && p < sorted_rows) {
    for (int ch = lane; ch < h8; ch += 64) {
      float u[8], v[8];
      unpack8(*reinterpret_cast<const u32x4*>(a + t * ld_a + ch * 8), u);
      unpack8(*reinterpret_cast<const u32x4*>(sorted + p * ld_s + ch * 8), v);
#pragma unroll
      for (int e = 0; e < 8; ++e) sum += u[e] * v[e];
    }
  }
  sum = wave_sum(sum);
  if (lane == 0) out[pair] = sum;
}

// ---------------------------------------------------------------- backward of SwiGLU under the router's weight
// An expert's output is linear in its activation, so with d[p] = W_down^T dout[token of p], not weighted yet, everything the
// backward needs of the weight s[p] = scores[order[p]] is formed here, where a row is 512 to 768 wide, instead of on rows of
// the hidden size: the weighted activation, which the down projection's weight gradient contracts with dout's rows as they
// are; s[p]'s own gradient <d[p], silu(gate) * up>; and the gradient of gate and up.  Products in fp32, silu rounded to bf16
// as in the forward, one rounding a result.  Bound by memory: 40960 rows of 512 42 us (0.25 GB); the plain SwiGLU backward 33, and the
// weight's gradient from the outputs' rows of 2048 33 more and a gather of the weights 6.
// one wave per row
template <typename T>
__global__ __launch_bounds__(256) void weighted_swiglu_bwd_kernel(const uint16_t* __restrict__ hid, int64_t ld,
                                                                  const int64_t* __restrict__ order,
                                                                  const float* __restrict__ scores,
                                                                  const uint16_t* __restrict__ dact, int64_t ld_d,
                                                                  uint16_t* __restrict__ dhid, int64_t ld_dh,
                                                                  uint16_t* __restrict__ act, int64_t ld_act,
                                                                  T* __restrict__ dscores, int64_t rows, int inter8) {
  const int64_t p = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (p >= rows) return;
  const int lane = threadIdx.x & 63;
  const int64_t pair = order[p];
  const float s = scores[pair];
  float sum = 0.f;
  for (int ch = lane; ch < inter8; ch += 64) {
    float g[8], u[8], d[8], og[8], ou[8], oa[8];
    unpack8(*reinterpret_cast<const u32x4*>(hid + p * ld + ch * 8), g);
    unpack8(*reinterpret_cast<const u32x4*>(hid + p * ld + inter8 * 8 + ch * 8), u);
    unpack8(*reinterpret_cast<const u32x4*>(dact + p * ld_d + ch * 8), d);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float sg = 1.f / (1.f + __expf(-g[e])), silu = g[e] * sg;
      oa[e] = bf16_bits_to_f32(f32_to_bf16_bits(silu)) * u[e];
      sum += d[e] * oa[e];
      oa[e] *= s;
      d[e] *= s;
      ou[e] = d[e] * silu;
      og[e] = d[e] * u[e] * (sg * (1.f + g[e] * (1.f - sg)));
    }
    *reinterpret_cast<u32x4*>(dhid + p * ld_dh + ch * 8) = pack8(og);
    *reinterpret_cast<u32x4*>(dhid + p * ld_dh + inter8 * 8 + ch * 8) = pack8(ou);
    if (act) *reinterpret_cast<u32x4*>(act + p * ld_act + ch * 8) = pack8(oa);
  }
  if (!dscores) return;
  sum = wave_sum(sum);
  if (lane == 0) {
    if constexpr (sizeof(T) == 2) dscores[pair] = (T)f32_to_bf16_bits(sum);
    else dscores[pair] = sum;
  }
}

// ---------------------------------------------------------------- (token, slot) pairs sorted by expert
// A stable counting sort in three launches.  A wave owns `per_wave` consecutive pairs (a multiple of 64): it counts
// them per expert, the scan turns the counts into first positions (expert-major, waves in their order inside an
// expert), and the wave walks its pairs again, 64 at a time, giving every pair the position of its expert's next free
// row -- lanes of the same expert rank themselves by the ballots of the id's bits, lower lanes first, so the order
// inside an expert is the order of the pairs.  Bound by latency.
constexpr int kSortWaves = 4;         // waves per workgroup
constexpr int kSortMaxExperts = 2048;  // LDS counters: kSortWaves * experts * 4 bytes

__device__ __forceinline__ int sort_expert(const int64_t* __restrict__ idx, int64_t i, int experts) {
  const int64_t e = idx[i];
  return (int)(e < 0 ? 0 : e >= experts ? experts - 1 : e);
}

__global__ __launch_bounds__(64 * kSortWaves) void sort_count_kernel(const int64_t* __restrict__ idx, int64_t pairs,
                                                                     int experts, int per_wave, int waves,
                                                                     int32_t* __restrict__ counts) {
  extern __shared__ int32_t cnt[];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, wave = blockIdx.x * kSortWaves + w;
  int32_t* const mine = cnt + w * experts;
  for (int e = lane; e < experts; e += 64) mine[e] = 0;
  __syncthreads();
  const int64_t first = (int64_t)wave * per_wave, last = min(first + per_wave, pairs);
  if (wave < waves)
    for (int64_t i = first + lane; i < last; i += 64) atomicAdd(&mine[sort_expert(idx, i, experts)], 1);
  __syncthreads();
  if (wave < waves)
    for (int e = lane; e < experts; e += 64) counts[(int64_t)wave * experts + e] = mine[e];
}

// counts[wave][e] -> first position of the wave's pairs of expert e; offsets[e] = first row of expert e
__global__ __launch_bounds__(1024) void sort_scan_kernel(int32_t* __restrict__ counts, int experts, int waves,
                                                         int32_t* __restrict__ offsets) {
  __shared__ int32_t sums[1024];
  const int t = threadIdx.x;
  const int per = (experts + 1023) / 1024;  // experts a thread: one contiguous run
  int total = 0;
  for (int j = 0; j < per; ++j) {
    const int e = t * per + j;
    if (e >= experts) break;
    int run = 0;
    int w = 0;
    for (; w + 8 <= waves; w += 8) {
      int32_t v[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) v[u] = counts[(int64_t)(w + u) * experts + e];
#pragma unroll
      for (int u = 0; u < 8; ++u) run += v[u];
    }
    for (; w < waves; ++w) run += counts[(int64_t)w * experts + e];
    total += run;
  }
  sums[t] = total;
  __syncthreads();
  for (int d = 1; d < 1024; d <<= 1) {
    const int v = t >= d ? sums[t - d] : 0;
    __syncthreads();
    sums[t] += v;
    __syncthreads();
  }
  int at = sums[t] - total;
  for (int j = 0; j < per; ++j) {
    const int e = t * per + j;
    if (e >= experts) break;
    offsets[e] = at;
    int w = 0;
    for (; w + 8 <= waves; w += 8) {
      int32_t v[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) v[u] = counts[(int64_t)(w + u) * experts + e];
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        counts[(int64_t)(w + u) * experts + e] = at;
        at += v[u];
      }
    }
    for (; w < waves; ++w) {
      const int v = counts[(int64_t)w * experts + e];
      counts[(int64_t)w * experts + e] = at;
      at += v;
    }
  }
  if (t == 1023) offsets[experts] = sums[1023];
}

__global__ __launch_bounds__(64 * kSortWaves) void sort_scatter_kernel(
    const int64_t* __restrict__ idx, int64_t pairs, int experts, int bits, int k, int per_wave, int waves,
    const int32_t* __restrict__ counts, int64_t* __restrict__ order, int32_t* __restrict__ src_row,
    int32_t* __restrict__ pos) {
  extern __shared__ int32_t cnt[];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, wave = blockIdx.x * kSortWaves + w;
  if (wave >= waves) return;  // (no barrier below: a wave touches its own counters only)
  volatile int32_t* const mine = cnt + w * experts;
  for (int e = lane; e < experts; e += 64) mine[e] = counts[(int64_t)wave * experts + e];
  const int64_t first = (int64_t)wave * per_wave, last = min(first + per_wave, pairs);
  for (int64_t i0 = first; i0 < last; i0 += 64) {
    const int64_t i = i0 + lane;
    const bool live = i < last;
    const int e = live ? sort_expert(idx, i, experts) : 0;
    uint64_t same = __ballot(live);
    for (int b = 0; b < bits; ++b) {
      const uint64_t bal = __ballot((e >> b) & 1);
      same &= ((e >> b) & 1) ? bal : ~bal;
    }
    const int rank = __popcll(same & ((1ull << lane) - 1));
    int at = 0;
    if (live) at = mine[e] + rank;
    __builtin_amdgcn_wave_barrier();
    if (live && rank == 0) mine[e] = at + __popcll(same);
    __builtin_amdgcn_wave_barrier();
    if (live) {
      order[at] = i;
      src_row[at] = (int32_t)(i / k);
      pos[i] = at;
    }
  }
}

}  // namespace moe
}  // namespace spx

using namespace spx;

static bool al16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

extern "C" int spx_moe_gather_rows(const void* x, int64_t ld_x, int64_t src_rows, const int32_t* src_row,
                                   const float* scale, void* out, int64_t ld_out, int64_t rows, int64_t H,
                                   void* stream) {
  SPX_REQUIRE(rows > 0 && src_rows > 0 && H > 0 && H % 8 == 0, "rows > 0 and H a positive multiple of 8");
  SPX_REQUIRE(x && src_row && out && al16(x) && al16(out), "null or unaligned buffer");
  SPX_REQUIRE(ld_x % 8 == 0 && ld_out % 8 == 0 && ld_x >= H && ld_out >= H, "row strides must be multiples of 8 and at least H");
  const int64_t items = rows * (H / 8);
  hipLaunchKernelGGL(moe::gather_rows_kernel, dim3((unsigned)((items + 255) / 256)), dim3(256), 0,
                     reinterpret_cast<hipStream_t>(stream), reinterpret_cast<const uint16_t*>(x), ld_x, src_row,
                     scale, reinterpret_cast<uint16_t*>(out), ld_out, rows, src_rows, (int)(H / 8));
  return check_launch(__func__);
}

extern "C" int spx_moe_combine_rows(const void* sorted, int64_t ld_sorted, int64_t sorted_rows,
                                    const int32_t* pos, const float* weight, void* out, int64_t ld_out,
                                    int64_t tokens, int32_t k, int64_t H, void* stream) {
  SPX_REQUIRE(tokens > 0 && k > 0 && sorted_rows > 0 && H > 0 && H % 8 == 0, "tokens, k > 0 and H a positive multiple of 8");
  SPX_REQUIRE(sorted && pos && out && al16(sorted) && al16(out), "null or unaligned buffer");
  SPX_REQUIRE(ld_sorted % 8 == 0 && ld_out % 8 == 0 && ld_sorted >= H && ld_out >= H,
              "row strides must be multiples of 8 and at least H");
  const int64_t items = tokens * (H / 8);
  hipLaunchKernelGGL(moe::combine_rows_kernel, dim3((unsigned)((items + 255) / 256)), dim3(256), 0,
                     reinterpret_cast<hipStream_t>(stream), reinterpret_cast<const uint16_t*>(sorted), ld_sorted,
                     pos, weight, reinterpret_cast<uint16_t*>(out), ld_out, tokens, (int)k, sorted_rows,
                     (int)(H / 8));
  return check_launch(__func__);
}

extern "C" int spx_moe_pair_dot(const void* a, int64_t ld_a, const void* sorted, int64_t ld_sorted,
                                int64_t sorted_rows, const int32_t* pos, float* out, int64_t tokens,
                                int32_t k, int64_t H, void* stream) {
  SPX_REQUIRE(tokens > 0 && k > 0 && sorted_rows > 0 && H > 0 && H % 8 == 0, "tokens, k > 0 and H a positive multiple of 8");
  SPX_REQUIRE(a && sorted && pos && out && al16(a) && al16(sorted), "null or unaligned buffer");
  SPX_REQUIRE(ld_a % 8 == 0 && ld_sorted % 8 == 0 && ld_a >= H && ld_sorted >= H,
              "row strides must be multiples of 8 and at least H");
  const int64_t pairs = tokens * k;
  hipLaunchKernelGGL(moe::pair_dot_kernel, dim3((unsigned)((pairs + 3) / 4)), dim3(256), 0,
                     reinterpret_cast<hipStream_t>(stream), reinterpret_cast<const uint16_t*>(a), ld_a,
                     reinterpret_cast<const uint16_t*>(sorted), ld_sorted, pos, out, pairs, (int)k, sorted_rows,
                     (int)(H / 8));
  return check_launch(__func__);
}

extern "C" int spx_moe_swiglu_bwd(const void* hid, int64_t ld_hid, const int64_t* order, const float* scores, const void* dact,
                                   int64_t ld_dact, void* dhid, int64_t ld_dhid, void* act, int64_t ld_act,
                                  void* dscores, int dscores_f32, int64_t rows, int64_t inter, void* stream) {
  SPX_REQUIRE(rows > 0 && inter > 0 && inter % 8 == 0 && inter < (1ll << 30), "rows > 0 and the width a positive multiple of 8");
  SPX_REQUIRE(hid && order && scores && dact && dhid && al16(hid) && al16(dact) && al16(dhid) && al16(act),
              "null or unaligned buffer");
  SPX_REQUIRE(ld_hid % 8 == 0 && ld_dact % 8 == 0 && ld_dhid % 8 == 0 && ld_hid >= 2 * inter && ld_dhid >= 2 * inter &&
                  ld_dact >= inter && (!act || (ld_act % 8 == 0 && ld_act >= inter)),
              "row strides must be multiples of 8 and at least the rows' width");
  SPX_REQUIRE((rows + 3) / 4 < (1ll << 31), "too many rows");
  const dim3 grid((unsigned)((rows + 3) / 4)), block(256);
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  const uint16_t *const h = reinterpret_cast<const uint16_t*>(hid), *const d = reinterpret_cast<const uint16_t*>(dact);
  uint16_t *const o = reinterpret_cast<uint16_t*>(dhid), *const w = reinterpret_cast<uint16_t*>(act);
  if (dscores_f32)
    hipLaunchKernelGGL(moe::weighted_swiglu_bwd_kernel<float>, grid, block, 0, st, h, ld_hid, order, scores, d, ld_dact, o, ld_dhid, w, ld_act,
                       reinterpret_cast<float*>(dscores), rows, (int)(inter / 8));
  else
    hipLaunchKernelGGL(moe::weighted_swiglu_bwd_kernel<uint16_t>, grid, block, 0, st, h, ld_hid, order, scores, d, ld_dact, o, ld_dhid, w, ld_act,
                       reinterpret_cast<uint16_t*>(dscores), rows, (int)(inter / 8));
  return check_launch(__func__);
}

static int sort_plan(int64_t pairs, int& per_wave) {
  // about 128 waves at most: the scan reads one row of counts per wave
  per_wave = 256;
  while ((pairs + per_wave - 1) / per_wave > 128) per_wave *= 2;
  return (int)((pairs + per_wave - 1) / per_wave);
}

extern "C" int64_t spx_moe_sort_workspace_bytes(int64_t pairs, int64_t experts) {
  if (pairs <= 0 || experts <= 0) return 0;
  int per_wave;
  return (int64_t)sort_plan(pairs, per_wave) * experts * (int64_t)sizeof(int32_t);
}

extern "C" int spx_moe_sort_pairs(const int64_t* idx, int64_t tokens, int32_t k, int64_t experts, int64_t* order,
                                  int32_t* src_row, int32_t* pos, int32_t* offsets, void* workspace,
                                  int64_t workspace_bytes, void* stream) {
  SPX_REQUIRE(tokens > 0 && k > 0, "tokens and k must be positive");
  SPX_REQUIRE(tokens * k < (1ll << 31), "too many pairs");
  SPX_REQUIRE(experts > 0 && experts <= spx::moe::kSortMaxExperts, "1 .. 2048 experts");
  SPX_REQUIRE(idx && order && src_row && pos && offsets && workspace, "null buffer");
  SPX_REQUIRE(((uintptr_t)workspace) % 4 == 0, "unaligned workspace");
  const int64_t pairs = tokens * k;
  SPX_REQUIRE(workspace_bytes >= spx_moe_sort_workspace_bytes(pairs, experts), "workspace too small");
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  int per_wave;
  const int waves = sort_plan(pairs, per_wave);
  int32_t* const counts = reinterpret_cast<int32_t*>(workspace);
  const dim3 grid((unsigned)((waves + spx::moe::kSortWaves - 1) / spx::moe::kSortWaves)),
      block(64 * spx::moe::kSortWaves);
  const int smem = spx::moe::kSortWaves * (int)experts * 4;
  int bits = 0;
  while ((1ll << bits) < experts) ++bits;
  hipLaunchKernelGGL(spx::moe::sort_count_kernel, grid, block, smem, st, idx, pairs, (int)experts, per_wave, waves, counts);
  hipLaunchKernelGGL(spx::moe::sort_scan_kernel, dim3(1), dim3(1024), 0, st, counts, (int)experts, waves, offsets);
  hipLaunchKernelGGL(spx::moe::sort_scatter_kernel, grid, block, smem, st, idx, pairs, (int)experts, bits, (int)k,
                     per_wave, waves, counts, order, src_row, pos);
  return spx::check_launch(__func__);
}
