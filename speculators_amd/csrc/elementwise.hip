// HBM-bound glue of the draft decoder layer for gfx950: RMSNorm, rotary
// embedding fused with the [T, heads*D] -> [heads, T, D] relayout, and the
// SwiGLU gate.  bf16 in / out, fp32 inside, 16-byte accesses.  Rounding points
// follow the HF blocks the reference is built from (LlamaRMSNorm,
// apply_rotary_pos_emb, LlamaMLP): every bf16 tensor op of the eager path is
// one rounding here.

#include "loss_common.h"
#include "spx_common.h"
#include "../../include/spx.h"

namespace spx {

__device__ __forceinline__ float round_bf16(float v) { return bf16_bits_to_f32(f32_to_bf16_bits(v)); }

__device__ __forceinline__ void unpack8f(u32x4 raw, float v[8]) {
  v[0] = bf16_lo(raw.x); v[1] = bf16_hi(raw.x);
  v[2] = bf16_lo(raw.y); v[3] = bf16_hi(raw.y);
  v[4] = bf16_lo(raw.z); v[5] = bf16_hi(raw.z);
  v[6] = bf16_lo(raw.w); v[7] = bf16_hi(raw.w);
}
__device__ __forceinline__ u32x4 pack8f(const float v[8]) {
  u32x4 r;
  r.x = pack_bf16x2(v[0], v[1]); r.y = pack_bf16x2(v[2], v[3]);
  r.z = pack_bf16x2(v[4], v[5]); r.w = pack_bf16x2(v[6], v[7]);
  return r;
}

template <int WAVES>
__device__ __forceinline__ float block_sum(float v, float* lds) {
  v = wave_sum(v);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) lds[threadIdx.x >> 6] = v;
  __syncthreads();
  float s = lds[0];
#pragma unroll
  for (int i = 1; i < WAVES; ++i) s += lds[i];
  return s;
}

// ---------------------------------------------------------------- RMSNorm
// y = w * bf16(x * rsqrt(mean(x^2) + eps));  one workgroup per row (H >= 512) or one
// wave per row (small H, e.g. per-head q/k norm).  MAXC = 16-byte chunks a lane keeps.
// RES: x is the sum of two tensors, x = bf16(x + res) (one rounding, as a bf16 tensor add),
// which is also written to `sum` for the residual stream.
// The kernel is bound by HBM where the rows fill the chip and by the launch below that: the two norms
// of the first layer (PAIR) are one launch of twice the workgroups, the upper half of the grid's y
// working on the second norm (T = 512, H = 2048: 3.7 us for the pair, 4.1 us for each one alone).
// PARTS: that second tensor is a product whose contraction was cut (rows of H, one after the other; stride floats from
// part to part): its partial results are added in their order and rounded here as the product's own last pass does, which
// saves that launch and the rounded tensor's way out and back.  T = 512, H = 2048: forward, four parts, 4.7 us for the pass
// and 4.3 for the norm before, 5.7 now; backward, eight parts, 6.6 and 5.5 before, 9.4 now (33 MB of partial results at
// 3.6 TB/s; four parts' loads in flight by hand measured the same).
struct NormParts {
  const float* at;
  int64_t stride;
  int count;
  __device__ __forceinline__ void sum(int64_t offset, float v[8]) const {
    f32x4 lo = {0.f, 0.f, 0.f, 0.f}, hi = lo;
    const float* src = at + offset;
    for (int p = 0; p < count; ++p, src += stride) {
      lo += *reinterpret_cast<const f32x4*>(src);
      hi += *reinterpret_cast<const f32x4*>(src + 4);
    }
    const float f[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
    unpack8f(pack8f(f), v);
  }
};

struct NormFwdSet {
  const uint16_t* x;
  int64_t ld_x;
  const uint16_t* w;
  uint16_t* y;
  int64_t ld_y;
  float* rstd;
};

template <int MAXC, bool WAVE_ROWS, bool RES = false, bool PAIR = false, int NT = 256, bool PARTS = false>
__global__ __launch_bounds__(NT) void rmsnorm_fwd_kernel(
    NormFwdSet one, NormFwdSet two, int64_t rows, int H,
    float eps, const uint16_t* __restrict__ res = nullptr, int64_t ld_res = 0,
    uint16_t* __restrict__ sum = nullptr, int64_t ld_sum = 0, NormParts parts = NormParts{}) {
  __shared__ float red[NT / 64];
  const bool second = PAIR && blockIdx.y;
  const uint16_t* __restrict__ x = second ? two.x : one.x;
  const uint16_t* __restrict__ w = second ? two.w : one.w;
  uint16_t* __restrict__ y = second ? two.y : one.y;
  float* __restrict__ rstd = second ? two.rstd : one.rstd;
  const int64_t ld_x = second ? two.ld_x : one.ld_x, ld_y = second ? two.ld_y : one.ld_y;
  const int nthr = WAVE_ROWS ? 64 : NT;
  const int t = WAVE_ROWS ? (threadIdx.x & 63) : threadIdx.x;
  const int64_t row = WAVE_ROWS ? (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6) : blockIdx.x;
  if (WAVE_ROWS && row >= rows) return;
  const int nch = H / 8;
  float v[MAXC][8];
  float ss = 0.f;
#pragma unroll
  for (int c = 0; c < MAXC; ++c) {
    const int ch = t + c * nthr;
    if (ch < nch) {
      unpack8f(*reinterpret_cast<const u32x4*>(x + row * ld_x + ch * 8), v[c]);
      if (RES) {
        float b[8];
        if (PARTS) parts.sum(row * H + ch * 8, b);
        else unpack8f(*reinterpret_cast<const u32x4*>(res + row * ld_res + ch * 8), b);
#pragma unroll
        for (int e = 0; e < 8; ++e) v[c][e] += b[e];
        const u32x4 packed = pack8f(v[c]);
        *reinterpret_cast<u32x4*>(sum + row * ld_sum + ch * 8) = packed;
        unpack8f(packed, v[c]);
      }
#pragma unroll
      for (int e = 0; e < 8; ++e) ss = fmaf(v[c][e], v[c][e], ss);
    }
  }
  ss = WAVE_ROWS ? wave_sum(ss) : block_sum<NT / 64>(ss, red);
  const float r = rsqrtf(ss / (float)H + eps);
  if (t == 0 && rstd) rstd[row] = r;
#pragma unroll
  for (int c = 0; c < MAXC; ++c) {
    const int ch = t + c * nthr;
    if (ch < nch) {
      float wv[8], o[8];
      unpack8f(*reinterpret_cast<const u32x4*>(w + ch * 8), wv);
#pragma unroll
      for (int e = 0; e < 8; ++e) o[e] = wv[e] * round_bf16(v[c][e] * r);
      *reinterpret_cast<u32x4*>(y + row * ld_y + ch * 8) = pack8f(o);
    }
  }
}

// dx = rstd * (g - xhat * mean(g * xhat)), g = dy * w, xhat = x * rstd;
// dw partial sums: block b accumulates the rows b, b + gridDim.x, ... per column.
// dres (may be null): gradient that reaches x along the residual stream, added before the
// one rounding of dx.  dx may be null (only dw wanted).  accumulate: the partial sums start from
// what dw_part holds (a gain that is applied several times per forward: one buffer, one final sum).
// Bound by HBM (x, dy, dres in, dx out; the partial sums are 1024 rows of fp32, read and written).  A
// lane keeps at most two 16-byte chunks of a row: with eight (wide rows on 256 threads) the four
// arrays took 256 registers and 8192 x 8192 took 233 us (2.3 TB/s); 512 or 1024 threads share such a row
// now: 106 us.
// The narrow form (one wave per row) adds its four waves' sums through LDS: the final sum over the
// slots has a quarter of the rows to read (a q / k norm of 128: 8192 slots before).
// PAIR as in the forward: the upper half of the grid's y is the second norm.
struct NormBwdSet {
  const uint16_t* x;
  int64_t ld_x;
  const uint16_t* w;
  const uint16_t* dy;
  int64_t ld_dy;
  const float* rstd;
  uint16_t* dx;
  int64_t ld_dx;
  float* dw_part;
  const uint16_t* dres;
  int64_t ld_dres;
  int accumulate;
};

template <int MAXC, bool WAVE_ROWS, bool PAIR = false, int NT = 256, bool PARTS = false>
__global__ __launch_bounds__(NT) void rmsnorm_bwd_kernel(NormBwdSet one, NormBwdSet two, int64_t rows, int H,
                                                         NormParts parts = NormParts{}) {
  __shared__ float red[WAVE_ROWS ? 4 * 512 : NT / 64];
  const bool second = PAIR && blockIdx.y;
  const uint16_t* __restrict__ x = second ? two.x : one.x;
  const uint16_t* __restrict__ w = second ? two.w : one.w;
  const uint16_t* __restrict__ dy = second ? two.dy : one.dy;
  const float* __restrict__ rstd = second ? two.rstd : one.rstd;
  uint16_t* __restrict__ dx = second ? two.dx : one.dx;
  float* __restrict__ dw_part = second ? two.dw_part : one.dw_part;
  const uint16_t* __restrict__ dres = second ? two.dres : one.dres;
  const int64_t ld_x = second ? two.ld_x : one.ld_x, ld_dy = second ? two.ld_dy : one.ld_dy;
  const int64_t ld_dx = second ? two.ld_dx : one.ld_dx, ld_dres = second ? two.ld_dres : one.ld_dres;
  const int accumulate = second ? two.accumulate : one.accumulate;
  const int nthr = WAVE_ROWS ? 64 : NT;
  const int t = WAVE_ROWS ? (threadIdx.x & 63) : threadIdx.x;
  const int wave = threadIdx.x >> 6;
  const int nch = H / 8;
  float wv[MAXC][8], dwacc[MAXC][8];
#pragma unroll
  for (int c = 0; c < MAXC; ++c) {
    const int ch = t + c * nthr;
    if (ch < nch) unpack8f(*reinterpret_cast<const u32x4*>(w + ch * 8), wv[c]);
#pragma unroll
    for (int e = 0; e < 8; ++e) dwacc[c][e] = 0.f;
    if (accumulate && dw_part && ch < nch && !(WAVE_ROWS && wave)) {
      const float* o = dw_part + (int64_t)blockIdx.x * H + ch * 8;
      const f32x4 a = *reinterpret_cast<const f32x4*>(o), b = *reinterpret_cast<const f32x4*>(o + 4);
      dwacc[c][0] = a.x; dwacc[c][1] = a.y; dwacc[c][2] = a.z; dwacc[c][3] = a.w;
      dwacc[c][4] = b.x; dwacc[c][5] = b.y; dwacc[c][6] = b.z; dwacc[c][7] = b.w;
    }
  }
  const int64_t first = WAVE_ROWS ? (int64_t)blockIdx.x * 4 + wave : blockIdx.x;
  const int64_t stride = WAVE_ROWS ? (int64_t)gridDim.x * 4 : gridDim.x;
  for (int64_t row = first; row < rows; row += stride) {
    const float r = rstd[row];
    float xh[MAXC][8], g[MAXC][8];
    float dot = 0.f;
#pragma unroll
    for (int c = 0; c < MAXC; ++c) {
      const int ch = t + c * nthr;
      if (ch < nch) {
        float xv[8], dv[8];
        unpack8f(*reinterpret_cast<const u32x4*>(x + row * ld_x + ch * 8), xv);
        if (PARTS) parts.sum(row * H + ch * 8, dv);
        else unpack8f(*reinterpret_cast<const u32x4*>(dy + row * ld_dy + ch * 8), dv);
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          xh[c][e] = xv[e] * r;
          g[c][e] = dv[e] * wv[c][e];
          dot = fmaf(g[c][e], xh[c][e], dot);
          dwacc[c][e] = fmaf(dv[e], xh[c][e], dwacc[c][e]);
        }
      }
    }
    if (dx == nullptr) continue;  // uniform: only the weight gradient is wanted
    dot = WAVE_ROWS ? wave_sum(dot) : block_sum<NT / 64>(dot, red);
    const float mean = dot / (float)H;
#pragma unroll
    for (int c = 0; c < MAXC; ++c) {
      const int ch = t + c * nthr;
      if (ch < nch) {
        float o[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) o[e] = r * (g[c][e] - xh[c][e] * mean);
        if (dres) {
          float dr[8];
          unpack8f(*reinterpret_cast<const u32x4*>(dres + row * ld_dres + ch * 8), dr);
#pragma unroll
          for (int e = 0; e < 8; ++e) o[e] += dr[e];
        }
        *reinterpret_cast<u32x4*>(dx + row * ld_dx + ch * 8) = pack8f(o);
      }
    }
  }
  if (dw_part) {
    if (WAVE_ROWS) {
#pragma unroll
      for (int c = 0; c < MAXC; ++c) {
        const int ch = t + c * nthr;
        if (ch < nch) {
#pragma unroll
          for (int e = 0; e < 8; ++e) red[wave * H + ch * 8 + e] = dwacc[c][e];
        }
      }
      __syncthreads();
      for (int c = threadIdx.x; c < H; c += NT)
        dw_part[(int64_t)blockIdx.x * H + c] = (red[c] + red[H + c]) + (red[2 * H + c] + red[3 * H + c]);
      return;
    }
#pragma unroll
    for (int c = 0; c < MAXC; ++c) {
      const int ch = t + c * nthr;
      if (ch < nch) {
        float* o = dw_part + (int64_t)blockIdx.x * H + ch * 8;
        f32x4 a = {dwacc[c][0], dwacc[c][1], dwacc[c][2], dwacc[c][3]};
        f32x4 b = {dwacc[c][4], dwacc[c][5], dwacc[c][6], dwacc[c][7]};
        *reinterpret_cast<f32x4*>(o) = a;
        *reinterpret_cast<f32x4*>(o + 4) = b;
      }
    }
  }
}

// dw[c] = sum_s dw_part[s, c]  (fixed order: deterministic), bf16 or fp32 out, of up to kSumSets gains in one launch.  One
// workgroup sums 32 columns of one of them (one 128-byte line per slot row): lane = (slot row j of 128, 4 columns),
// thread j adds the slots j, j + 128, ..., then the 128 partial sums are combined through LDS
// in a fixed order.  A latency-bound read of few megabytes by few workgroups: 1024 threads have
// eight loads each to wait for at 1024 slots (256 threads had 32: 11.6 us at H = 4096, 3.5 us now).
// Gains whose gradients are ready together end in one launch: fourteen of three layers of width 2048 14 x 5 -> 18 us, and their
// launches and casts off the host's path.
constexpr int kSumSets = 16;
struct SumSets {
  const float* part[kSumSets];
  void* out[kSumSets];
  int slots[kSumSets], H[kSumSets], end[kSumSets];  // end: workgroups, running
  uint32_t f32;                                     // bit i: out[i] is fp32
};
__global__ __launch_bounds__(1024) void colsum_kernel(SumSets p) {
  __shared__ float red[128][33];
  __shared__ float sub[8][33];
  int set = 0;
  while ((int)blockIdx.x >= p.end[set]) ++set;  // (the last end is the grid)
  const int block = blockIdx.x - (set ? p.end[set - 1] : 0);
  const float* const part = p.part[set];
  const int H = p.H[set], slots = p.slots[set];
  const int q = threadIdx.x & 7, j = threadIdx.x >> 3;
  const int c = block * 32 + q * 4;
  f32x4 s = {0.f, 0.f, 0.f, 0.f};
  if (c < H) {
#pragma unroll 8
    for (int i = j; i < slots; i += 128) {
      const f32x4 v = *reinterpret_cast<const f32x4*>(part + (int64_t)i * H + c);
      s.x += v.x; s.y += v.y; s.z += v.z; s.w += v.w;
    }
  }
  red[j][q * 4 + 0] = s.x; red[j][q * 4 + 1] = s.y; red[j][q * 4 + 2] = s.z; red[j][q * 4 + 3] = s.w;
  __syncthreads();
  const int col = threadIdx.x & 31, g = threadIdx.x >> 5;
  if (g < 8) {
    float t = 0.f;
#pragma unroll
    for (int k = 0; k < 16; ++k) t += red[g * 16 + k][col];
    sub[g][col] = t;
  }
  __syncthreads();
  const int at = block * 32 + (int)threadIdx.x;
  if (threadIdx.x < 32 && at < H) {
    float t = 0.f;
#pragma unroll
    for (int k = 0; k < 8; ++k) t += sub[k][threadIdx.x];
    if (p.f32 >> set & 1) static_cast<float*>(p.out[set])[at] = t;
    else static_cast<uint16_t*>(p.out[set])[at] = (uint16_t)f32_to_bf16_bits(t);
  }
}
static SumSets one_sum(const float* part, int64_t slots, int64_t H, void* out) {
  SumSets p{};
  p.part[0] = part; p.out[0] = out; p.slots[0] = (int)slots; p.H[0] = (int)H; p.end[0] = (int)((H + 31) / 32);
  return p;
}
static void launch_sums(const SumSets& p, int count, hipStream_t st) {
  hipLaunchKernelGGL(colsum_kernel, dim3((unsigned)p.end[count - 1]), dim3(1024), 0, st, p);
}

// ---------------------------------------------------------------- RoPE + relayout
// forward:  out[h, t, :] = rope(x[t, h, :], pos[t])      x: [T, heads*D] (row stride ld_x)
// inverse:  out[t, h, :] = rope^T(x[h, t, :], pos[t])    (the backward of the above)
// rotate == 0: relayout only (used for V).  cos / sin are evaluated in fp32 from
// pos * inv_freq and rounded to bf16, as the HF rotary module does.
template <bool INVERSE>
__global__ __launch_bounds__(256) void rope_kernel(const uint16_t* __restrict__ x, int64_t ld_x,
                                                   const int64_t* __restrict__ pos,
                                                   const float* __restrict__ inv_freq,
                                                   uint16_t* __restrict__ out, int64_t ld_out, int T,
                                                   int heads, int D, int rotate, int64_t pos_offset,
                                                   int tok_head_stride, int rot, float table_scale) {
  // one thread: 8 consecutive d of the first half of the rotated part and the matching 8 of its
  // second half, or 16 consecutive d of the part that passes unrotated (rot < D: partial rotary)
  const int per_row = D / 16;
  const int64_t item = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int64_t total = (int64_t)T * heads * per_row;
  if (item >= total) return;
  const int d0 = (int)(item % per_row) * 8;
  const int h = (int)((item / per_row) % heads);
  const int t = (int)(item / ((int64_t)per_row * heads));
  const bool pass = d0 * 2 >= rot;  // items past the rotated part copy 16 contiguous elements
  const int half = pass ? 8 : rot / 2;
  const int dA = pass ? d0 * 2 : d0;
  // the head-major side is [heads][T][D] with a head stride of its own (0 = T * D, contiguous):
  // it may be a window of a longer key / value cache
  const int64_t hs = INVERSE ? (ld_x ? ld_x : (int64_t)T * D) : (ld_out ? ld_out : (int64_t)T * D);
  const uint16_t* src = INVERSE ? x + (int64_t)h * hs + (int64_t)t * D : x + (int64_t)t * ld_x + h * tok_head_stride;
  uint16_t* dst = INVERSE ? out + (int64_t)t * ld_out + h * tok_head_stride : out + (int64_t)h * hs + (int64_t)t * D;
  float a[8], b[8], oa[8], ob[8];
  unpack8f(*reinterpret_cast<const u32x4*>(src + dA), a);
  unpack8f(*reinterpret_cast<const u32x4*>(src + half + dA), b);
  if (rotate && !pass) {
    const float p = (float)(pos[t] + pos_offset);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float ang = p * inv_freq[d0 + e];
      // (table_scale: the attention factor some frequency scalings put on both tables, 1 otherwise)
      float sn, cs;
      sincosf(ang, &sn, &cs);
      const float c = round_bf16(cs * table_scale);
      float s = round_bf16(sn * table_scale);
      if (INVERSE) s = -s;
      // x*cos + rotate_half(x)*sin with each bf16 op rounded
      oa[e] = round_bf16(a[e] * c) + round_bf16(-b[e] * s);
      ob[e] = round_bf16(b[e] * c) + round_bf16(a[e] * s);
    }
  } else {
#pragma unroll
    for (int e = 0; e < 8; ++e) { oa[e] = a[e]; ob[e] = b[e]; }
  }
  *reinterpret_cast<u32x4*>(dst + dA) = pack8f(oa);
  *reinterpret_cast<u32x4*>(dst + half + dA) = pack8f(ob);
}

// The relayout of a merged q/k/v projection [T, (hq + 2 hkv) * D] (row stride ld) in one launch: q and k
// rotated, v moved.  Head-major sides [heads][T][D] with a head stride each (k and v may be windows of a
// cache).  INVERSE: the other way with the transposed rotation; a null source is a gradient of zeros.
// Bound by HBM, and by the evaluation of cos / sin where every head does its own: a thread works on the
// same 16 elements of HEADS heads of one token (head i * groups + hg: neighbouring lanes stay on
// neighbouring heads of the token-major row) and evaluates the angles once.  4096 tokens of 48 heads of
// 128: 32 us, three launches of the kernel above 47 us; 512 tokens of 48 x 64: 6.0 us for 20.
template <bool INVERSE, int HEADS>
__global__ __launch_bounds__(256) void rope_qkv_kernel(uint16_t* __restrict__ tok, int64_t ld,
                                                       uint16_t* __restrict__ q, int64_t hs_q,
                                                       uint16_t* __restrict__ k, int64_t hs_k,
                                                       uint16_t* __restrict__ v, int64_t hs_v,
                                                       const int64_t* __restrict__ pos,
                                                       const float* __restrict__ inv_freq, int T, int hq, int hkv,
                                                       int D, int rot, int64_t pos_offset, float table_scale) {
  const unsigned per_row = (unsigned)D / 16;
  const int heads = hq + 2 * hkv;
  const unsigned groups = (unsigned)(heads + HEADS - 1) / HEADS;
  const unsigned item = blockIdx.x * 256u + threadIdx.x;
  if (item >= (unsigned)T * groups * per_row) return;
  const int d0 = (int)(item % per_row) * 8;
  const unsigned rest = item / per_row;
  const int hg = (int)(rest % groups);
  const int t = (int)(rest / groups);
  const bool pass = d0 * 2 >= rot;
  const int half = pass ? 8 : rot / 2;
  const int dA = pass ? d0 * 2 : d0;
  u32x4 ra[HEADS], rb[HEADS];
#pragma unroll
  for (int i = 0; i < HEADS; ++i) {
    const int h = i * (int)groups + hg;
    ra[i] = u32x4{0, 0, 0, 0};
    rb[i] = u32x4{0, 0, 0, 0};
    if (h < heads) {
      const uint16_t* src;
      if (INVERSE) {
        src = h < hq ? q : (h < hq + hkv ? k : v);
        const int64_t hs = h < hq ? hs_q : (h < hq + hkv ? hs_k : hs_v);
        const int hh = h < hq ? h : (h < hq + hkv ? h - hq : h - hq - hkv);
        if (src) src += (int64_t)hh * hs + (int64_t)t * D;
      } else {
        src = tok + (int64_t)t * ld + h * D;
      }
      if (!INVERSE || src) {
        ra[i] = *reinterpret_cast<const u32x4*>(src + dA);
        rb[i] = *reinterpret_cast<const u32x4*>(src + half + dA);
      }
    }
  }
  float c[8], s[8];
  if (!pass && hg < hq + hkv) {
    const float p = (float)(pos[t] + pos_offset);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float ang = p * inv_freq[d0 + e];
      float sn, cs;
      sincosf(ang, &sn, &cs);  // one argument reduction for both
      c[e] = round_bf16(cs * table_scale);
      s[e] = round_bf16(sn * table_scale);
      if (INVERSE) s[e] = -s[e];
    }
  }
#pragma unroll
  for (int i = 0; i < HEADS; ++i) {
    const int h = i * (int)groups + hg;
    if (h < heads) {
      uint16_t* dst;
      if (INVERSE) {
        dst = tok + (int64_t)t * ld + h * D;
      } else {
        const int64_t hs = h < hq ? hs_q : (h < hq + hkv ? hs_k : hs_v);
        const int hh = h < hq ? h : (h < hq + hkv ? h - hq : h - hq - hkv);
        dst = (h < hq ? q : (h < hq + hkv ? k : v)) + (int64_t)hh * hs + (int64_t)t * D;
      }
      if (!pass && h < hq + hkv) {
        float a[8], b[8], oa[8], ob[8];
        unpack8f(ra[i], a);
        unpack8f(rb[i], b);
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          oa[e] = round_bf16(a[e] * c[e]) + round_bf16(-b[e] * s[e]);
          ob[e] = round_bf16(b[e] * c[e]) + round_bf16(a[e] * s[e]);
        }
        ra[i] = pack8f(oa);
        rb[i] = pack8f(ob);
      }
      *reinterpret_cast<u32x4*>(dst + dA) = ra[i];
      *reinterpret_cast<u32x4*>(dst + half + dA) = rb[i];
    }
  }
}

// ---------------------------------------------------------------- per-head RMSNorm + rotary embedding + relayout
// Heads 0 .. n_heads - 1 of a token row (n_heads * D elements, head h at h * D) are normed over their D elements, rotated
// and written head-major; the n_pass heads behind them are only moved (the values).  The rounding points are those of the
// separate kernels: bf16(x * rstd), its product with the gain, each product and the sum of the rotation.  D / 16 lanes share
// a head, each with the two chunks of eight that rotate together; a thread works on HEADS heads of one token and evaluates
// the angles once.  Bound by HBM where the rows fill the chip; one read and one write of q and k where the norm and the
// relayout made two each (16384 tokens, 16 + 2 heads of 256: 345 us -> 91, the way back 375 -> 120).  A layer's queries and its
// keys with the values go in one launch: workgroups from `first` on have the second set (three layers of 888 / 2665
// rows of 32 and 8 + 8 heads of 64, forward 42 -> 28 us, back 49 -> 39; five of 8192 / 16384 of 128 378 -> 351, 530 -> 484).
struct HeadSets {
  spx_head_norm set[2];
  int first;      // workgroups of set 0
};
template <int D, int HEADS>
__global__ __launch_bounds__(256) void head_norm_rope_kernel(HeadSets sets, const float* __restrict__ inv_freq,
                                                             int64_t pos_offset, float table_scale) {
  constexpr int L = D / 16;
  const int which = (int)blockIdx.x >= sets.first;
  const spx_head_norm& in = sets.set[which];
  const uint16_t* __restrict__ const tok = reinterpret_cast<const uint16_t*>(in.tok);
  const uint16_t* __restrict__ const gain = reinterpret_cast<const uint16_t*>(in.gain);
  uint16_t* __restrict__ const out = reinterpret_cast<uint16_t*>(in.out);
  uint16_t* __restrict__ const pass = reinterpret_cast<uint16_t*>(in.pass);
  float* __restrict__ const rstd = in.rstd;
  const int64_t* __restrict__ const pos = in.position_ids;
  const int64_t ld = in.ld_tok, hs_out = in.out_head_stride, hs_pass = in.pass_head_stride;
  const int T = (int)in.T, n_heads = in.n_heads, n_pass = in.n_pass;
  const float eps = in.eps;
  const int heads = n_heads + n_pass, groups = (heads + HEADS - 1) / HEADS;
  const int64_t item = (int64_t)((int)blockIdx.x - (which ? sets.first : 0)) * (256 / L) + threadIdx.x / L;
  if (item >= (int64_t)T * groups) return;  // (all lanes of a head together)
  const int hg = (int)(item % groups), t = (int)(item / groups);
  const int part = threadIdx.x % L, d0 = part * 8;
  u32x4 ra[HEADS], rb[HEADS];
#pragma unroll
  for (int i = 0; i < HEADS; ++i) {
    const int h = i * groups + hg;
    ra[i] = rb[i] = u32x4{0, 0, 0, 0};
    if (h < heads) {
      const uint16_t* src = tok + (int64_t)t * ld + h * D + d0;
      ra[i] = *reinterpret_cast<const u32x4*>(src);
      rb[i] = *reinterpret_cast<const u32x4*>(src + D / 2);
    }
  }
  float c[8], s[8], wa[8], wb[8];
  if (hg < n_heads) {
    unpack8f(*reinterpret_cast<const u32x4*>(gain + d0), wa);
    unpack8f(*reinterpret_cast<const u32x4*>(gain + D / 2 + d0), wb);
    const float p = (float)(pos[t] + pos_offset);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      float sn, cs;
      sincosf(p * inv_freq[d0 + e], &sn, &cs);
      c[e] = round_bf16(cs * table_scale);
      s[e] = round_bf16(sn * table_scale);
    }
  }
#pragma unroll
  for (int i = 0; i < HEADS; ++i) {
    const int h = i * groups + hg;
    float a[8], b[8], ss = 0.f;
    unpack8f(ra[i], a);
    unpack8f(rb[i], b);
#pragma unroll
    for (int e = 0; e < 8; ++e) ss = fmaf(a[e], a[e], fmaf(b[e], b[e], ss));
#pragma unroll
    for (int m = 1; m < L; m <<= 1) ss += __shfl_xor(ss, m, 64);
    if (h >= heads) continue;
    uint16_t* dst;
    if (h < n_heads) {
      const float r = rsqrtf(ss / (float)D + eps);
      if (part == 0) rstd[(int64_t)t * n_heads + h] = r;
      float oa[8], ob[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        a[e] = round_bf16(wa[e] * round_bf16(a[e] * r));
        b[e] = round_bf16(wb[e] * round_bf16(b[e] * r));
        oa[e] = round_bf16(a[e] * c[e]) + round_bf16(-b[e] * s[e]);
        ob[e] = round_bf16(b[e] * c[e]) + round_bf16(a[e] * s[e]);
      }
      ra[i] = pack8f(oa);
      rb[i] = pack8f(ob);
      dst = out + (int64_t)h * hs_out;
    } else {
      dst = pass + (int64_t)(h - n_heads) * hs_pass;
    }
    dst += (int64_t)t * D + d0;
    *reinterpret_cast<u32x4*>(dst) = ra[i];
    *reinterpret_cast<u32x4*>(dst + D / 2) = rb[i];
  }
}

// The way back: dtok from the head-major gradients (rotated back, then through the norm), and the gain's partial sums, one
// row of D per workgroup (slots as spx_rmsnorm_bwd_slots; accumulate: they start from what dw_part holds).
template <int D, int HEADS>
__global__ __launch_bounds__(256) void head_norm_rope_bwd_kernel(HeadSets sets, const float* __restrict__ inv_freq,
                                                                 int64_t pos_offset, float table_scale) {
  constexpr int L = D / 16, PER = 256 / L;
  const int which = (int)blockIdx.x >= sets.first;
  const spx_head_norm& in = sets.set[which];
  const uint16_t* __restrict__ const tok = reinterpret_cast<const uint16_t*>(in.tok);
  const uint16_t* __restrict__ const gain = reinterpret_cast<const uint16_t*>(in.gain);
  const uint16_t* __restrict__ const dout = reinterpret_cast<const uint16_t*>(in.out);
  const uint16_t* __restrict__ const dpass = reinterpret_cast<const uint16_t*>(in.pass);
  const float* __restrict__ const rstd = in.rstd;
  const int64_t* __restrict__ const pos = in.position_ids;
  uint16_t* __restrict__ const dtok = reinterpret_cast<uint16_t*>(in.dtok);
  float* __restrict__ const dw_part = in.dw_scratch;
  const int64_t ld = in.ld_tok, hs_out = in.out_head_stride, hs_pass = in.pass_head_stride, ld_d = in.ld_dtok;
  const int T = (int)in.T, n_heads = in.n_heads, n_pass = in.n_pass, accumulate = in.accumulate;
  const int block = (int)blockIdx.x - (which ? sets.first : 0), blocks = which ? (int)gridDim.x - sets.first : sets.first;
  __shared__ float red[PER * D];
  const int heads = n_heads + n_pass, groups = (heads + HEADS - 1) / HEADS;
  const int part = threadIdx.x % L, d0 = part * 8;
  const int64_t items = (int64_t)T * groups;
  float wa[8], wb[8], dwa[8], dwb[8];
  unpack8f(*reinterpret_cast<const u32x4*>(gain + d0), wa);
  unpack8f(*reinterpret_cast<const u32x4*>(gain + D / 2 + d0), wb);
#pragma unroll
  for (int e = 0; e < 8; ++e) dwa[e] = dwb[e] = 0.f;
  for (int64_t item = (int64_t)block * PER + threadIdx.x / L; item < items; item += (int64_t)blocks * PER) {
    const int hg = (int)(item % groups), t = (int)(item / groups);
    u32x4 ga[HEADS], gb[HEADS], xa[HEADS], xb[HEADS];
    float r[HEADS];
#pragma unroll
    for (int i = 0; i < HEADS; ++i) {
      const int h = i * groups + hg;
      ga[i] = gb[i] = xa[i] = xb[i] = u32x4{0, 0, 0, 0};
      r[i] = 0.f;
      if (h < heads) {
        const uint16_t* g = (h < n_heads ? dout + (int64_t)h * hs_out : dpass + (int64_t)(h - n_heads) * hs_pass) +
                            (int64_t)t * D + d0;
        ga[i] = *reinterpret_cast<const u32x4*>(g);
        gb[i] = *reinterpret_cast<const u32x4*>(g + D / 2);
        if (h < n_heads) {
          const uint16_t* x = tok + (int64_t)t * ld + h * D + d0;
          xa[i] = *reinterpret_cast<const u32x4*>(x);
          xb[i] = *reinterpret_cast<const u32x4*>(x + D / 2);
          r[i] = rstd[(int64_t)t * n_heads + h];
        }
      }
    }
    float c[8], s[8];
    if (hg < n_heads) {
      const float p = (float)(pos[t] + pos_offset);
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        float sn, cs;
        sincosf(p * inv_freq[d0 + e], &sn, &cs);
        c[e] = round_bf16(cs * table_scale);
        s[e] = -round_bf16(sn * table_scale);
      }
    }
#pragma unroll
    for (int i = 0; i < HEADS; ++i) {
      const int h = i * groups + hg;
      if (h < n_heads) {  // (uniform over the lanes of a head)
        float a[8], b[8], ha[8], hb[8], dot = 0.f;
        unpack8f(ga[i], a);
        unpack8f(gb[i], b);
        unpack8f(xa[i], ha);
        unpack8f(xb[i], hb);
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          // the gradient of the norm's output, as the separate kernel would have stored it
          const float da = round_bf16(round_bf16(a[e] * c[e]) + round_bf16(-b[e] * s[e]));
          const float db = round_bf16(round_bf16(b[e] * c[e]) + round_bf16(a[e] * s[e]));
          ha[e] *= r[i];
          hb[e] *= r[i];
          dwa[e] = fmaf(da, ha[e], dwa[e]);
          dwb[e] = fmaf(db, hb[e], dwb[e]);
          a[e] = da * wa[e];
          b[e] = db * wb[e];
          dot = fmaf(a[e], ha[e], fmaf(b[e], hb[e], dot));
        }
#pragma unroll
        for (int m = 1; m < L; m <<= 1) dot += __shfl_xor(dot, m, 64);
        const float mean = dot / (float)D;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          a[e] = r[i] * (a[e] - ha[e] * mean);
          b[e] = r[i] * (b[e] - hb[e] * mean);
        }
        ga[i] = pack8f(a);
        gb[i] = pack8f(b);
      }
      if (h < heads) {
        uint16_t* dst = dtok + (int64_t)t * ld_d + h * D + d0;
        *reinterpret_cast<u32x4*>(dst) = ga[i];
        *reinterpret_cast<u32x4*>(dst + D / 2) = gb[i];
      }
    }
  }
  if (!dw_part) return;
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    red[threadIdx.x / L * D + d0 + e] = dwa[e];
    red[threadIdx.x / L * D + D / 2 + d0 + e] = dwb[e];
  }
  __syncthreads();
  if (threadIdx.x < D) {
    float* const o = dw_part + (int64_t)block * D + threadIdx.x;
    float sum = accumulate ? *o : 0.f;
#pragma unroll
    for (int k = 0; k < PER; ++k) sum += red[k * D + threadIdx.x];
    *o = sum;
  }
}

// ---------------------------------------------------------------- weight staging
// Up to eight matrices, bf16 or fp32, one after the other as bf16: the merged compute weights of a forward (q, k
// and v; gate and up), and the bf16 copies of fp32 master weights, all of a layer's in one launch.  Bound by HBM; a thread has kCastAhead chunks of eight on
// their way before it stores the first.  ONCE: more than the 256 MB of the last-level cache is read and written, loads that
// nothing reads again leave it alone (gate and up of the 8B shape from fp32, 705 MB: 112 us, 128 without; two 8192 x 2048
// matrices, 201 MB: 37 us, 30 without).  q, k and v of the 1B shape from fp32: 21 us in three copies -> 12.  A workgroup
// whose chunks are of one part takes it in scalar registers and loads without conditions (two 8192 x 2048 from fp32 36.2 ->
// 31.6 us, 8192 x 8192 and two of 1024 rows 52.7 -> 49.8, 2048 x 2048 5.8 -> 5.2; bf16 sources the same); parts chosen by
// an index into the arguments: three times the time.
constexpr int kCastAhead = 4, kCastParts = 8;
struct CastArgs {
  const void* src[kCastParts];
  int64_t end[kCastParts];  // chunks of eight, running
  int f32;                  // bit i: src[i] is fp32
};
template <bool ONCE>
__global__ __launch_bounds__(256) void cat_bf16_kernel(CastArgs p, u32x4* __restrict__ out, int64_t n) {
  const int64_t first = (int64_t)blockIdx.x * kCastAhead * 256, last = min(first + kCastAhead * 256, n) - 1;
  const int64_t i0 = first + threadIdx.x;
  auto load = [](const u32x4* q) { return ONCE ? __builtin_nontemporal_load(q) : *q; };
  auto cast = [](u32x4 a, u32x4 b) {
    float v[8];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      v[e] = __uint_as_float(a[e]);
      v[4 + e] = __uint_as_float(b[e]);
    }
    return pack8f(v);
  };
  auto part_of = [&](int64_t i) {
    int s = 0;
#pragma unroll
    for (int k = 0; k < kCastParts - 1; ++k) s += i >= p.end[k];
    return s;
  };
  // (constant indices only: the arguments stay in scalar registers)
  auto pick = [&](int s, int64_t i) {
    const void* src = p.src[0];
    int64_t begin = 0;
#pragma unroll
    for (int k = 1; k < kCastParts; ++k) {
      src = s == k ? p.src[k] : src;
      begin = s == k ? p.end[k - 1] : begin;
    }
    return reinterpret_cast<const u32x4*>(src) + ((p.f32 >> s) & 1 ? 2 : 1) * (i - begin);
  };
  u32x4 lo[kCastAhead], hi[kCastAhead];
  const int s0 = part_of(first);
  if (first + kCastAhead * 256 <= n && part_of(last) == s0) {  // whole workgroups of one part: nearly all
    if ((p.f32 >> s0) & 1) {
      const u32x4* const src = pick(s0, first) + 2 * threadIdx.x;
#pragma unroll
      for (int u = 0; u < kCastAhead; ++u) {
        lo[u] = load(src + u * 512);
        hi[u] = load(src + u * 512 + 1);
      }
#pragma unroll
      for (int u = 0; u < kCastAhead; ++u) out[i0 + u * 256] = cast(lo[u], hi[u]);
    } else {
      const u32x4* const src = pick(s0, first) + threadIdx.x;
#pragma unroll
      for (int u = 0; u < kCastAhead; ++u) lo[u] = load(src + u * 256);
#pragma unroll
      for (int u = 0; u < kCastAhead; ++u) out[i0 + u * 256] = lo[u];
    }
    return;
  }
  bool wide[kCastAhead];
#pragma unroll
  for (int u = 0; u < kCastAhead; ++u) {
    const int64_t i = i0 + u * 256;
    lo[u] = hi[u] = u32x4{0, 0, 0, 0};
    wide[u] = false;
    if (i < n) {
      const int s = part_of(i);
      const u32x4* const src = pick(s, i);
      wide[u] = (p.f32 >> s) & 1;
      lo[u] = load(src);
      if (wide[u]) hi[u] = load(src + 1);
    }
  }
#pragma unroll
  for (int u = 0; u < kCastAhead; ++u) {
    const int64_t i = i0 + u * 256;
    if (i < n) out[i] = wide[u] ? cast(lo[u], hi[u]) : lo[u];
  }
}

// out[b][c][r] = in[b][r][c] for a stack of bf16 matrices (the per-expert transposes the input
// gradient products of a stack of expert weights need).  One wave = one 64 x 64 tile, one lane =
// one 8 x 8 block transposed in registers: every load and store instruction moves whole 128-byte
// row segments (8 lanes x 16 bytes) and no LDS is involved.
__global__ __launch_bounds__(256) void transpose_stack_kernel(const uint16_t* __restrict__ in, int64_t ld_in,
                                                              int64_t bs_in, uint16_t* __restrict__ out,
                                                              int64_t ld_out, int64_t bs_out, int R, int C,
                                                              int tiles_r, int tiles_c, int64_t n_tiles) {
  const int64_t tile = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (tile >= n_tiles) return;
  const int lane = threadIdx.x & 63;
  const int tc = (int)(tile % tiles_c);
  const int tr = (int)((tile / tiles_c) % tiles_r);
  const int64_t b = tile / ((int64_t)tiles_c * tiles_r);
  const int r0 = tr * 64 + (lane >> 3) * 8, c0 = tc * 64 + (lane & 7) * 8;
  if (r0 >= R || c0 >= C) return;  // R and C are multiples of 8: a block is inside or outside
  const uint16_t* src = in + b * bs_in + (int64_t)r0 * ld_in + c0;
  uint16_t* dst = out + b * bs_out + (int64_t)c0 * ld_out + r0;
  u32x4 v[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) v[i] = *reinterpret_cast<const u32x4*>(src + (int64_t)i * ld_in);
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    uint32_t o[4];
#pragma unroll
    for (int ip = 0; ip < 4; ++ip) {
      const uint32_t a = v[2 * ip][j >> 1], c = v[2 * ip + 1][j >> 1];
      o[ip] = (j & 1) ? ((a >> 16) | (c & 0xffff0000u)) : ((a & 0xffffu) | (c << 16));
    }
    u32x4 w;
    w.x = o[0]; w.y = o[1]; w.z = o[2]; w.w = o[3];
    *reinterpret_cast<u32x4*>(dst + (int64_t)j * ld_out) = w;
  }
}

// Output gate of the gated attention (Qwen3-Next): y = bf16(o * bf16(sigmoid(gate))), every tensor
// [rows, heads, D] with a row stride and a head stride of its own (the gate is the second half of
// every head's 2 D columns of the widened q projection).  One thread: 8 consecutive elements.
__global__ __launch_bounds__(256) void sigmoid_gate_fwd_kernel(
    const uint16_t* __restrict__ o, int64_t ld_o, const uint16_t* __restrict__ gate, int64_t ld_g, int hs_g,
    uint16_t* __restrict__ y, int64_t ld_y, int64_t rows, int heads, int D) {
  const int per_head = D / 8;
  const int64_t item = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (item >= rows * heads * per_head) return;
  const int d0 = (int)(item % per_head) * 8;
  const int h = (int)((item / per_head) % heads);
  const int64_t r = item / ((int64_t)per_head * heads);
  float a[8], g[8], out[8];
  unpack8f(*reinterpret_cast<const u32x4*>(o + r * ld_o + h * D + d0), a);
  unpack8f(*reinterpret_cast<const u32x4*>(gate + r * ld_g + (int64_t)h * hs_g + d0), g);
#pragma unroll
  for (int e = 0; e < 8; ++e) out[e] = a[e] * round_bf16(1.f / (1.f + __expf(-g[e])));
  *reinterpret_cast<u32x4*>(y + r * ld_y + h * D + d0) = pack8f(out);
}

// do = bf16(dy * sig), dgate = bf16(dy * o * sig * (1 - sig)), sig = sigmoid(gate) in fp32
__global__ __launch_bounds__(256) void sigmoid_gate_bwd_kernel(
    const uint16_t* __restrict__ o, int64_t ld_o, const uint16_t* __restrict__ gate, int64_t ld_g, int hs_g,
    const uint16_t* __restrict__ dy, int64_t ld_dy, uint16_t* __restrict__ d_o, int64_t ld_do,
    uint16_t* __restrict__ dgate, int64_t ld_dg, int hs_dg, int64_t rows, int heads, int D) {
  const int per_head = D / 8;
  const int64_t item = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (item >= rows * heads * per_head) return;
  const int d0 = (int)(item % per_head) * 8;
  const int h = (int)((item / per_head) % heads);
  const int64_t r = item / ((int64_t)per_head * heads);
  float a[8], g[8], d[8], oa[8], og[8];
  unpack8f(*reinterpret_cast<const u32x4*>(o + r * ld_o + h * D + d0), a);
  unpack8f(*reinterpret_cast<const u32x4*>(gate + r * ld_g + (int64_t)h * hs_g + d0), g);
  unpack8f(*reinterpret_cast<const u32x4*>(dy + r * ld_dy + h * D + d0), d);
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const float sg = 1.f / (1.f + __expf(-g[e]));
    oa[e] = d[e] * sg;
    og[e] = d[e] * a[e] * sg * (1.f - sg);
  }
  *reinterpret_cast<u32x4*>(d_o + r * ld_do + h * D + d0) = pack8f(oa);
  *reinterpret_cast<u32x4*>(dgate + r * ld_dg + (int64_t)h * hs_dg + d0) = pack8f(og);
}

// ---------------------------------------------------------------- SwiGLU
// rows x F elements per tensor, every tensor with its own row stride (so gate and up may be the
// two column halves of one merged projection output); chunk = 8 consecutive elements of a row
__global__ __launch_bounds__(256) void swiglu_fwd_kernel(const uint16_t* __restrict__ g, int64_t ld_g,
                                                         const uint16_t* __restrict__ u, int64_t ld_u,
                                                         uint16_t* __restrict__ out, int64_t ld_o,
                                                         int64_t rows, int64_t f8) {
  const int64_t n8 = rows * f8;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n8; i += (int64_t)gridDim.x * 256) {
    const int64_t r = i / f8, c = (i - r * f8) * 8;
    float gv[8], uv[8], o[8];
    unpack8f(*reinterpret_cast<const u32x4*>(g + r * ld_g + c), gv);
    unpack8f(*reinterpret_cast<const u32x4*>(u + r * ld_u + c), uv);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float sg = 1.f / (1.f + __expf(-gv[e]));
      o[e] = round_bf16(gv[e] * sg) * uv[e];
    }
    *reinterpret_cast<u32x4*>(out + r * ld_o + c) = pack8f(o);
  }
}

__global__ __launch_bounds__(256) void swiglu_bwd_kernel(const uint16_t* __restrict__ g, int64_t ld_g,
                                                         const uint16_t* __restrict__ u, int64_t ld_u,
                                                         const uint16_t* __restrict__ dout, int64_t ld_d,
                                                         uint16_t* __restrict__ dg, int64_t ld_dg,
                                                         uint16_t* __restrict__ du, int64_t ld_du,
                                                         int64_t rows, int64_t f8) {
  const int64_t n8 = rows * f8;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n8; i += (int64_t)gridDim.x * 256) {
    const int64_t r = i / f8, c = (i - r * f8) * 8;
    float gv[8], uv[8], dv[8], og[8], ou[8];
    unpack8f(*reinterpret_cast<const u32x4*>(g + r * ld_g + c), gv);
    unpack8f(*reinterpret_cast<const u32x4*>(u + r * ld_u + c), uv);
    unpack8f(*reinterpret_cast<const u32x4*>(dout + r * ld_d + c), dv);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float sg = 1.f / (1.f + __expf(-gv[e]));
      const float act = gv[e] * sg;
      ou[e] = dv[e] * act;
      og[e] = dv[e] * uv[e] * (sg * (1.f + gv[e] * (1.f - sg)));
    }
    *reinterpret_cast<u32x4*>(dg + r * ld_dg + c) = pack8f(og);
    *reinterpret_cast<u32x4*>(du + r * ld_du + c) = pack8f(ou);
  }
}

static bool al16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

// ---- packed rows: map of the live rows, and back to one row per position
// A row is live where row_grad[r] != 0 and, with labels, labels[r] != ignore_index.
__global__ __launch_bounds__(1024) void pack_row_map_kernel(const float* __restrict__ row_grad,
                                                            const int64_t* __restrict__ labels,
                                                            int64_t ignore_index, int rows,
                                                            int32_t* __restrict__ row_map,
                                                            int32_t* __restrict__ count) {
  pack_row_map([&](int r) { return row_grad[r] != 0.f && (!labels || labels[r] != ignore_index); }, rows, row_map,
               count);
}

// out[r, :] = row_map[r] >= 0 ? packed[row_map[r], :] : 0 for r < rows, 0 for rows <= r < total_rows;
// with row_scale every live row is multiplied by row_scale[r] on its way (fp32, one rounding) -- and with
// scale by row_scale[r] * (*scale * factor)
__global__ __launch_bounds__(256) void unpack_rows_kernel(const uint16_t* __restrict__ packed, int64_t ld,
                                                          const int32_t* __restrict__ row_map, int rows,
                                                          int cols8, uint16_t* __restrict__ out,
                                                          int64_t ld_out,
                                                          const float* __restrict__ row_scale = nullptr,
                                                          const float* __restrict__ scale = nullptr,
                                                          float factor = 1.f) {
  const int r = blockIdx.x;
  const int src = r < rows ? row_map[r] : -1;
  u32x4* o = reinterpret_cast<u32x4*>(out + (int64_t)r * ld_out);
  if (src < 0) {
    const u32x4 z = {0, 0, 0, 0};
    for (int c = threadIdx.x; c < cols8; c += 256) o[c] = z;
    return;
  }
  const u32x4* in = reinterpret_cast<const u32x4*>(packed + (int64_t)src * ld);
  if (!row_scale) {
    for (int c = threadIdx.x; c < cols8; c += 256) o[c] = in[c];
    return;
  }
  const float f = scale ? row_scale[r] * (*scale * factor) : row_scale[r];
  for (int c = threadIdx.x; c < cols8; c += 256) {
    const u32x4 v = in[c];
    u32x4 w;
    w.x = pack_bf16x2(bf16_lo(v.x) * f, bf16_hi(v.x) * f);
    w.y = pack_bf16x2(bf16_lo(v.y) * f, bf16_hi(v.y) * f);
    w.z = pack_bf16x2(bf16_lo(v.z) * f, bf16_hi(v.z) * f);
    w.w = pack_bf16x2(bf16_lo(v.w) * f, bf16_hi(v.w) * f);
    o[c] = w;
  }
}

}  // namespace spx

using namespace spx;

#define SPX_REQ_FN(cond, what) do { if (!(cond)) return spx::fail_arg(fn, what); } while (0)

extern "C" int spx_pack_row_map(const float* row_grad, const int64_t* labels, int64_t ignore_index,
                                int64_t rows, int32_t* row_map, int32_t* count, void* stream) {
  SPX_REQUIRE(rows > 0 && rows < (1ll << 31), "rows out of range");
  SPX_REQUIRE(row_grad && row_map && count, "null buffer");
  hipLaunchKernelGGL(pack_row_map_kernel, dim3(1), dim3(1024), 0, reinterpret_cast<hipStream_t>(stream), row_grad,
                     labels, ignore_index, (int)rows, row_map, count);
  return check_launch(__func__);
}

extern "C" int spx_unpack_rows(const void* packed, int64_t ld_packed, const int32_t* row_map, int64_t rows,
                               int64_t total_rows, int64_t cols, void* out, int64_t ld_out, void* stream) {
  SPX_REQUIRE(rows > 0 && total_rows >= rows && total_rows < (1ll << 31), "rows out of range");
  SPX_REQUIRE(cols > 0 && cols % 8 == 0 && ld_packed % 8 == 0 && ld_out % 8 == 0 && ld_packed >= cols && ld_out >= cols,
              "cols and the row strides must be multiples of 8 (bf16), strides at least cols");
  SPX_REQUIRE(packed && row_map && out, "null buffer");
  SPX_REQUIRE(al16(packed) && al16(out), "buffers must be 16-byte aligned");
  hipLaunchKernelGGL(unpack_rows_kernel, dim3((unsigned)total_rows), dim3(256), 0,
                     reinterpret_cast<hipStream_t>(stream), reinterpret_cast<const uint16_t*>(packed), ld_packed,
                     row_map, (int)rows, (int)(cols / 8), reinterpret_cast<uint16_t*>(out), ld_out);
  return check_launch(__func__);
}

extern "C" int spx_unpack_rows_graded(const void* packed, int64_t ld_packed, const int32_t* row_map,
                                      const float* row_scale, const float* scale, float factor, int64_t rows,
                                      int64_t total_rows, int64_t cols, void* out, int64_t ld_out, void* stream) {
  SPX_REQUIRE(rows > 0 && total_rows >= rows && total_rows < (1ll << 31), "rows out of range");
  SPX_REQUIRE(cols > 0 && cols % 8 == 0 && ld_packed % 8 == 0 && ld_out % 8 == 0 && ld_packed >= cols && ld_out >= cols,
              "cols and the row strides must be multiples of 8 (bf16), strides at least cols");
  SPX_REQUIRE(packed && row_map && row_scale && out, "null buffer");
  SPX_REQUIRE(al16(packed) && al16(out), "buffers must be 16-byte aligned");
  hipLaunchKernelGGL(unpack_rows_kernel, dim3((unsigned)total_rows), dim3(256), 0,
                     reinterpret_cast<hipStream_t>(stream), reinterpret_cast<const uint16_t*>(packed), ld_packed,
                     row_map, (int)rows, (int)(cols / 8), reinterpret_cast<uint16_t*>(out), ld_out, row_scale, scale,
                     factor);
  return check_launch(__func__);
}

extern "C" int spx_unpack_rows_scaled(const void* packed, int64_t ld_packed, const int32_t* row_map,
                                      const float* row_scale, int64_t rows, int64_t total_rows, int64_t cols,
                                      void* out, int64_t ld_out, void* stream) {
  return spx_unpack_rows_graded(packed, ld_packed, row_map, row_scale, nullptr, 1.f, rows, total_rows, cols, out,
                                ld_out, stream);
}

// one slot per workgroup, four workgroups per compute unit (narrow rows: one row per wave, eight)
extern "C" int64_t spx_rmsnorm_bwd_slots(int64_t rows, int64_t H) {
  if (H <= 512) return rows < 8192 ? (rows + 3) / 4 : 2048;
  return rows < 1024 ? rows : 1024;
}

// Threads per row: a lane keeps at most two chunks of 8 elements (see rmsnorm_bwd_kernel)
#define SPX_NORM_FORMS(LAUNCH)                      \
  do {                                              \
    if (H <= 512) LAUNCH(1, true, 256);             \
    else if (H <= 2048) LAUNCH(1, false, 256);      \
    else if (H <= 4096) LAUNCH(2, false, 256);      \
    else if (H <= 8192) LAUNCH(2, false, 512);      \
    else LAUNCH(2, false, 1024);                    \
  } while (0)

static int rmsnorm_fwd_launch(const char* fn, const void* x, int64_t ld_x, const void* res, int64_t ld_res,
                              void* sum, int64_t ld_sum, const void* weight, void* y, int64_t ld_y,
                              float* rstd, int64_t rows, int64_t H, float eps, void* stream,
                              const NormParts& parts = NormParts{}) {
  if (!(rows >= 0 && H > 0)) return fail_arg(fn, "bad sizes");
  if (!(H % 8 == 0 && ld_x % 8 == 0 && ld_y % 8 == 0 && ld_res % 8 == 0 && ld_sum % 8 == 0))
    return fail_arg(fn, "H and the row strides must be multiples of 8");
  if (H > 16384) return fail_arg(fn, "H must be at most 16384");
  if (rows >= (1ll << 31)) return fail_arg(fn, "too many rows");
  if (rows == 0) return SPX_OK;
  if (!(x && weight && y)) return fail_arg(fn, "null buffer");
  if (!(al16(x) && al16(weight) && al16(y) && al16(res) && al16(sum)))
    return fail_arg(fn, "buffers must be 16-byte aligned");
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  auto rp = reinterpret_cast<const uint16_t*>(res);
  auto sp = reinterpret_cast<uint16_t*>(sum);
  const NormFwdSet set = {reinterpret_cast<const uint16_t*>(x), ld_x, reinterpret_cast<const uint16_t*>(weight),
                          reinterpret_cast<uint16_t*>(y), ld_y, rstd};
#define SPX_LAUNCH(MAXC, WR, NT)                                                                             \
  do {                                                                                                       \
    const unsigned grid = (unsigned)(WR ? (rows + 3) / 4 : rows);                                            \
    if (parts.count)                                                                                         \
      hipLaunchKernelGGL((rmsnorm_fwd_kernel<MAXC, WR, true, false, NT, true>), dim3(grid), dim3(NT), 0, st, \
                         set, set, rows, (int)H, eps, nullptr, 0, sp, ld_sum, parts);                        \
    else if (res)                                                                                            \
      hipLaunchKernelGGL((rmsnorm_fwd_kernel<MAXC, WR, true, false, NT>), dim3(grid), dim3(NT), 0, st, set,  \
                         set, rows, (int)H, eps, rp, ld_res, sp, ld_sum, parts);                             \
    else                                                                                                     \
      hipLaunchKernelGGL((rmsnorm_fwd_kernel<MAXC, WR, false, false, NT>), dim3(grid), dim3(NT), 0, st, set, \
                         set, rows, (int)H, eps, nullptr, 0, nullptr, 0, parts);                             \
  } while (0)
  SPX_NORM_FORMS(SPX_LAUNCH);
#undef SPX_LAUNCH
  return check_launch(fn);
}

extern "C" int spx_rmsnorm_fwd(const void* x, int64_t ld_x, const void* weight, void* y, int64_t ld_y,
                               float* rstd, int64_t rows, int64_t H, float eps, void* stream) {
  return rmsnorm_fwd_launch(__func__, x, ld_x, nullptr, 0, nullptr, 0, weight, y, ld_y, rstd, rows, H, eps,
                            stream);
}

extern "C" int spx_add_rmsnorm_fwd(const void* a, int64_t ld_a, const void* b, int64_t ld_b, void* sum,
                                   int64_t ld_sum, const void* weight, void* y, int64_t ld_y, float* rstd,
                                   int64_t rows, int64_t H, float eps, void* stream) {
  SPX_REQUIRE(rows == 0 || (b && sum), "null buffer");
  return rmsnorm_fwd_launch(__func__, a, ld_a, b, ld_b, sum, ld_sum, weight, y, ld_y, rstd, rows, H, eps,
                            stream);
}

// the rules of partial results in place of a bf16 tensor of rows of H
static int parts_check(const char* fn, const float* partial, int32_t parts, int64_t rows, int64_t H) {
  if (!(partial && al16(partial) && parts >= 1)) return fail_arg(fn, "null or unaligned partial results");
  if (!(rows > 0 && H > 0 && H % 8 == 0)) return fail_arg(fn, "rows > 0 and H a multiple of 8");
  return SPX_OK;
}

extern "C" int spx_add_rmsnorm_fwd_parts(const void* a, int64_t ld_a, const float* partial, int32_t parts, void* sum,
                                         int64_t ld_sum, const void* weight, void* y, int64_t ld_y, float* rstd,
                                         int64_t rows, int64_t H, float eps, void* stream) {
  if (int rc = parts_check(__func__, partial, parts, rows, H)) return rc;
  SPX_REQUIRE(sum, "null buffer");
  return rmsnorm_fwd_launch(__func__, a, ld_a, nullptr, 0, sum, ld_sum, weight, y, ld_y, rstd, rows, H, eps, stream,
                            NormParts{partial, rows * H, parts});
}

extern "C" int spx_rmsnorm_pair_fwd(const void* a, int64_t ld_a, const void* weight_a, const void* b, int64_t ld_b,
                                    const void* weight_b, void* y, int64_t ld_y, float* rstd, int64_t rows,
                                    int64_t H, float eps, void* stream) {
  SPX_REQUIRE(rows > 0 && rows < (1ll << 31) && H > 0 && H % 8 == 0 && H <= 16384,
              "rows > 0 and H a multiple of 8, at most 16384");
  SPX_REQUIRE(ld_a % 8 == 0 && ld_b % 8 == 0 && ld_y % 8 == 0 && ld_y >= 2 * H,
              "the row strides must be multiples of 8, that of y at least 2 H");
  SPX_REQUIRE(a && weight_a && b && weight_b && y && rstd, "null buffer");
  SPX_REQUIRE(al16(a) && al16(weight_a) && al16(b) && al16(weight_b) && al16(y), "buffers must be 16-byte aligned");
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  uint16_t* yp = reinterpret_cast<uint16_t*>(y);
  const NormFwdSet one = {reinterpret_cast<const uint16_t*>(a), ld_a, reinterpret_cast<const uint16_t*>(weight_a),
                          yp, ld_y, rstd};
  const NormFwdSet two = {reinterpret_cast<const uint16_t*>(b), ld_b, reinterpret_cast<const uint16_t*>(weight_b),
                          yp + H, ld_y, rstd + rows};
#define SPX_LAUNCH(MAXC, WR, NT)                                                                                 \
  hipLaunchKernelGGL((rmsnorm_fwd_kernel<MAXC, WR, false, true, NT>), dim3((unsigned)(WR ? (rows + 3) / 4 : rows), 2), \
                     dim3(NT), 0, st, one, two, rows, (int)H, eps, nullptr, 0, nullptr, 0, NormParts{})
  SPX_NORM_FORMS(SPX_LAUNCH);
#undef SPX_LAUNCH
  return check_launch(__func__);
}

static int rmsnorm_bwd_launch(const char* fn, const void* x, int64_t ld_x, const void* weight, const void* dy,
                              int64_t ld_dy, const void* dres, int64_t ld_dres, const float* rstd, void* dx,
                              int64_t ld_dx, void* dweight, float* dw_scratch, int64_t rows, int64_t H,
                              void* stream, bool partial_only = false, int accumulate = 0,
                              const NormParts& parts = NormParts{}) {
  if (!(rows > 0 && H > 0)) return fail_arg(fn, "bad sizes");
  if (!(H % 8 == 0 && ld_x % 8 == 0 && ld_dy % 8 == 0 && ld_dx % 8 == 0 && ld_dres % 8 == 0))
    return fail_arg(fn, "H and the row strides must be multiples of 8");
  if (H > 16384) return fail_arg(fn, "H must be at most 16384");
  if (!(x && weight && (dy || parts.count) && rstd)) return fail_arg(fn, "null buffer");
  if (!(dx || dweight || partial_only)) return fail_arg(fn, "neither dx nor dweight requested");
  if (partial_only && !dw_scratch) return fail_arg(fn, "null dw_scratch");
  if (dres && !dx) return fail_arg(fn, "a residual gradient needs dx");
  if (dweight && !dw_scratch)
    return fail_arg(fn, "dweight needs dw_scratch (spx_rmsnorm_bwd_slots(rows, H) * H floats)");
  if (!(al16(x) && al16(weight) && al16(dy) && al16(dx) && al16(dw_scratch) && al16(dres)))
    return fail_arg(fn, "buffers must be 16-byte aligned");
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  float* part = (dweight || partial_only) ? dw_scratch : nullptr;
  const NormBwdSet set = {reinterpret_cast<const uint16_t*>(x), ld_x, reinterpret_cast<const uint16_t*>(weight),
                          reinterpret_cast<const uint16_t*>(dy), ld_dy, rstd, reinterpret_cast<uint16_t*>(dx), ld_dx,
                          part, reinterpret_cast<const uint16_t*>(dres), ld_dres, accumulate};
  const int64_t slots = spx_rmsnorm_bwd_slots(rows, H);
#define SPX_LAUNCH(MAXC, WR, NT)                                                                                         \
  do {                                                                                                                   \
    if (parts.count)                                                                                                     \
      hipLaunchKernelGGL((rmsnorm_bwd_kernel<MAXC, WR, false, NT, true>), dim3((unsigned)slots), dim3(NT), 0, st, set,   \
                         set, rows, (int)H, parts);                                                                      \
    else                                                                                                                 \
      hipLaunchKernelGGL((rmsnorm_bwd_kernel<MAXC, WR, false, NT>), dim3((unsigned)slots), dim3(NT), 0, st, set, set,    \
                         rows, (int)H, parts);                                                                           \
  } while (0)
  SPX_NORM_FORMS(SPX_LAUNCH);
#undef SPX_LAUNCH
  if (dweight)
    launch_sums(one_sum(part, slots, H, dweight), 1, st);
  return check_launch(fn);
}

extern "C" int spx_rmsnorm_pair_bwd_partial(const void* a, int64_t ld_a, const void* weight_a, const void* b,
                                            int64_t ld_b, const void* weight_b, const void* dy, int64_t ld_dy,
                                            const void* dres_b, int64_t ld_dres, const float* rstd, void* da,
                                            void* db, int64_t ld_dx, float* scratch_a, int32_t accumulate_a,
                                            float* scratch_b, int32_t accumulate_b, int64_t rows, int64_t H,
                                            void* stream) {
  SPX_REQUIRE(rows > 0 && H > 0 && H % 8 == 0 && H <= 16384, "rows > 0 and H a multiple of 8, at most 16384");
  SPX_REQUIRE(ld_a % 8 == 0 && ld_b % 8 == 0 && ld_dy % 8 == 0 && ld_dy >= 2 * H && ld_dres % 8 == 0 &&
                  ld_dx % 8 == 0, "the row strides must be multiples of 8, that of dy at least 2 H");
  SPX_REQUIRE(a && weight_a && b && weight_b && dy && rstd && scratch_a && scratch_b, "null buffer");
  SPX_REQUIRE(!dres_b || db, "a residual gradient needs db");
  SPX_REQUIRE(al16(a) && al16(weight_a) && al16(b) && al16(weight_b) && al16(dy) && al16(dres_b) && al16(da) &&
                  al16(db) && al16(scratch_a) && al16(scratch_b), "buffers must be 16-byte aligned");
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  const uint16_t* dyp = reinterpret_cast<const uint16_t*>(dy);
  const NormBwdSet one = {reinterpret_cast<const uint16_t*>(a), ld_a, reinterpret_cast<const uint16_t*>(weight_a), dyp,
                          ld_dy, rstd, reinterpret_cast<uint16_t*>(da), ld_dx, scratch_a, nullptr, 0,
                          accumulate_a != 0};
  const NormBwdSet two = {reinterpret_cast<const uint16_t*>(b), ld_b, reinterpret_cast<const uint16_t*>(weight_b),
                          dyp + H, ld_dy, rstd + rows, reinterpret_cast<uint16_t*>(db), ld_dx, scratch_b,
                          reinterpret_cast<const uint16_t*>(dres_b), ld_dres, accumulate_b != 0};
  const int64_t slots = spx_rmsnorm_bwd_slots(rows, H);
#define SPX_LAUNCH(MAXC, WR, NT)                                                                                      \
  hipLaunchKernelGGL((rmsnorm_bwd_kernel<MAXC, WR, true, NT>), dim3((unsigned)slots, 2), dim3(NT), 0, st, one, two, \
                     rows, (int)H, NormParts{})
  SPX_NORM_FORMS(SPX_LAUNCH);
#undef SPX_LAUNCH
  return check_launch(__func__);
}

extern "C" int spx_rmsnorm_bwd(const void* x, int64_t ld_x, const void* weight, const void* dy,
                               int64_t ld_dy, const float* rstd, void* dx, int64_t ld_dx, void* dweight,
                               float* dw_scratch, int64_t rows, int64_t H, void* stream) {
  return rmsnorm_bwd_launch(__func__, x, ld_x, weight, dy, ld_dy, nullptr, 0, rstd, dx, ld_dx, dweight,
                            dw_scratch, rows, H, stream);
}

extern "C" int spx_add_rmsnorm_bwd(const void* x, int64_t ld_x, const void* weight, const void* dy,
                                   int64_t ld_dy, const void* dres, int64_t ld_dres, const float* rstd,
                                   void* dx, int64_t ld_dx, void* dweight, float* dw_scratch, int64_t rows,
                                   int64_t H, void* stream) {
  return rmsnorm_bwd_launch(__func__, x, ld_x, weight, dy, ld_dy, dres, ld_dres, rstd, dx, ld_dx, dweight,
                            dw_scratch, rows, H, stream);
}

extern "C" int spx_rmsnorm_bwd_partial(const void* x, int64_t ld_x, const void* weight, const void* dy,
                                       int64_t ld_dy, const void* dres, int64_t ld_dres, const float* rstd,
                                       void* dx, int64_t ld_dx, float* dw_scratch, int32_t accumulate,
                                       int64_t rows, int64_t H, void* stream) {
  return rmsnorm_bwd_launch(__func__, x, ld_x, weight, dy, ld_dy, dres, ld_dres, rstd, dx, ld_dx, nullptr,
                            dw_scratch, rows, H, stream, true, accumulate != 0);
}

extern "C" int spx_rmsnorm_bwd_parts(const void* x, int64_t ld_x, const void* weight, const float* partial, int32_t parts,
                                     const void* dres, int64_t ld_dres, const float* rstd, void* dx, int64_t ld_dx,
                                     float* dw_scratch, int32_t accumulate, int64_t rows, int64_t H, void* stream) {
  if (int rc = parts_check(__func__, partial, parts, rows, H)) return rc;
  return rmsnorm_bwd_launch(__func__, x, ld_x, weight, nullptr, 0, dres, ld_dres, rstd, dx, ld_dx, nullptr, dw_scratch, rows,
                            H, stream, dw_scratch != nullptr, accumulate != 0, NormParts{partial, rows * H, parts});
}

extern "C" int spx_rmsnorm_dweight(const float* dw_scratch, int64_t slots, int64_t H, void* dweight,
                                   void* stream) {
  const char* fn = __func__;
  if (!(slots > 0 && H > 0 && H % 8 == 0 && H <= 16384)) return fail_arg(fn, "bad sizes");
  if (!(dw_scratch && dweight && al16(dw_scratch))) return fail_arg(fn, "null or unaligned buffer");
  if (slots >= (1ll << 31)) return fail_arg(fn, "bad sizes");
  launch_sums(one_sum(dw_scratch, slots, H, dweight), 1, reinterpret_cast<hipStream_t>(stream));
  return check_launch(fn);
}

extern "C" int spx_rmsnorm_dweights(const float* const* dw_scratch, const int64_t* slots, const int64_t* H,
                                    void* const* dweight, const int32_t* is_f32, int32_t count, void* stream) {
  const char* fn = __func__;
  SPX_REQ_FN(dw_scratch && slots && H && dweight && is_f32 && count >= 1 && count <= kSumSets, "one to sixteen gains");
  SumSets p{};
  int end = 0;
  for (int i = 0; i < count; ++i) {
    SPX_REQ_FN(slots[i] > 0 && slots[i] < (1ll << 31) && H[i] > 0 && H[i] % 8 == 0 && H[i] <= 16384, "bad sizes");
    SPX_REQ_FN(dw_scratch[i] && dweight[i] && al16(dw_scratch[i]), "null or unaligned buffer");
    end += (int)((H[i] + 31) / 32);
    p.part[i] = dw_scratch[i]; p.out[i] = dweight[i]; p.slots[i] = (int)slots[i]; p.H[i] = (int)H[i]; p.end[i] = end;
    p.f32 |= (is_f32[i] ? 1u : 0u) << i;
  }
  launch_sums(p, count, reinterpret_cast<hipStream_t>(stream));
  return check_launch(fn);
}

static int rope_relayout_impl(const char* fn, const void* x, int64_t ld_x, const int64_t* position_ids,
                              const float* inv_freq, void* out, int64_t ld_out, int64_t T, int32_t heads,
                              int32_t D, int32_t rotate, int32_t inverse, int64_t position_offset,
                              int32_t tok_head_stride, int32_t rot, float table_scale, void* stream);

extern "C" int spx_rope_relayout(const void* x, int64_t ld_x, const int64_t* position_ids,
                                 const float* inv_freq, void* out, int64_t ld_out, int64_t T,
                                 int32_t heads, int32_t D, int32_t rotate, int32_t inverse,
                                 int64_t position_offset, void* stream) {
  return rope_relayout_impl(__func__, x, ld_x, position_ids, inv_freq, out, ld_out, T, heads, D, rotate,
                            inverse, position_offset, D, D, 1.f, stream);
}

extern "C" int spx_rope_relayout_partial(const void* x, int64_t ld_x, int32_t x_head_stride,
                                         const int64_t* position_ids, const float* inv_freq, void* out,
                                         int64_t ld_out, int64_t T, int32_t heads, int32_t D,
                                         int32_t rotary_dim, int32_t rotate, int32_t inverse,
                                         int64_t position_offset, float table_scale, void* stream) {
  return rope_relayout_impl(__func__, x, ld_x, position_ids, inv_freq, out, ld_out, T, heads, D, rotate,
                            inverse, position_offset, x_head_stride, rotary_dim, table_scale, stream);
}

extern "C" int spx_transpose_bf16(const void* in, int64_t ld_in, int64_t batch_stride_in, void* out,
                                  int64_t ld_out, int64_t batch_stride_out, int64_t R, int64_t C,
                                  int64_t batches, void* stream) {
  const char* fn = __func__;
  SPX_REQ_FN(R > 0 && C > 0 && batches > 0 && R % 8 == 0 && C % 8 == 0 && R < (1ll << 31) && C < (1ll << 31),
             "R and C must be positive multiples of 8");
  SPX_REQ_FN(in && out && in != out && al16(in) && al16(out), "null, aliased or unaligned buffer");
  SPX_REQ_FN(ld_in % 8 == 0 && ld_out % 8 == 0 && ld_in >= C && ld_out >= R, "row strides must be multiples of 8, ld_in >= C, ld_out >= R");
  SPX_REQ_FN(batch_stride_in % 8 == 0 && batch_stride_out % 8 == 0 && batch_stride_in >= 0 && batch_stride_out >= 0,
             "batch strides must be multiples of 8");
  const int tiles_r = (int)((R + 63) / 64), tiles_c = (int)((C + 63) / 64);
  const int64_t n_tiles = (int64_t)tiles_r * tiles_c * batches;
  SPX_REQ_FN((n_tiles + 3) / 4 < (1ll << 31), "too many tiles");
  hipLaunchKernelGGL(transpose_stack_kernel, dim3((unsigned)((n_tiles + 3) / 4)), dim3(256), 0,
                     reinterpret_cast<hipStream_t>(stream), reinterpret_cast<const uint16_t*>(in), ld_in,
                     batch_stride_in, reinterpret_cast<uint16_t*>(out), ld_out, batch_stride_out, (int)R, (int)C,
                     tiles_r, tiles_c, n_tiles);
  return check_launch(fn);
}

extern "C" int spx_sigmoid_gate_fwd(const void* o, int64_t ld_o, const void* gate, int64_t ld_gate,
                                    int32_t gate_head_stride, void* y, int64_t ld_y, int64_t rows,
                                    int32_t heads, int32_t D, void* stream) {
  const char* fn = __func__;
  SPX_REQ_FN(rows > 0 && heads > 0 && D > 0 && D % 8 == 0, "rows, heads > 0 and D a positive multiple of 8");
  SPX_REQ_FN(o && gate && y && al16(o) && al16(gate) && al16(y), "null or unaligned buffer");
  const int64_t hd = (int64_t)heads * D;
  SPX_REQ_FN(ld_o % 8 == 0 && ld_y % 8 == 0 && ld_gate % 8 == 0 && gate_head_stride % 8 == 0, "strides must be multiples of 8");
  SPX_REQ_FN(ld_o >= hd && ld_y >= hd && gate_head_stride >= D && ld_gate >= (int64_t)(heads - 1) * gate_head_stride + D,
             "stride too small");
  const int64_t items = rows * heads * (D / 8);
  hipLaunchKernelGGL(sigmoid_gate_fwd_kernel, dim3((unsigned)((items + 255) / 256)), dim3(256), 0,
                     reinterpret_cast<hipStream_t>(stream), reinterpret_cast<const uint16_t*>(o), ld_o,
                     reinterpret_cast<const uint16_t*>(gate), ld_gate, (int)gate_head_stride,
                     reinterpret_cast<uint16_t*>(y), ld_y, rows, (int)heads, (int)D);
  return check_launch(fn);
}

extern "C" int spx_sigmoid_gate_bwd(const void* o, int64_t ld_o, const void* gate, int64_t ld_gate,
                                    int32_t gate_head_stride, const void* dy, int64_t ld_dy, void* d_o,
                                    int64_t ld_do, void* dgate, int64_t ld_dgate,
                                    int32_t dgate_head_stride, int64_t rows, int32_t heads, int32_t D,
                                    void* stream) {
  const char* fn = __func__;
  SPX_REQ_FN(rows > 0 && heads > 0 && D > 0 && D % 8 == 0, "rows, heads > 0 and D a positive multiple of 8");
  SPX_REQ_FN(o && gate && dy && d_o && dgate, "null buffer");
  SPX_REQ_FN(al16(o) && al16(gate) && al16(dy) && al16(d_o) && al16(dgate), "buffers must be 16-byte aligned");
  const int64_t hd = (int64_t)heads * D;
  SPX_REQ_FN(ld_o % 8 == 0 && ld_dy % 8 == 0 && ld_do % 8 == 0 && ld_gate % 8 == 0 && ld_dgate % 8 == 0 &&
                 gate_head_stride % 8 == 0 && dgate_head_stride % 8 == 0, "strides must be multiples of 8");
  SPX_REQ_FN(ld_o >= hd && ld_dy >= hd && ld_do >= hd && gate_head_stride >= D && dgate_head_stride >= D &&
                 ld_gate >= (int64_t)(heads - 1) * gate_head_stride + D &&
                 ld_dgate >= (int64_t)(heads - 1) * dgate_head_stride + D, "stride too small");
  const int64_t items = rows * heads * (D / 8);
  hipLaunchKernelGGL(sigmoid_gate_bwd_kernel, dim3((unsigned)((items + 255) / 256)), dim3(256), 0,
                     reinterpret_cast<hipStream_t>(stream), reinterpret_cast<const uint16_t*>(o), ld_o,
                     reinterpret_cast<const uint16_t*>(gate), ld_gate, (int)gate_head_stride,
                     reinterpret_cast<const uint16_t*>(dy), ld_dy, reinterpret_cast<uint16_t*>(d_o), ld_do,
                     reinterpret_cast<uint16_t*>(dgate), ld_dgate, (int)dgate_head_stride, rows, (int)heads, (int)D);
  return check_launch(fn);
}

static int rope_relayout_impl(const char* fn, const void* x, int64_t ld_x, const int64_t* position_ids,
                              const float* inv_freq, void* out, int64_t ld_out, int64_t T, int32_t heads,
                              int32_t D, int32_t rotate, int32_t inverse, int64_t position_offset,
                              int32_t tok_head_stride, int32_t rot, float table_scale, void* stream) {
  SPX_REQ_FN(table_scale > 0.f && table_scale < 1e4f, "the table scale must be positive and finite");
  SPX_REQ_FN(T > 0 && heads > 0 && D > 0 && D % 16 == 0, "T, heads > 0 and D a multiple of 16");
  SPX_REQ_FN(rot > 0 && rot <= D && rot % 16 == 0, "the rotary dimension must be a multiple of 16 in 16 .. D");
  SPX_REQ_FN(tok_head_stride >= D && tok_head_stride % 8 == 0, "bad head stride of the token-major side");
  SPX_REQ_FN(x && out && (!rotate || (position_ids && inv_freq)), "null buffer");
  SPX_REQ_FN(al16(x) && al16(out), "buffers must be 16-byte aligned");
  const int64_t tok_row = (int64_t)(heads - 1) * tok_head_stride + D;
  if (inverse) {
    SPX_REQ_FN(ld_out % 8 == 0 && ld_out >= tok_row, "bad output row stride");
    SPX_REQ_FN(ld_x == 0 || (ld_x % 8 == 0 && ld_x >= T * D), "bad head stride of the head-major input");
  } else {
    SPX_REQ_FN(ld_x % 8 == 0 && ld_x >= tok_row, "bad input row stride");
    SPX_REQ_FN(ld_out == 0 || (ld_out % 8 == 0 && ld_out >= T * D), "bad head stride of the head-major output");
  }
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  const int64_t total = T * heads * (D / 16);
  const unsigned grid = (unsigned)((total + 255) / 256);
  auto xp = reinterpret_cast<const uint16_t*>(x);
  auto op = reinterpret_cast<uint16_t*>(out);
  if (inverse)
    hipLaunchKernelGGL(rope_kernel<true>, dim3(grid), dim3(256), 0, st, xp, ld_x, position_ids, inv_freq, op,
                       ld_out, (int)T, (int)heads, (int)D, (int)rotate, position_offset, (int)tok_head_stride, (int)rot,
                       table_scale);
  else
    hipLaunchKernelGGL(rope_kernel<false>, dim3(grid), dim3(256), 0, st, xp, ld_x, position_ids, inv_freq, op,
                       ld_out, (int)T, (int)heads, (int)D, (int)rotate, position_offset, (int)tok_head_stride, (int)rot,
                       table_scale);
  return check_launch(fn);
}

extern "C" int spx_rope_qkv(void* tok, int64_t ld_tok, void* q, int64_t q_head_stride, void* k,
                            int64_t k_head_stride, void* v, int64_t v_head_stride, const int64_t* position_ids,
                            const float* inv_freq, int64_t T, int32_t hq, int32_t hkv, int32_t D,
                            int32_t rotary_dim, int32_t inverse, int64_t position_offset, float table_scale,
                            void* stream) {
  const char* fn = __func__;
  SPX_REQ_FN(table_scale > 0.f && table_scale < 1e4f, "the table scale must be positive and finite");
  SPX_REQ_FN(T > 0 && hq > 0 && hkv > 0 && D > 0 && D % 16 == 0, "T, heads > 0 and D a multiple of 16");
  SPX_REQ_FN(rotary_dim > 0 && rotary_dim <= D && rotary_dim % 16 == 0,
             "the rotary dimension must be a multiple of 16 in 16 .. D");
  const int64_t heads = (int64_t)hq + 2 * (int64_t)hkv;
  SPX_REQ_FN(ld_tok % 8 == 0 && ld_tok >= heads * D, "bad row stride of the token-major side");
  SPX_REQ_FN(tok && position_ids && inv_freq && (inverse || (q && k && v)), "null buffer");
  SPX_REQ_FN(al16(tok) && al16(q) && al16(k) && al16(v), "buffers must be 16-byte aligned");
  const int64_t win = T * D;
  SPX_REQ_FN(q_head_stride % 8 == 0 && k_head_stride % 8 == 0 && v_head_stride % 8 == 0 &&
                 q_head_stride >= win && k_head_stride >= win && v_head_stride >= win,
             "head strides of the head-major sides must be multiples of 8, at least T * D");
  const int64_t items = T * heads * (D / 16);
  SPX_REQ_FN(items < (1ll << 31), "too many elements");
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  auto tp = reinterpret_cast<uint16_t*>(tok);
  auto qp = reinterpret_cast<uint16_t*>(q);
  auto kp = reinterpret_cast<uint16_t*>(k);
  auto vp = reinterpret_cast<uint16_t*>(v);
  // heads per thread: as many as leave every compute unit two workgroups
#define SPX_LAUNCH(HEADS)                                                                                           \
  do {                                                                                                              \
    const int64_t n = T * ((heads + HEADS - 1) / HEADS) * (D / 16);                                                 \
    const dim3 grid((unsigned)((n + 255) / 256));                                                                   \
    if (inverse)                                                                                                    \
      hipLaunchKernelGGL((rope_qkv_kernel<true, HEADS>), grid, dim3(256), 0, st, tp, ld_tok, qp, q_head_stride, kp, \
                         k_head_stride, vp, v_head_stride, position_ids, inv_freq, (int)T, (int)hq, (int)hkv,       \
                         (int)D, (int)rotary_dim, position_offset, table_scale);                                    \
    else                                                                                                            \
      hipLaunchKernelGGL((rope_qkv_kernel<false, HEADS>), grid, dim3(256), 0, st, tp, ld_tok, qp, q_head_stride,    \
                         kp, k_head_stride, vp, v_head_stride, position_ids, inv_freq, (int)T, (int)hq, (int)hkv,   \
                         (int)D, (int)rotary_dim, position_offset, table_scale);                                    \
  } while (0)
  if (items >= 4 * 512 * 256) SPX_LAUNCH(4);
  else if (items >= 2 * 512 * 256) SPX_LAUNCH(2);
  else SPX_LAUNCH(1);
#undef SPX_LAUNCH
  return check_launch(fn);
}

extern "C" int spx_cat_bf16(const void* const* srcs, const int64_t* elements, const int32_t* is_f32, int32_t count,
                            void* out, void* stream) {
  const char* fn = __func__;
  SPX_REQ_FN(srcs && elements && is_f32 && count >= 1 && count <= kCastParts, "one to eight matrices");
  SPX_REQ_FN(out && al16(out), "null or unaligned buffer");
  CastArgs p{};
  int64_t n = 0;
  for (int i = 0; i < kCastParts; ++i) {
    if (i < count) {
      SPX_REQ_FN(srcs[i] && al16(srcs[i]) && elements[i] > 0 && elements[i] % 8 == 0,
                 "null or unaligned matrix, or a size that is not a multiple of 8");
      n += elements[i] / 8;
      p.src[i] = srcs[i];
      p.f32 |= (is_f32[i] ? 1 : 0) << i;
    }
    p.end[i] = n;
  }
  SPX_REQ_FN(n < (1ll << 38), "too many elements");
  int64_t bytes = 0;
  for (int i = 0; i < count; ++i) bytes += elements[i] * (is_f32[i] ? 6 : 4);
  const dim3 grid((unsigned)((n + 256 * kCastAhead - 1) / (256 * kCastAhead)));
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  u32x4* const o = reinterpret_cast<u32x4*>(out);
  if (bytes > (256ll << 20)) hipLaunchKernelGGL(cat_bf16_kernel<true>, grid, dim3(256), 0, st, p, o, n);
  else hipLaunchKernelGGL(cat_bf16_kernel<false>, grid, dim3(256), 0, st, p, o, n);
  return check_launch(fn);
}

static unsigned swiglu_grid(int64_t n8) {
  return (unsigned)((n8 + 255) / 256 < 65536 ? (n8 + 255) / 256 : 65536);
}

static int head_norm_rope_checks(const char* fn, int64_t ld, int64_t T, int32_t n_heads, int32_t n_pass, int32_t D,
                                 int64_t hs, int64_t hs_pass, float table_scale) {
  SPX_REQ_FN(table_scale > 0.f && table_scale < 1e4f, "the table scale must be positive and finite");
  SPX_REQ_FN(T > 0 && n_heads > 0 && n_pass >= 0, "T and heads must be positive");
  SPX_REQ_FN(D == 64 || D == 128 || D == 256, "head_dim must be 64, 128 or 256");
  SPX_REQ_FN(ld % 8 == 0 && ld >= (int64_t)(n_heads + n_pass) * D, "bad row stride of the token-major side");
  SPX_REQ_FN(hs % 8 == 0 && hs >= T * D && (!n_pass || (hs_pass % 8 == 0 && hs_pass >= T * D)),
             "head strides must be multiples of 8, at least T * D");
  SPX_REQ_FN(T * (n_heads + n_pass) * (D / 16) < (1ll << 31), "too many elements");
  return SPX_OK;
}
// heads per thread: as many as leave every compute unit two workgroups
static int heads_per_thread(int64_t threads) { return threads >= 4 * 512 * 256 ? 4 : threads >= 2 * 512 * 256 ? 2 : 1; }

#define SPX_LAUNCH_D(HEADS)                                                                                           \
  do { if (D == 64) SPX_LAUNCH(64, HEADS); else if (D == 128) SPX_LAUNCH(128, HEADS); else SPX_LAUNCH(256, HEADS); } while (0)

static int head_norm_rope_launch(const char* fn, const spx_head_norm* sets, int32_t count, const float* inv_freq, int32_t D,
                                 int64_t position_offset, float table_scale, void* stream) {
  SPX_REQ_FN(sets && (count == 1 || count == 2) && inv_freq, "one or two sets of heads and their frequencies");
  HeadSets hs{};
  int64_t threads = 0;
  for (int i = 0; i < count; ++i) {
    const spx_head_norm& h = hs.set[i] = sets[i];
    if (int rc = head_norm_rope_checks(fn, h.ld_tok, h.T, h.n_heads, h.n_pass, D, h.out_head_stride, h.pass_head_stride,
                                       table_scale))
      return rc;
    SPX_REQ_FN(h.tok && h.out && h.position_ids && h.gain && h.rstd && (!h.n_pass || h.pass), "null buffer");
    SPX_REQ_FN(al16(h.tok) && al16(h.out) && al16(h.pass) && al16(h.gain), "buffers must be 16-byte aligned");
    threads += h.T * (h.n_heads + h.n_pass) * (D / 16);
  }
  const int per = heads_per_thread(threads);
  int64_t blocks = 0;
  for (int i = 0; i < count; ++i) {
    blocks += (hs.set[i].T * ((hs.set[i].n_heads + hs.set[i].n_pass + per - 1) / per) * (D / 16) + 255) / 256;
    if (i == 0) hs.first = (int)blocks;
  }
#define SPX_LAUNCH(DD, HEADS)                                                                                         \
  hipLaunchKernelGGL((head_norm_rope_kernel<DD, HEADS>), dim3((unsigned)blocks), dim3(256), 0,                        \
                     reinterpret_cast<hipStream_t>(stream), hs, inv_freq, position_offset, table_scale)
  if (per == 4) SPX_LAUNCH_D(4);
  else if (per == 2) SPX_LAUNCH_D(2);
  else SPX_LAUNCH_D(1);
#undef SPX_LAUNCH
  return check_launch(fn);
}

static int head_norm_rope_bwd_launch(const char* fn, const spx_head_norm* sets, int32_t count, const float* inv_freq,
                                     int32_t D, int64_t position_offset, float table_scale, void* stream) {
  SPX_REQ_FN(sets && (count == 1 || count == 2) && inv_freq, "one or two sets of heads and their frequencies");
  HeadSets hs{};
  int64_t threads = 0, blocks = 0;
  for (int i = 0; i < count; ++i) {
    const spx_head_norm& h = hs.set[i] = sets[i];
    if (int rc = head_norm_rope_checks(fn, h.ld_tok, h.T, h.n_heads, h.n_pass, D, h.out_head_stride, h.pass_head_stride,
                                       table_scale))
      return rc;
    SPX_REQ_FN(h.tok && h.out && h.position_ids && h.gain && h.rstd && h.dtok && (!h.n_pass || h.pass), "null buffer");
    SPX_REQ_FN(al16(h.tok) && al16(h.out) && al16(h.pass) && al16(h.gain) && al16(h.dtok), "buffers must be 16-byte aligned");
    SPX_REQ_FN(h.ld_dtok % 8 == 0 && h.ld_dtok >= (int64_t)(h.n_heads + h.n_pass) * D, "bad row stride of the gradient");
    threads += h.T * (h.n_heads + h.n_pass) * (D / 16);
    blocks += spx_rmsnorm_bwd_slots(h.T * h.n_heads, D);
    if (i == 0) hs.first = (int)blocks;
  }
  const int per = heads_per_thread(threads);
#define SPX_LAUNCH(DD, HEADS)                                                                                         \
  hipLaunchKernelGGL((head_norm_rope_bwd_kernel<DD, HEADS>), dim3((unsigned)blocks), dim3(256), 0,                    \
                     reinterpret_cast<hipStream_t>(stream), hs, inv_freq, position_offset, table_scale)
  if (per >= 2) SPX_LAUNCH_D(2);
  else SPX_LAUNCH_D(1);
#undef SPX_LAUNCH
#undef SPX_LAUNCH_D
  return check_launch(fn);
}

extern "C" int spx_head_norm_rope_sets(const spx_head_norm* sets, int32_t count, const float* inv_freq, int32_t D,
                                       int64_t position_offset, float table_scale, void* stream) {
  return head_norm_rope_launch(__func__, sets, count, inv_freq, D, position_offset, table_scale, stream);
}
extern "C" int spx_head_norm_rope_bwd_sets(const spx_head_norm* sets, int32_t count, const float* inv_freq, int32_t D,
                                           int64_t position_offset, float table_scale, void* stream) {
  return head_norm_rope_bwd_launch(__func__, sets, count, inv_freq, D, position_offset, table_scale, stream);
}
extern "C" int spx_head_norm_rope(const void* tok, int64_t ld_tok, void* out, int64_t out_head_stride, void* pass,
                                  int64_t pass_head_stride, const int64_t* position_ids, const float* inv_freq,
                                  const void* gain, float* rstd, int64_t T, int32_t n_heads, int32_t n_pass, int32_t D,
                                  int64_t position_offset, float table_scale, float eps, void* stream) {
  const spx_head_norm set = {tok, ld_tok, out, out_head_stride, pass, pass_head_stride, position_ids, gain, rstd, T, n_heads,
                             n_pass, eps, 0, nullptr, 0, nullptr};
  return head_norm_rope_launch(__func__, &set, 1, inv_freq, D, position_offset, table_scale, stream);
}
extern "C" int spx_head_norm_rope_bwd(const void* tok, int64_t ld_tok, const void* dout, int64_t dout_head_stride,
                                      const void* dpass, int64_t dpass_head_stride, const int64_t* position_ids,
                                      const float* inv_freq, const void* gain, const float* rstd, void* dtok,
                                      int64_t ld_dtok, float* dw_scratch, int32_t accumulate, int64_t T, int32_t n_heads,
                                      int32_t n_pass, int32_t D, int64_t position_offset, float table_scale,
                                      void* stream) {
  const spx_head_norm set = {tok, ld_tok, const_cast<void*>(dout), dout_head_stride, const_cast<void*>(dpass),
                             dpass_head_stride, position_ids, gain, const_cast<float*>(rstd), T, n_heads, n_pass, 0.f,
                             accumulate, dtok, ld_dtok, dw_scratch};
  return head_norm_rope_bwd_launch(__func__, &set, 1, inv_freq, D, position_offset, table_scale, stream);
}

#undef SPX_REQ_FN

extern "C" int spx_swiglu_rows_fwd(const void* gate, int64_t ld_gate, const void* up, int64_t ld_up,
                                   void* out, int64_t ld_out, int64_t rows, int64_t F, void* stream) {
  SPX_REQUIRE(rows > 0 && F > 0 && F % 8 == 0, "rows > 0 and F a positive multiple of 8");
  SPX_REQUIRE(ld_gate >= F && ld_up >= F && ld_out >= F && ld_gate % 8 == 0 && ld_up % 8 == 0 && ld_out % 8 == 0,
              "row strides must be multiples of 8 and at least F");
  SPX_REQUIRE(gate && up && out && al16(gate) && al16(up) && al16(out), "null or unaligned buffer");
  const int64_t f8 = F / 8;
  hipLaunchKernelGGL(swiglu_fwd_kernel, dim3(swiglu_grid(rows * f8)), dim3(256), 0,
                     reinterpret_cast<hipStream_t>(stream), reinterpret_cast<const uint16_t*>(gate), ld_gate,
                     reinterpret_cast<const uint16_t*>(up), ld_up, reinterpret_cast<uint16_t*>(out), ld_out,
                     rows, f8);
  return check_launch(__func__);
}

extern "C" int spx_swiglu_rows_bwd(const void* gate, int64_t ld_gate, const void* up, int64_t ld_up,
                                   const void* dout, int64_t ld_dout, void* dgate, int64_t ld_dgate,
                                   void* dup, int64_t ld_dup, int64_t rows, int64_t F, void* stream) {
  SPX_REQUIRE(rows > 0 && F > 0 && F % 8 == 0, "rows > 0 and F a positive multiple of 8");
  SPX_REQUIRE(ld_gate >= F && ld_up >= F && ld_dout >= F && ld_dgate >= F && ld_dup >= F &&
                  ld_gate % 8 == 0 && ld_up % 8 == 0 && ld_dout % 8 == 0 && ld_dgate % 8 == 0 && ld_dup % 8 == 0,
              "row strides must be multiples of 8 and at least F");
  SPX_REQUIRE(gate && up && dout && dgate && dup, "null buffer");
  SPX_REQUIRE(al16(gate) && al16(up) && al16(dout) && al16(dgate) && al16(dup), "buffers must be 16-byte aligned");
  const int64_t f8 = F / 8;
  hipLaunchKernelGGL(swiglu_bwd_kernel, dim3(swiglu_grid(rows * f8)), dim3(256), 0,
                     reinterpret_cast<hipStream_t>(stream), reinterpret_cast<const uint16_t*>(gate), ld_gate,
                     reinterpret_cast<const uint16_t*>(up), ld_up, reinterpret_cast<const uint16_t*>(dout), ld_dout,
                     reinterpret_cast<uint16_t*>(dgate), ld_dgate, reinterpret_cast<uint16_t*>(dup), ld_dup, rows,
                     f8);
  return check_launch(__func__);
}

extern "C" int spx_swiglu_fwd(const void* gate, const void* up, void* out, int64_t n, void* stream) {
  return spx_swiglu_rows_fwd(gate, n, up, n, out, n, 1, n, stream);
}

extern "C" int spx_swiglu_bwd(const void* gate, const void* up, const void* dout, void* dgate, void* dup,
                              int64_t n, void* stream) {
  return spx_swiglu_rows_bwd(gate, n, up, n, dout, n, dgate, n, dup, n, 1, n, stream);
}
