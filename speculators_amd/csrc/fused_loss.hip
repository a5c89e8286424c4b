// Fused vocabulary loss for gfx950: one workgroup streams one (draft row,
// target row) pair with 16-byte loads, keeps online soft-max statistics of
// both rows, the first-index arg-max of both rows and the loss reduction in
// registers, and never materialises probabilities.  HBM-bound: algorithmic
// traffic is 2 rows read (forward) and 2 rows read + 1 row written (backward).
//
// All exponentials run in the base-2 domain (v_exp_f32 is 2^x): logits are
// pre-scaled by log2(e), statistics are converted back at the end.

#include <algorithm>

#include "loss_common.h"
#include "../../include/spx.h"

namespace spx {

// ---- running statistics ----------------------------------------------------
struct RowStats {
  float md, zd;        // draft: running max (base-2 scaled) and sum of 2^(x' - md)
  float mt, zt, at;    // target: same, and sum of 2^(y' - mt) * (y - x); rkl: of 2^(x' - md) * ((x - bd) - (y - bt)) * kRklUnit
  float bd; int id;    // draft arg-max value / first index
  float bt; int it; float xt;  // target arg-max value / first index / draft logit there
};

// rkl walks a row once: its sum of 2^(x' - md) * ((x - bd) - (y - bt)) is kept beside the soft-max's, relative to the largest
// values so far (us, read twice / once: bf16 64 x 32000 16.8 / 11.4, 333 22.9 / 18.0, 3000 114 / 80, 1024 x 128256 158 / 98; fp32 333 x
// 32000 34.0 / 22.9, 1024 x 128256 312 / 185; against float64 its losses are off by 1e-7 in the place of 7e-7, its gradients by 5e-7 in
// the place of 1e-6).  It is kept in units of 2^32, exactly: there are up to as many terms as columns, each as large as the type has
// values where the target rules columns out that the draft gives weight, and only their mean has to be a number.
constexpr float kRklUnit = 0x1p-32f;
// that sum after the draft's largest value has risen by dx and the target's by dy
__device__ __forceinline__ float off_by(float at, float z, float dy, float dx) {
  return z == 0.f ? at : fmaf(z * kRklUnit, dy - dx, at);
}
// A wave's statistics in every lane of it.  The largest value and its first index come first, then every sum is scaled once.
// (A tree of pairwise merges, ten shuffles a level and two exponentials a sum, and a walk over the waves' results behind it took
// 2 us of a row: 64 rows of 32000 bf16, kl 13.4 -> 10.0 us, 333 rows 17.9 -> 16.4.)
// DRAFT: `at` is that of rkl.
template <bool DRAFT = false>
__device__ __forceinline__ RowStats wave_merge(RowStats s) {
  const auto most = [](float x, float y) { return fmaxf(x, y); };
  const auto least = [](int x, int y) { return min(x, y); };
  const auto add = [](float x, float y) { return x + y; };
  const float md = wave_all(s.md, most), mt = wave_all(s.mt, most);
  const float rd = fast_exp2(s.md - md), rt = fast_exp2(s.mt - mt);
  const float bd = wave_all(s.bd, most), bt = wave_all(s.bt, most);
  if (DRAFT)
    s.at = off_by(s.at, s.zd, fmaxf(bt, kNegBig) - fmaxf(s.bt, kNegBig), fmaxf(bd, kNegBig) - fmaxf(s.bd, kNegBig));
  s.zd = wave_all(s.zd * rd, add);
  s.zt = wave_all(s.zt * rt, add);
  s.at = wave_all(s.at * (DRAFT ? rd : rt), add);
  s.md = md;
  s.mt = mt;
  s.id = wave_all(s.bd == bd ? s.id : 0x7fffffff, least);
  const int it = wave_all(s.bt == bt ? s.it : 0x7fffffff, least);
  // (a row of the target without a value: no lane has an index, the first one's draft logit stands in, see settle)
  const unsigned long long has = __builtin_amdgcn_ballot_w64(s.bt == bt && s.it == it);
  s.xt = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(s.xt), has ? __builtin_ctzll(has) : 0));
  s.it = it;
  s.bd = bd;
  s.bt = bt;
  return s;
}

template <int WAVES>
__device__ __forceinline__ float block_sum(float v, float* lds) {
  v = wave_sum(v);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) lds[threadIdx.x >> 6] = v;
  __syncthreads();
  float t = 0.f;
#pragma unroll
  for (int w = 0; w < WAVES; ++w) t += lds[w];
  return t;
}
__device__ __forceinline__ RowStats no_stats() {
  RowStats s;
  s.md = kNegBig; s.zd = 0.f; s.mt = kNegBig; s.zt = 0.f; s.at = 0.f;
  s.bd = -INFINITY; s.id = 0x7fffffff; s.bt = -INFINITY; s.it = 0x7fffffff; s.xt = 0.f;
  return s;
}
// merges the statistics of all threads; every thread gets the result
template <int WAVES, bool DRAFT = false>
__device__ __forceinline__ RowStats block_merge(RowStats s, RowStats* part) {
  const int lane = threadIdx.x & 63;
  s = wave_merge<DRAFT>(s);
  if (lane == 0) part[threadIdx.x >> 6] = s;
  __syncthreads();
  s = no_stats();
  if (lane < WAVES) s = part[lane];
  return wave_merge<DRAFT>(s);
}

// log p - log m and log q - log m of the mean m of two probabilities p and q with the logarithms ldp and ltp: the larger one's
// logarithm cancels, so no term of its size stands in either.  In natural units: a column at the type's lowest value on one side has
// a finite difference, and 0 times it is nothing (times log2(e) it would be infinite, and the row not a number).  (No expression that
// the compiler could fuse in one direction and not in the other.)
struct MixLogs { float p, q; };
__device__ __forceinline__ MixLogs mix_logs(float ldp, float ltp) {
  const float d = ldp - ltp;
  const float w = 1.f - fast_log2(1.f + fast_exp2(-fabsf(d) * kLog2e));
  return {fmaf(w, kLn2, fminf(d, 0.f)), fmaf(w, kLn2, -fmaxf(d, 0.f))};
}

__device__ __forceinline__ void store_flag(void* p, int kind, int64_t i, bool v) {
  switch (kind) {
    case SPX_KIND_U8: reinterpret_cast<uint8_t*>(p)[i] = v ? 1 : 0; break;
    case SPX_KIND_I32: reinterpret_cast<int32_t*>(p)[i] = v ? 1 : 0; break;
    case SPX_KIND_I64: reinterpret_cast<int64_t*>(p)[i] = v ? 1 : 0; break;
    case SPX_KIND_F32: reinterpret_cast<float*>(p)[i] = v ? 1.f : 0.f; break;
    default: reinterpret_cast<uint16_t*>(p)[i] = v ? 0x3f80 : 0; break;
  }
}

// ---- what one TTT step adds to the row pass --------------------------------------
// d2t != nullptr: `targets` are full-vocabulary rows (vt wide) and target element i is read at
// i + d2t[i] (model.py:161-169, train/vocab_mapping.py:86-96); `gathered` (may be nullptr) then
// receives the draft-vocabulary row, for the later steps and the backward.
// counts != nullptr: the row's part of the acceptance chain (models/metrics.py:6-36): with
// m = mask[r] != 0, was = prev[r] != 0, hit = argmax_draft == argmax_target, now = was && hit:
//   counts[0] += m && now,  counts[1] += m,  counts[2] += was,  prev[r] = now.
// Integer atomics: the sums do not depend on the order of the rows.
struct StepArgs {
  const int64_t* d2t; int64_t vt;
  void* gathered; int64_t ld_gathered;
  const void* mask; int mask_kind;
  void* prev; int prev_kind;
  int32_t* counts;
};

// eight target elements through the offset table (ascending indices: neighbouring lanes read
// neighbouring sectors of the full row)
template <typename T>
__device__ __forceinline__ void load8_gather(const T* full, const int64_t* __restrict__ d2t, int64_t base,
                                             int64_t n, int64_t vt, float v[8]) {
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    float val = kNegBig;  // tail padding, like load8_guard
    if (base + i < n) {
      const int64_t j = base + i + d2t[base + i];
      val = (j >= 0 && j < vt) ? load1(full + j) : -INFINITY;
    }
    v[i] = val;
  }
}

// eight elements of both rows into a thread's statistics
template <int OP, bool KNOWN>
__device__ __forceinline__ void add_chunk(RowStats& s, const float (&x)[8], const float (&y)[8], int64_t base,
                                          float lt2_known) {
  const float mx_was = fmaxf(s.bd, kNegBig), my_was = fmaxf(s.bt, kNegBig);
  float cx = x[0], cy = y[0];
#pragma unroll
  for (int i = 1; i < 8; ++i) cx = fmaxf(cx, x[i]);
  if (!KNOWN) {
#pragma unroll
    for (int i = 1; i < 8; ++i) cy = fmaxf(cy, y[i]);
  }
  if (cx > s.bd) {  // strict: an earlier chunk of this thread keeps a tie
    int k = 7;
#pragma unroll
    for (int i = 6; i >= 0; --i) k = (x[i] == cx) ? i : k;
    s.bd = cx; s.id = (int)base + k;
  }
  if (!KNOWN && cy > s.bt) {
    int k = 7;
    float xv = x[7];
#pragma unroll
    for (int i = 6; i >= 0; --i) {
      const bool hit = y[i] == cy;
      k = hit ? i : k;
      xv = hit ? x[i] : xv;
    }
    s.bt = cy; s.it = (int)base + k; s.xt = xv;
  }
  {
    const float cxs = cx * kLog2e;
    float mn = s.md, z = s.zd, a = s.at;
    const float mx = fmaxf(s.bd, kNegBig), my = fmaxf(s.bt, kNegBig);
    if (OP == SPX_LOSS_RKL && (mx > mx_was || my > my_was)) a = off_by(a, z, my - my_was, mx - mx_was);
    if (cxs > mn) {  // the running max moves rarely once a few chunks have been seen
      const float by = fast_exp2(mn - cxs);
      z *= by;
      if (OP == SPX_LOSS_RKL) a *= by;
      mn = cxs;
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float e = fast_exp2(fmaf(x[i], kLog2e, -mn));
      z += e;
      if (OP == SPX_LOSS_RKL) a = fmaf(e, fmaf(x[i], kRklUnit, -mx * kRklUnit) - fmaf(y[i], kRklUnit, -my * kRklUnit), a);
    }
    s.zd = z; s.md = mn;
    if (OP == SPX_LOSS_RKL) s.at = a;
  }
  if (KNOWN && OP == SPX_LOSS_KL) {
    float a = s.at;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float pr = fast_exp2(fmaf(y[i], kLog2e, -lt2_known));  // the target probability
      a = fmaf(pr, y[i] - x[i], a);
    }
    s.at = a;
  } else if (OP != SPX_LOSS_CE) {
    float mn = fmaxf(s.mt, cy * kLog2e);
    float rs = fast_exp2(s.mt - mn);
    float z = s.zt * rs, a = s.at * rs;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      float e = fast_exp2(fmaf(y[i], kLog2e, -mn));
      z += e;
      if (OP == SPX_LOSS_KL) a = fmaf(e, y[i] - x[i], a);
    }
    s.zt = z; s.mt = mn;
    if (OP == SPX_LOSS_KL) s.at = a;
  }
}

// what the second walk over a row adds: rkl (where other terms want it, too), jsd, tv
template <int OP>
__device__ __forceinline__ void add_second(float& acc, float& ext, const float (&x)[8], const float (&y)[8], float lse_d,
                                           float lse_t) {
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const float ldp = x[i] - lse_d, ltp = y[i] - lse_t, a = ldp * kLog2e, b = ltp * kLog2e;
    if (OP == SPX_LOSS_RKL) {
      acc = fmaf(fast_exp2(a), ldp - ltp, acc);
    } else if (OP == SPX_LOSS_JSD) {
      const MixLogs l = mix_logs(ldp, ltp);
      acc = fmaf(fast_exp2(a), l.p, acc);
      ext = fmaf(fast_exp2(b), l.q, ext);
    } else {  // TV
      const float dp = fast_exp2(a), tp = fast_exp2(b);
      acc += fminf(dp, tp);
      ext += (dp <= tp) ? dp : 0.f;
    }
  }
}

// The arg-max of a row without a value above -infinity (all of it -infinity or NaN, where tail padding may have won, too) is
// 0, as torch has it: whatever a row holds and whatever known statistics say, the indices are columns of it.
template <typename T>
__device__ __forceinline__ void settle(RowStats& s, const T* xrow, int64_t vocab) {
  if ((uint32_t)s.id >= (uint32_t)vocab) s.id = 0;
  if ((uint32_t)s.it >= (uint32_t)vocab) { s.it = 0; s.xt = load1(xrow); }
}

// one thread writes what a row leaves behind
template <bool KNOWN>
__device__ __forceinline__ void store_row(int64_t r, const RowStats& s, float row_loss, float lse_d, float lse_t,
                                          float* __restrict__ loss, float* __restrict__ lse_draft,
                                          float* __restrict__ lse_target, int32_t* __restrict__ argmax_draft,
                                          int32_t* __restrict__ argmax_target, const StepArgs& sa) {
  loss[r] = row_loss;
  lse_draft[r] = lse_d;
  if (argmax_draft) argmax_draft[r] = s.id;
  if (!KNOWN) {
    lse_target[r] = lse_t;
    if (argmax_target) argmax_target[r] = s.it;
  }
  if (sa.counts) {
    const bool m = sa.mask ? mask_value(sa.mask, sa.mask_kind, r) != 0.f : true;
    const bool was = sa.prev ? mask_value(sa.prev, sa.prev_kind, r) != 0.f : true;
    const bool now = was && (s.id == s.it);
    if (m && now) atomicAdd(&sa.counts[0], 1);
    if (m) atomicAdd(&sa.counts[1], 1);
    if (was) atomicAdd(&sa.counts[2], 1);
    if (sa.prev) store_flag(sa.prev, sa.prev_kind, r, now);
  }
}

// ---- forward ---------------------------------------------------------------
// eight elements as they come from memory
template <typename T>
struct RawChunk;
template <>
struct RawChunk<uint16_t> {
  u32x4 a;
  // KEEP: the row is read again, from L2
  template <bool KEEP>
  __device__ __forceinline__ void load(const uint16_t* p) { a = KEEP ? *reinterpret_cast<const u32x4*>(p) : ld16(p); }
  __device__ __forceinline__ void pin() { asm volatile("" : "+v"(a)); }
  __device__ __forceinline__ void get(float (&v)[8]) const {
    v[0] = bf16_lo(a.x); v[1] = bf16_hi(a.x); v[2] = bf16_lo(a.y); v[3] = bf16_hi(a.y);
    v[4] = bf16_lo(a.z); v[5] = bf16_hi(a.z); v[6] = bf16_lo(a.w); v[7] = bf16_hi(a.w);
  }
};
template <>
struct RawChunk<float> {
  u32x4 a, b;
  template <bool KEEP>
  __device__ __forceinline__ void load(const float* p) {
    a = KEEP ? *reinterpret_cast<const u32x4*>(p) : ld16(p);
    b = KEEP ? *reinterpret_cast<const u32x4*>(p + 4) : ld16(p + 4);
  }
  __device__ __forceinline__ void pin() { asm volatile("" : "+v"(a), "+v"(b)); }
  __device__ __forceinline__ void get(float (&v)[8]) const {
#pragma unroll
    for (int i = 0; i < 4; ++i) { v[i] = __uint_as_float(a[i]); v[4 + i] = __uint_as_float(b[i]); }
  }
};

constexpr int gather_stage_bytes(int threads) { return threads * 128; }

// KNOWN: lse_target / argmax_target are INPUTS (the target row's statistics from an
// earlier pass over the same row); the target max / sum / arg-max tracking is skipped and
// the cross-entropy reduction does not read the target row at all.
// GATHER: the target row is read through the d2t offset table (see StepArgs).
// NT: threads per row.  A call of few rows leaves compute units idle with 256 (see threads_per_row).
// HELD: chunks of each row that a thread keeps in registers between the first walk and the second (jsd, tv; 0: none, the second
// walk reads memory again).
template <typename T, int OP, bool VEC, bool KNOWN, bool GATHER, int NT, int HELD>
__global__ __launch_bounds__(NT, HELD * sizeof(T) > 16 ? 2 : HELD ? 4 : 1) void loss_fwd_kernel(
    const T* __restrict__ logits, int64_t ld_logits, const T* __restrict__ targets,
    int64_t ld_targets, int64_t vocab, float* __restrict__ loss, float* __restrict__ lse_draft,
    float* __restrict__ lse_target, float* __restrict__ extra, int32_t* __restrict__ argmax_draft,
    int32_t* __restrict__ argmax_target, StepArgs sa, bool keep) {
  static_assert(!KNOWN || OP == SPX_LOSS_KL || OP == SPX_LOSS_CE, "the others form the target's statistics as they go");
  const int64_t r = blockIdx.x;
  const T* xrow = logits + r * ld_logits;
  const T* yrow = targets + r * ld_targets;
  T* grow = (GATHER && sa.gathered) ? reinterpret_cast<T*>(sa.gathered) + r * sa.ld_gathered : nullptr;
  const int tid = threadIdx.x;
  const int64_t nchunks = (vocab + 7) >> 3;

  const float lt2_known = KNOWN ? lse_target[r] * kLog2e : 0.f;  // base-2 target lse
  const bool read_y = !(KNOWN && OP == SPX_LOSS_CE);
  RowStats s = no_stats();

  // GATHER: the draft ids of one tile (256 chunks) map to an ascending span of the full row.
  // The span is brought into LDS with coalesced 16-byte loads and the eight elements of a lane
  // are picked from there; a span that does not fit (or rows without 16-byte alignment) and any
  // id that falls outside the span (a table that is not ascending) read the row directly.
  constexpr int kStageElems = GATHER ? gather_stage_bytes(NT) / (int)sizeof(T) : 1;
  extern __shared__ __attribute__((aligned(16))) uint8_t stage_mem[];
  T* const stage = reinterpret_cast<T*>(stage_mem);
  // Without the gather: four chunks of each row are requested before the first is worked on (a row of 32000 is 16 trips of
  // 256 threads, each of which waited a memory latency).
  constexpr bool kStream = VEC && !GATHER;
  constexpr bool kTwice = (OP == SPX_LOSS_JSD || OP == SPX_LOSS_TV) && !HELD;
  constexpr int U = 4;
  const int64_t nfull = vocab >> 3;
  RawChunk<T> xh[HELD ? HELD : 1], yh[HELD ? HELD : 1];
  if constexpr (HELD > 0) {
    static_assert(kStream && (OP == SPX_LOSS_JSD || OP == SPX_LOSS_TV), "rows that are walked twice");
#pragma unroll
    for (int k = 0; k < HELD; ++k)
      if (tid + k * NT < nfull) {
        xh[k].template load<true>(xrow + ((int64_t)(tid + k * NT) << 3));
        yh[k].template load<true>(yrow + ((int64_t)(tid + k * NT) << 3));
      }
#pragma unroll
    for (int k = 0; k < HELD; ++k)
      if (tid + k * NT < nfull) {
        float x[8], y[8];
        xh[k].get(x);
        yh[k].get(y);
        add_chunk<OP, KNOWN>(s, x, y, (int64_t)(tid + k * NT) << 3, lt2_known);
      }
  } else if (kStream) {
    auto walk = [&](auto kept) __attribute__((always_inline)) {
      constexpr bool kKeep = decltype(kept)::value;
      for (int64_t c = tid; c < nfull; c += NT * U) {
        RawChunk<T> xr[U], yr[U];
#pragma unroll
        for (int u = 0; u < U; ++u)
          if (c + u * NT < nfull) {
            xr[u].template load<kKeep>(xrow + ((c + u * NT) << 3));
            if (read_y) yr[u].template load<kKeep && OP != SPX_LOSS_CE>(yrow + ((c + u * NT) << 3));
          }
#pragma unroll
        for (int u = 0; u < U; ++u)
          if (c + u * NT < nfull) {
            float x[8], y[8] = {};
            xr[u].get(x);
            if (read_y) yr[u].get(y);
            add_chunk<OP, KNOWN>(s, x, y, (c + u * NT) << 3, lt2_known);
          }
      }
    };
    if (kTwice || keep) walk(std::true_type{});
    else walk(std::false_type{});
  }
  // (streaming: what is left is an incomplete last chunk, in the thread whose turn it is)
  for (int64_t c0 = kStream ? nfull / NT * NT : 0; c0 < nchunks; c0 += NT) {
    const int64_t c = c0 + tid;
    if (kStream && c < nfull) continue;
    const bool active = c < nchunks;
    const int64_t base = c << 3;
    float x[8], y[8];
    if (GATHER) {
      // this lane's draft row chunk and its eight target columns first: their latency runs
      // under the staging of the span
      int64_t jj[8];
      if (active) {
        load8<T, VEC>(xrow, base, vocab, x);
        if (base + 8 <= vocab && ptr_aligned16(sa.d2t)) {
          const u32x4* dp = reinterpret_cast<const u32x4*>(sa.d2t + base);
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const u32x4 w = dp[q];
            jj[2 * q] = base + 2 * q + (int64_t)(((uint64_t)w.y << 32) | w.x);
            jj[2 * q + 1] = base + 2 * q + 1 + (int64_t)(((uint64_t)w.w << 32) | w.z);
          }
        } else {
#pragma unroll
          for (int i = 0; i < 8; ++i) jj[i] = base + i < vocab ? base + i + sa.d2t[base + i] : -1;
        }
      }
      const int64_t i0 = c0 << 3, i1 = min(vocab, (c0 + NT) << 3) - 1;
      int64_t lo = i0 + sa.d2t[i0], hi = i1 + sa.d2t[i1] + 1;
      lo = max((int64_t)0, min(lo, sa.vt)) & ~(int64_t)7;
      hi = max(lo, min(hi, sa.vt));
      constexpr int EPV = 16 / (int)sizeof(T);  // elements per 16-byte access
      const bool staged = VEC && (hi - lo) <= kStageElems && ((ld_targets & 7) == 0) &&
                          ptr_aligned16(targets);
      if (staged) {
        __syncthreads();  // the previous tile's picks are done
        for (int64_t e = (int64_t)tid * EPV; lo + e < hi; e += NT * EPV) {
          if (lo + e + EPV <= sa.vt)
            *reinterpret_cast<u32x4*>(&stage[e]) = ld16(yrow + lo + e);
          else
            for (int q = 0; q < EPV; ++q)
              if (lo + e + q < sa.vt) stage[e + q] = yrow[lo + e + q];
        }
        __syncthreads();
      }
      if (active) {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          float val = kNegBig;  // tail padding, like load8_guard
          if (base + i < vocab) {
            const int64_t j = jj[i];
            if (staged && j >= lo && j < hi) val = load1(&stage[j - lo]);
            else val = (j >= 0 && j < sa.vt) ? load1(yrow + j) : -INFINITY;
          }
          y[i] = val;
        }
        if (grow) store8<T, VEC>(grow, base, vocab, y);
      }
    } else if (active) {
      load8<T, VEC>(xrow, base, vocab, x);
      if (read_y) load8<T, VEC>(yrow, base, vocab, y);
    }
    if (!active) continue;
    add_chunk<OP, KNOWN>(s, x, y, base, lt2_known);
  }

  __shared__ RowStats part[NT / 64];
  __shared__ float red[NT / 64];
  s = block_merge<NT / 64, OP == SPX_LOSS_RKL>(s, part);

  float lse_d = (s.md + fast_log2(s.zd)) * kLn2;
  float lse_t = KNOWN ? lse_target[r]
                      : ((OP != SPX_LOSS_CE) ? (s.mt + fast_log2(s.zt)) * kLn2 : 0.f);
  // (what follows takes them rounded, as they are stored for the backward, and not as the product inside a fused difference: the
  // gradients of nearly equal rows live on the two directions' errors being the same)
  if (OP == SPX_LOSS_RKL || OP == SPX_LOSS_JSD || OP == SPX_LOSS_TV) asm volatile("" : "+v"(lse_d), "+v"(lse_t));
  if (KNOWN) s.it = argmax_target ? argmax_target[r] : 0;
  settle(s, xrow, vocab);
  if (KNOWN && OP == SPX_LOSS_CE) s.xt = load1(xrow + s.it);

  float row_loss = 0.f, row_extra = 0.f;
  if (OP == SPX_LOSS_KL) {
    row_loss = (KNOWN ? s.at : s.at / s.zt) - lse_t + lse_d;
    row_extra = row_loss;
  } else if (OP == SPX_LOSS_CE) {
    row_loss = lse_d - s.xt;
  } else if (OP == SPX_LOSS_RKL) {
    // the mean of x - y under the draft's probabilities, less the log-sum-exps' difference, both counted from the rows' largest
    // values: for the loss what lies between those cancels (but for the rounding of md and mt), for the backward it is formed from
    // what is stored and subtracted there, too (rows that are nearly equal, or but for a constant, keep their digits)
    const float bd = fmaxf(s.bd, kNegBig), bt = fmaxf(s.bt, kNegBig), mean = s.at / s.zd * (1.f / kRklUnit);
    row_loss = mean - (fast_log2(s.zd / s.zt) - (fmaf(bd, kLog2e, -s.md) - fmaf(bt, kLog2e, -s.mt))) * kLn2;
    row_extra = mean + ((bd - lse_d) - (bt - lse_t));
  } else {
    float acc = 0.f, ext = 0.f;
    if constexpr (HELD > 0) {
#pragma unroll
      for (int k = 0; k < HELD; ++k) { xh[k].pin(); yh[k].pin(); }  // (what stays in registers are the chunks as they came)
#pragma unroll
      for (int k = 0; k < HELD; ++k)
        if (tid + k * NT < nfull) {
          float x[8], y[8];
          xh[k].get(x);
          yh[k].get(y);
          add_second<OP>(acc, ext, x, y, lse_d, lse_t);
        }
    } else if (kStream)
      for (int64_t c = tid; c < nfull; c += NT * U) {
        RawChunk<T> xr[U], yr[U];
#pragma unroll
        for (int u = 0; u < U; ++u)
          if (c + u * NT < nfull) {
            xr[u].template load<false>(xrow + ((c + u * NT) << 3));
            yr[u].template load<false>(yrow + ((c + u * NT) << 3));
          }
#pragma unroll
        for (int u = 0; u < U; ++u)
          if (c + u * NT < nfull) {
            float x[8], y[8];
            xr[u].get(x);
            yr[u].get(y);
            add_second<OP>(acc, ext, x, y, lse_d, lse_t);
          }
      }
    for (int64_t c = kStream ? nfull / NT * NT + tid : tid; c < nchunks; c += NT) {
      if (kStream && c < nfull) continue;
      const int64_t base = c << 3;
      float x[8], y[8];
      load8<T, VEC>(xrow, base, vocab, x);
      if (GATHER && grow) load8<T, VEC>(grow, base, vocab, y);  // (this thread's own stores)
      else if (GATHER) load8_gather<T>(yrow, sa.d2t, base, vocab, sa.vt, y);
      else load8<T, VEC>(yrow, base, vocab, y);
      add_second<OP>(acc, ext, x, y, lse_d, lse_t);
    }
    acc = block_sum<NT / 64>(acc, red);
    ext = block_sum<NT / 64>(ext, red);
    if (OP == SPX_LOSS_JSD) { row_loss = 0.5f * (acc + ext); row_extra = acc; }
    else { row_loss = 1.f - acc; row_extra = ext; }
  }
  if (tid == 0) {
    extra[r] = row_extra;
    store_row<KNOWN>(r, s, row_loss, lse_d, lse_t, loss, lse_draft, lse_target, argmax_draft, argmax_target, sa);
  }
}

// ---- forward and logits gradient in one pass -------------------------------------------------------
// The head of a TTT step is frozen while the draft layers train, and which rows carry a gradient is
// known before the loss is (the loss mask): the row pass can then leave the gradient of the logits
// behind as well, and the row pair is read ONCE instead of once by the forward and once more by the
// backward.  One workgroup of 512 threads holds a whole row pair in registers (eight 16-byte chunks of
// each row per thread as they come from memory, requested before anything is computed: vocab <= 32768,
// bf16), reduces it to the row statistics exactly like loss_fwd_kernel, and, for a row that row_map
// sends to a slot >= 0, goes over its registers a second time and writes
//   grad[slot, :] = softmax(x) - softmax(y)   (kl)      softmax(x) - onehot(argmax y)   (ce)
// -- the gradient for a row weight of ONE; the input-gradient product, which is linear in it, applies the weight the reduction
// behind the loss gives the row to its fp32 sums, before their one rounding (spx_gemm_bf16_rows_graded).  Rows mapped to -1 get
// no gradient row, and with the target statistics handed in (KNOWN) their target row is not read at
// all, no soft-max of their draft row is formed and their loss is written as zero: a masked row's loss enters
// no sum.  (Their arg-max outputs and their part of the acceptance chain are those of any row.)
constexpr int kFgThreads = 512, kFgWaves = kFgThreads / 64, kFgChunks = 8;
template <int OP, bool KNOWN>
__global__ __launch_bounds__(kFgThreads) __attribute__((amdgpu_waves_per_eu(4, 4))) void loss_fwd_grad_kernel(
    const uint16_t* __restrict__ logits, int64_t ld_logits, const uint16_t* __restrict__ targets,
    int64_t ld_targets, int64_t vocab, float* __restrict__ loss, float* __restrict__ lse_draft,
    float* __restrict__ lse_target, float* __restrict__ extra, int32_t* __restrict__ argmax_draft,
    int32_t* __restrict__ argmax_target, StepArgs sa, const int32_t* __restrict__ row_map,
    uint16_t* __restrict__ grad, int64_t ld_grad) {
  const int64_t r = blockIdx.x;
  const int tid = threadIdx.x;
  const int nchunks = (int)(vocab >> 3);  // vocab is a multiple of 8 here
  const int slot = row_map[r];
  const bool live = slot >= 0;
  const uint16_t* xrow = logits + r * ld_logits;
  const uint16_t* yrow = targets ? targets + r * ld_targets : nullptr;
  const bool read_y = !(KNOWN && (OP == SPX_LOSS_CE || !live));
  u32x4 xr[kFgChunks], yr[kFgChunks];
#pragma unroll
  for (int k = 0; k < kFgChunks; ++k) {
    const int c = tid + k * kFgThreads;
    if (c < nchunks) {
      xr[k] = ld16(xrow + ((int64_t)c << 3));
      if (read_y) yr[k] = ld16(yrow + ((int64_t)c << 3));
    }
  }
  const float lt2_known = KNOWN ? lse_target[r] * kLog2e : 0.f;  // base-2 target lse
  // a masked row whose target statistics are known needs nothing but the draft row's arg-max
  const bool soft_x = live || !KNOWN;
  RowStats s = no_stats();
  auto unpack = [](u32x4 raw, float v[8]) {
    v[0] = bf16_lo(raw.x); v[1] = bf16_hi(raw.x); v[2] = bf16_lo(raw.y); v[3] = bf16_hi(raw.y);
    v[4] = bf16_lo(raw.z); v[5] = bf16_hi(raw.z); v[6] = bf16_lo(raw.w); v[7] = bf16_hi(raw.w);
  };
#pragma unroll
  for (int k = 0; k < kFgChunks; ++k) {
    const int c = tid + k * kFgThreads;
    if (c >= nchunks) continue;
    const int base = c << 3;
    float x[8], y[8];
    unpack(xr[k], x);
    if (read_y) unpack(yr[k], y);
    float cx = x[0];
#pragma unroll
    for (int i = 1; i < 8; ++i) cx = fmaxf(cx, x[i]);
    if (cx > s.bd) {  // strict: an earlier chunk of this thread keeps a tie
      int kk = 7;
#pragma unroll
      for (int i = 6; i >= 0; --i) kk = (x[i] == cx) ? i : kk;
      s.bd = cx; s.id = base + kk;
    }
    if (soft_x) {
      const float cxs = cx * kLog2e;
      float mn = s.md, z = s.zd;
      if (cxs > mn) {
        z *= fast_exp2(mn - cxs);
        mn = cxs;
      }
#pragma unroll
      for (int i = 0; i < 8; ++i) z += fast_exp2(fmaf(x[i], kLog2e, -mn));
      s.zd = z; s.md = mn;
    }
    if (!KNOWN) {
      float cy = y[0];
#pragma unroll
      for (int i = 1; i < 8; ++i) cy = fmaxf(cy, y[i]);
      if (cy > s.bt) {
        int kk = 7;
        float xv = x[7];
#pragma unroll
        for (int i = 6; i >= 0; --i) {
          const bool hit = y[i] == cy;
          kk = hit ? i : kk;
          xv = hit ? x[i] : xv;
        }
        s.bt = cy; s.it = base + kk; s.xt = xv;
      }
      if (OP != SPX_LOSS_CE) {
        float mn = fmaxf(s.mt, cy * kLog2e);
        float rs = fast_exp2(s.mt - mn);
        float z = s.zt * rs, a = s.at * rs;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          float e = fast_exp2(fmaf(y[i], kLog2e, -mn));
          z += e;
          a = fmaf(e, y[i] - x[i], a);
        }
        s.zt = z; s.at = a; s.mt = mn;
      }
    } else if (OP != SPX_LOSS_CE && live) {
      float a = s.at;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const float pr = fast_exp2(fmaf(y[i], kLog2e, -lt2_known));  // the target probability
        a = fmaf(pr, y[i] - x[i], a);
      }
      s.at = a;
    }
  }
  __shared__ RowStats part[kFgWaves];
  s = block_merge<kFgWaves>(s, part);

  const float lse_d = soft_x ? (s.md + fast_log2(s.zd)) * kLn2 : 0.f;
  const float lse_t = KNOWN ? lse_target[r]
                            : ((OP != SPX_LOSS_CE) ? (s.mt + fast_log2(s.zt)) * kLn2 : 0.f);
  if (KNOWN) s.it = argmax_target[r];
  settle(s, xrow, vocab);
  if (KNOWN && OP == SPX_LOSS_CE) s.xt = load1(xrow + s.it);
  if (tid == 0) {
    float row_loss;
    if (!soft_x) row_loss = 0.f;
    else if (OP == SPX_LOSS_KL) row_loss = (KNOWN ? s.at : s.at / s.zt) - lse_t + lse_d;
    else row_loss = lse_d - s.xt;
    loss[r] = row_loss;
    lse_draft[r] = lse_d;
    extra[r] = OP == SPX_LOSS_KL ? row_loss : 0.f;
    if (argmax_draft) argmax_draft[r] = s.id;
    if (!KNOWN) {
      lse_target[r] = lse_t;
      if (argmax_target) argmax_target[r] = s.it;
    }
    if (sa.counts) {
      const bool m = sa.mask ? mask_value(sa.mask, sa.mask_kind, r) != 0.f : true;
      const bool was = sa.prev ? mask_value(sa.prev, sa.prev_kind, r) != 0.f : true;
      const bool now = was && (s.id == s.it);
      if (m && now) atomicAdd(&sa.counts[0], 1);
      if (m) atomicAdd(&sa.counts[1], 1);
      if (was) atomicAdd(&sa.counts[2], 1);
      if (sa.prev) store_flag(sa.prev, sa.prev_kind, r, now);
    }
  }
  if (!live) return;
  uint16_t* grow = grad + (int64_t)slot * ld_grad;
  const float cd = -lse_d * kLog2e, ct = -lse_t * kLog2e;
  const int label = s.it;
  // (the packed chunks are what stays in registers between the passes, not their 64 + 64 unpacked values)
#pragma unroll
  for (int k = 0; k < kFgChunks; ++k) {
    asm volatile("" : "+v"(xr[k].x), "+v"(xr[k].y), "+v"(xr[k].z), "+v"(xr[k].w));
    if (OP != SPX_LOSS_CE) asm volatile("" : "+v"(yr[k].x), "+v"(yr[k].y), "+v"(yr[k].z), "+v"(yr[k].w));
  }
#pragma unroll
  for (int k = 0; k < kFgChunks; ++k) {
    const int c = tid + k * kFgThreads;
    if (c >= nchunks) continue;
    const int base = c << 3;
    float x[8], y[8], o[8];
    unpack(xr[k], x);
    if (OP != SPX_LOSS_CE) unpack(yr[k], y);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float dp = fast_exp2(fmaf(x[i], kLog2e, cd));
      if (OP == SPX_LOSS_CE) o[i] = dp - ((base + i) == label ? 1.f : 0.f);
      else o[i] = dp - fast_exp2(fmaf(y[i], kLog2e, ct));
    }
    store8_vec<uint16_t>(grow + ((int64_t)c << 3), o);
  }
}

// The same for a weighted sum of terms (any of the five, each at most once), and for rkl, jsd and tv alone: row losses of
// every term, statistics, arg-maxes, acceptance chain and the gradient of the sum from ONE read of the row pair.  What a
// term needs beyond the soft-max statistics (rkl, jsd, tv: both log-sum-exps first) is a second walk over the registers,
// the gradient a third; its terms are added in fp32 and rounded once.
//   grad[slot, :] = sum_t w_t dL_t/dx        loss[t][r] for the t-th term in the order of the ops
// {"ce": 0.1, "tv": 0.9} over 3001 rows of 32000, 70 % of them live, target statistics known: 135 us (4.2 TB/s; bound by
// vector instructions as much as by memory) where the two terms' forward passes, backward passes and the sum of their
// gradients took 121 + 69 + 104 + 73 + 89; and the head's input gradient runs over the live rows only (695 -> 490).
struct LossTerms {
  int mask;      // bit op: the term is there
  float w[5];    // by op
};

template <bool KNOWN, bool KL>
__global__ __launch_bounds__(kFgThreads) __attribute__((amdgpu_waves_per_eu(4, 4))) void loss_terms_grad_kernel(
    const uint16_t* __restrict__ logits, int64_t ld_logits, const uint16_t* __restrict__ targets, int64_t ld_targets,
    int64_t rows, int64_t vocab, float* __restrict__ loss, float* __restrict__ lse_draft,
    float* __restrict__ lse_target, int32_t* __restrict__ argmax_draft, int32_t* __restrict__ argmax_target, StepArgs sa,
    LossTerms tm, const int32_t* __restrict__ row_map, uint16_t* __restrict__ grad, int64_t ld_grad) {
  const int64_t r = blockIdx.x;
  const int tid = threadIdx.x;
  const int nchunks = (int)(vocab >> 3);
  const int slot = row_map[r];
  const bool live = slot >= 0;
  // (a masked row whose target statistics are known needs nothing but the draft row's arg-max)
  const bool soft = live || !KNOWN;
  const uint16_t* xrow = logits + r * ld_logits;
  const uint16_t* yrow = targets + r * ld_targets;
  u32x4 xr[kFgChunks], yr[kFgChunks];
#pragma unroll
  for (int k = 0; k < kFgChunks; ++k) {
    const int c = tid + k * kFgThreads;
    if (c < nchunks) {
      xr[k] = ld16(xrow + ((int64_t)c << 3));
      if (soft) yr[k] = ld16(yrow + ((int64_t)c << 3));
    }
  }
  auto unpack = [](u32x4 raw, float (&v)[8]) __attribute__((always_inline)) {
    v[0] = bf16_lo(raw.x); v[1] = bf16_hi(raw.x); v[2] = bf16_lo(raw.y); v[3] = bf16_hi(raw.y);
    v[4] = bf16_lo(raw.z); v[5] = bf16_hi(raw.z); v[6] = bf16_lo(raw.w); v[7] = bf16_hi(raw.w);
  };
  // the packed chunks are what stays in registers between the walks, not their unpacked values
  auto pin = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int k = 0; k < kFgChunks; ++k) {
      asm volatile("" : "+v"(xr[k].x), "+v"(xr[k].y), "+v"(xr[k].z), "+v"(xr[k].w));
      asm volatile("" : "+v"(yr[k].x), "+v"(yr[k].y), "+v"(yr[k].z), "+v"(yr[k].w));
    }
  };
  const float lt2_known = KNOWN ? lse_target[r] * kLog2e : 0.f;
  RowStats s = no_stats();
#pragma unroll
  for (int k = 0; k < kFgChunks; ++k) {
    const int c = tid + k * kFgThreads;
    if (c >= nchunks) continue;
    float x[8], y[8];
    unpack(xr[k], x);
    if (soft) {
      unpack(yr[k], y);
      // (ce with known statistics: the draft row's only; tv without: both rows', no sum over their difference)
      add_chunk<KL ? SPX_LOSS_KL : KNOWN ? SPX_LOSS_CE : SPX_LOSS_TV, KNOWN>(s, x, y, (int64_t)c << 3, lt2_known);
    } else {
#pragma unroll
      for (int i = 0; i < 8; ++i)
        if (x[i] > s.bd) { s.bd = x[i]; s.id = (c << 3) + i; }
    }
  }
  __shared__ RowStats part[kFgWaves];
  __shared__ float red[kFgWaves];
  s = block_merge<kFgWaves>(s, part);
  const float lse_d = soft ? (s.md + fast_log2(s.zd)) * kLn2 : 0.f;
  const float lse_t = KNOWN ? lse_target[r] : (s.mt + fast_log2(s.zt)) * kLn2;
  if (KNOWN) s.it = argmax_target[r];
  settle(s, xrow, vocab);
  if (KNOWN) s.xt = load1(xrow + s.it);

  const bool has_tv = tm.mask >> SPX_LOSS_TV & 1, has_rkl = tm.mask >> SPX_LOSS_RKL & 1, has_jsd = tm.mask >> SPX_LOSS_JSD & 1;
  // (both walks form the probabilities alike, so that q <= p of tv resolves alike)
  const float cd = -lse_d * kLog2e, ct = -lse_t * kLog2e;
  float sum_r = 0.f, sum_j = 0.f, ext_j = 0.f, sum_v = 0.f, ext_v = 0.f;
  if (soft && (has_tv || has_rkl || has_jsd)) {
    pin();
#pragma unroll
    for (int k = 0; k < kFgChunks; ++k) {
      if (tid + k * kFgThreads >= nchunks) continue;
      float x[8], y[8], none = 0.f;
      unpack(xr[k], x);
      unpack(yr[k], y);
      if (has_tv) {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const float dp = fast_exp2(fmaf(x[i], kLog2e, cd)), tp = fast_exp2(fmaf(y[i], kLog2e, ct));
          sum_v += fminf(dp, tp);
          ext_v += dp <= tp ? dp : 0.f;
        }
      }
      if (has_rkl) add_second<SPX_LOSS_RKL>(sum_r, none, x, y, lse_d, lse_t);
      if (has_jsd) add_second<SPX_LOSS_JSD>(sum_j, ext_j, x, y, lse_d, lse_t);
    }
    if (has_tv) { sum_v = block_sum<kFgWaves>(sum_v, red); ext_v = block_sum<kFgWaves>(ext_v, red); }
    if (has_rkl) sum_r = block_sum<kFgWaves>(sum_r, red);
    if (has_jsd) { sum_j = block_sum<kFgWaves>(sum_j, red); ext_j = block_sum<kFgWaves>(ext_j, red); }
  }
  if (tid == 0) {
    const float of[5] = {(KNOWN ? s.at : s.at / s.zt) - lse_t + lse_d, sum_r, 0.5f * (sum_j + ext_j), lse_d - s.xt, 1.f - sum_v};
    float first = 0.f;
    int64_t t = 0;
#pragma unroll
    for (int op = 0; op < 5; ++op)
      if (tm.mask >> op & 1) {
        const float v = soft ? of[op] : 0.f;
        if (t == 0) first = v;
        else loss[t * rows + r] = v;
        ++t;
      }
    store_row<KNOWN>(r, s, first, lse_d, lse_t, loss, lse_draft, lse_target, argmax_draft, argmax_target, sa);
  }
  if (!live) return;
  uint16_t* grow = grad + (int64_t)slot * ld_grad;
  // every term's gradient is the draft probability times a factor, less w_kl times the target's and w_ce at the label
  const float w_ce = tm.w[SPX_LOSS_CE], w_kl = tm.w[SPX_LOSS_KL], w_tv = has_tv ? tm.w[SPX_LOSS_TV] : 0.f;
  const float base_f = w_ce + (KL ? w_kl : 0.f), above = fmaf(w_tv, ext_v, base_f), below = above - w_tv;
  const int label = s.it;
  pin();
#pragma unroll
  for (int k = 0; k < kFgChunks; ++k) {
    const int c = tid + k * kFgThreads;
    if (c >= nchunks) continue;
    float x[8], y[8], o[8];
    unpack(xr[k], x);
    unpack(yr[k], y);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float dp = fast_exp2(fmaf(x[i], kLog2e, cd)), tp = fast_exp2(fmaf(y[i], kLog2e, ct));
      o[i] = dp * (dp <= tp ? below : above);
      if (KL) o[i] = fmaf(-w_kl, tp, o[i]);
    }
    if (has_rkl || has_jsd) {
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const float ldp = x[i] - lse_d, ltp = y[i] - lse_t, dp = fast_exp2(fmaf(x[i], kLog2e, cd));
        if (has_rkl) o[i] = fmaf(tm.w[SPX_LOSS_RKL] * dp, ldp - ltp - sum_r, o[i]);
        if (has_jsd) o[i] = fmaf(0.5f * tm.w[SPX_LOSS_JSD] * dp, mix_logs(ldp, ltp).p - sum_j, o[i]);
      }
    }
    if (c == label >> 3) {
#pragma unroll
      for (int i = 0; i < 8; ++i) o[i] -= i == (label & 7) ? w_ce : 0.f;
    }
    store8_vec<uint16_t>(grow + ((int64_t)c << 3), o);
  }
}

// ---- forward with the d2t gather, pipelined ------------------------------------------------------
// The first step of a TTT loop whose targets arrive as full-vocabulary verifier logits: the same row pass
// as loss_fwd_kernel<.., GATHER> (gather through d2t, both online soft-maxes, KL or CE, both arg-maxes,
// the gathered row written out, the acceptance chain), arranged so that nothing waits for memory:
//   * the draft ids are walked in tiles of 2048; the ascending span [lo, hi) of the full row that a tile
//     maps to is known for every tile before the loop starts (a table in LDS, built from 2 table reads
//     per tile), so the span of tile t + 2 and that tile's piece of the draft row are requested -- global
//     -> LDS directly, no registers -- while tile t is reduced: a ring of three slots, one workgroup
//     barrier per tile, a fixed number of loads per wave and tile so that one s_waitcnt constant tells
//     when a slot has landed;
//   * picking element i + d2t[i] out of the staged span is done with lane = id (consecutive lanes read
//     LDS addresses a few bytes apart: about two lanes per bank) instead of lane = chunk of 8 ids (lanes
//     64 bytes apart: 16 lanes per bank); each wave then turns its 512 picks into 8-id chunks through a
//     1 KB LDS strip of its own, so the gathered row is written 16 bytes per lane;
//   * a tile whose span does not fit a slot (a table that is not spread evenly) reads its elements
//     from global memory directly, as the general kernel does.
// bf16 rows, 16-byte aligned, KL or CE; everything else stays with loss_fwd_kernel<.., GATHER>.
constexpr int kPipeTileIds = kLossThreads * 8;        // 2048 draft ids per tile
constexpr int kPipeSpanLoads = 5;                     // 1 KB wave-loads per wave and span
constexpr int kPipeCap = kPipeSpanLoads * kLossWaves * 512;  // 10240 elements of the full row per slot
constexpr int kPipeSlotBytes = kPipeCap * 2 + kPipeTileIds * 2;  // span + the tile's draft-row piece
constexpr int kPipeSlots = 3;
constexpr int kPipeMaxTiles = 128;                    // draft vocabulary <= 262144
constexpr int kPipeOffY = kPipeSlots * kPipeSlotBytes;  // byte offsets inside the dynamic LDS block
constexpr int kPipeOffSpan = kPipeOffY + kPipeTileIds * 2;
constexpr int kPipeSmem = kPipeOffSpan + kPipeMaxTiles * 2 * 4;
static_assert(2 * kPipeSmem + 1024 <= 160 * 1024, "two workgroups per compute unit");

template <int OP>
__global__ __launch_bounds__(kLossThreads) void loss_fwd_gather_pipe_kernel(
    const uint16_t* __restrict__ logits, int64_t ld_logits, const uint16_t* __restrict__ targets,
    int64_t ld_targets, int64_t vocab, float* __restrict__ loss, float* __restrict__ lse_draft,
    float* __restrict__ lse_target, float* __restrict__ extra, int32_t* __restrict__ argmax_draft,
    int32_t* __restrict__ argmax_target, StepArgs sa) {
  extern __shared__ __attribute__((aligned(16))) uint8_t psm[];
  uint16_t* const ybuf = reinterpret_cast<uint16_t*>(psm + kPipeOffY);  // [4 waves][512]
  int* const span = reinterpret_cast<int*>(psm + kPipeOffSpan);         // [tiles][2]: lo, length (-1: direct)
  const int64_t r = blockIdx.x;
  const uint16_t* xrow = logits + r * ld_logits;
  const uint16_t* yrow = targets + r * ld_targets;
  uint16_t* grow = sa.gathered ? reinterpret_cast<uint16_t*>(sa.gathered) + r * sa.ld_gathered : nullptr;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int ntiles = (int)((vocab + kPipeTileIds - 1) / kPipeTileIds);

  for (int t = tid; t < ntiles; t += kLossThreads) {
    const int64_t i0 = (int64_t)t * kPipeTileIds, i1 = min(vocab, i0 + kPipeTileIds) - 1;
    int64_t lo = i0 + sa.d2t[i0], hi = i1 + sa.d2t[i1] + 1;
    lo = max((int64_t)0, min(lo, sa.vt)) & ~(int64_t)7;
    hi = max(lo, min(hi, sa.vt));
    span[2 * t] = (int)lo;
    span[2 * t + 1] = (hi - lo <= kPipeCap) ? (int)(hi - lo) : -1;
  }
  __syncthreads();

  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)psm;
  // Per-lane byte offsets that never change: every tile moves the BASE of its buffer resources (scalar
  // arithmetic) and sets their size to what the tile may touch, so lanes past a span's end, past the
  // draft vocabulary or past the table fetch nothing and deliver zeros, without a vector instruction
  int span_voff[kPipeSpanLoads];
#pragma unroll
  for (int k = 0; k < kPipeSpanLoads; ++k) span_voff[k] = ((k * kLossWaves + wave) * 512 + lane * 8) * 2;
  const int x_voff = (wave * 512 + lane * 8) * 2;
  const int off_voff = lane * 8;
  // tile u into slot u % 3: kPipeSpanLoads wave-loads of the span (the four waves interleaved) and one of
  // this wave's 512 ids of the draft row -- always six loads, also for a tile past the last one (resources
  // of size zero)
  auto request = [&](int u) __attribute__((always_inline)) {
    const bool live = u < ntiles;
    const int lo = live ? span[2 * u] : 0, len = live ? span[2 * u + 1] : -1;
    // (sizes in whole 16-byte pieces: a load that straddles the end of a resource delivers nothing at
    // all, and the rows' pitch, a multiple of 8 elements, covers the rounding)
    const u32x4 yres = make_rsrc(yrow + lo, len > 0 ? (uint32_t)((len + 7) & ~7) * 2u : 0u);
    const int64_t x0 = (int64_t)u * kPipeTileIds;
    const u32x4 xres = make_rsrc(xrow + x0,
                                 live ? (uint32_t)((min((int64_t)kPipeTileIds, vocab - x0) + 7) & ~(int64_t)7) * 2u : 0u);
    const uint32_t dst = lds0 + (u % kPipeSlots) * kPipeSlotBytes;
#pragma unroll
    for (int k = 0; k < kPipeSpanLoads; ++k)
      load_to_lds16<0>(yres, dst + (k * kLossWaves + wave) * 1024, span_voff[k], 0);
    load_to_lds16<0>(xres, dst + kPipeCap * 2 + wave * 1024, x_voff, 0);
  };
  // The table entries of this lane's 8 picks of tile u (lane = id inside the wave's 512 ids; the low
  // words of the int64 offsets: |d2t| < 2^31; 0 past the vocabulary).  The loads are statements the
  // compiler does not look into, like the span requests: it would otherwise guard their first use with a
  // wait that also covers every span request issued since (it does not count those), and the ring would
  // run one tile deep.  Their registers must not be read before `landed` has named them.
  auto load_offsets = [&](int u, int (&d)[8]) __attribute__((always_inline)) {
    const int64_t w0 = (int64_t)u * kPipeTileIds + wave * 512;
    const u32x4 dres = make_rsrc(sa.d2t + min(w0, vocab), (uint32_t)max((int64_t)0, min((int64_t)512, vocab - w0)) * 8u);
#define SPX_LOAD_OFF(K) \
    asm volatile("buffer_load_dword %0, %1, %2, 0 offen offset:%3" : "=v"(d[K]) : "v"(off_voff), "s"(dres), "n"(K * 512) : "memory")
    SPX_LOAD_OFF(0); SPX_LOAD_OFF(1); SPX_LOAD_OFF(2); SPX_LOAD_OFF(3);
    SPX_LOAD_OFF(4); SPX_LOAD_OFF(5); SPX_LOAD_OFF(6); SPX_LOAD_OFF(7);
#undef SPX_LOAD_OFF
  };
  // all vector-memory operations but the newest six have completed; d is what the wait releases.
  // (No branch may stand between a load_offsets and the `landed` that names its registers: a merge of
  // two paths lets the compiler copy the registers, and a copy made before the wait copies stale data.)
  auto landed = [&](int (&d)[8]) __attribute__((always_inline)) {
    asm volatile("s_waitcnt vmcnt(6)"
                 : "+v"(d[0]), "+v"(d[1]), "+v"(d[2]), "+v"(d[3]), "+v"(d[4]), "+v"(d[5]), "+v"(d[6]), "+v"(d[7])
                 :: "memory");
  };

  RowStats s = no_stats();

  // One tile.  Order of the vector-memory operations (they complete in order): offsets(0), slot(0),
  // slot(1), and per tile t: offsets(t + 1), the gathered row's store of t, slot(t + 2) -- every tile,
  // also those past the last one, whose loads fetch nothing.  At the top of tile t the six newest are
  // slot(t + 1): waiting for all but six says offsets(t) and slot(t) are in
  auto tile = [&](int t, int (&cur)[8], int (&nxt)[8]) __attribute__((always_inline)) {
    landed(cur);
    __syncthreads();  // every wave's part of slot(t) has landed, every wave is done with slot(t - 1)
    load_offsets(t + 1, nxt);
    const bool live = t < ntiles;
    const int lo = live ? span[2 * t] : 0, len = live ? span[2 * t + 1] : -1;
    const uint8_t* const slot = psm + (t % kPipeSlots) * kPipeSlotBytes;
    const uint16_t* const buf = reinterpret_cast<const uint16_t*>(slot);
    const int64_t wbase = (int64_t)t * kPipeTileIds + wave * 512;
    uint16_t* const ystrip = ybuf + wave * 512;
    // (32-bit arithmetic: ids and columns are below 2^30 here)
    const int id0 = (int)wbase + lane, nvocab = (int)vocab, nvt = (int)sa.vt;
    const unsigned ulen = len > 0 ? (unsigned)len : 0u;
    const int delta = id0 - lo;
    bool need = false;  // some pick of this lane is not in the staged span
    int rel[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      rel[k] = cur[k] + delta + 64 * k;  // column - lo
      const bool staged = (unsigned)rel[k] < ulen;
      need |= !staged;
      ystrip[lane + 64 * k] = buf[staged ? rel[k] : 0];
    }
    if (__any(need)) {  // (wave-uniform: the common case issues no global load here)
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        const int j = rel[k] + lo;
        if ((id0 + 64 * k < nvocab) && !((unsigned)rel[k] < ulen))  // -inf: a column outside the full row
          ystrip[lane + 64 * k] = ((unsigned)j < (unsigned)nvt) ? yrow[j] : (uint16_t)0xff80;
      }
    }
    // the strip is private to the wave: its own writes, in order, then its own reads
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    const int64_t base = wbase + lane * 8;
    const u32x4 yraw = *reinterpret_cast<const u32x4*>(ystrip + lane * 8);
    const u32x4 xraw = *reinterpret_cast<const u32x4*>(slot + kPipeCap * 2 + wave * 1024 + lane * 16);
    if (grow && base + 8 <= vocab) st16(grow + base, yraw);
    request(t + 2);
    if (base < vocab) {
      float x[8], y[8];
      x[0] = bf16_lo(xraw.x); x[1] = bf16_hi(xraw.x); x[2] = bf16_lo(xraw.y); x[3] = bf16_hi(xraw.y);
      x[4] = bf16_lo(xraw.z); x[5] = bf16_hi(xraw.z); x[6] = bf16_lo(xraw.w); x[7] = bf16_hi(xraw.w);
      y[0] = bf16_lo(yraw.x); y[1] = bf16_hi(yraw.x); y[2] = bf16_lo(yraw.y); y[3] = bf16_hi(yraw.y);
      y[4] = bf16_lo(yraw.z); y[5] = bf16_hi(yraw.z); y[6] = bf16_lo(yraw.w); y[7] = bf16_hi(yraw.w);
      if (base + 8 > vocab) {  // the draft vocabulary ends inside this chunk (the last tile only)
        const uint32_t yw[4] = {yraw.x, yraw.y, yraw.z, yraw.w};
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          if (base + i < vocab) {
            if (grow) grow[base + i] = (uint16_t)(yw[i >> 1] >> (16 * (i & 1)));
          } else {
            x[i] = kNegBig; y[i] = kNegBig;  // tail padding, like load8_guard
          }
        }
      }
      float cx = x[0], cy = y[0];
#pragma unroll
      for (int i = 1; i < 8; ++i) { cx = fmaxf(cx, x[i]); cy = fmaxf(cy, y[i]); }
      if (cx > s.bd) {  // strict: an earlier chunk of this thread keeps a tie
        int k = 7;
#pragma unroll
        for (int i = 6; i >= 0; --i) k = (x[i] == cx) ? i : k;
        s.bd = cx; s.id = (int)base + k;
      }
      if (cy > s.bt) {
        int k = 7;
        float xv = x[7];
#pragma unroll
        for (int i = 6; i >= 0; --i) {
          const bool hit = y[i] == cy;
          k = hit ? i : k;
          xv = hit ? x[i] : xv;
        }
        s.bt = cy; s.it = (int)base + k; s.xt = xv;
      }
      {
        const float cxs = cx * kLog2e;
        float mn = s.md, z = s.zd;
        if (cxs > mn) {
          z *= fast_exp2(mn - cxs);
          mn = cxs;
        }
#pragma unroll
        for (int i = 0; i < 8; ++i) z += fast_exp2(fmaf(x[i], kLog2e, -mn));
        s.zd = z; s.md = mn;
      }
      if (OP != SPX_LOSS_CE) {
        float mn = fmaxf(s.mt, cy * kLog2e);
        float rs = fast_exp2(s.mt - mn);
        float z = s.zt * rs, a = s.at * rs;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          float e = fast_exp2(fmaf(y[i], kLog2e, -mn));
          z += e;
          a = fmaf(e, y[i] - x[i], a);
        }
        s.zt = z; s.at = a; s.mt = mn;
      }
    }
  };

  int off_a[8], off_b[8];
  load_offsets(0, off_a);
  request(0);
  request(1);
  // two tiles per trip: the two register sets swap roles, nothing is copied; an odd tile count runs one
  // tile past the end (all of its work is switched off by its ids)
  for (int t = 0; t < ntiles; t += 2) {
    tile(t, off_a, off_b);
    tile(t + 1, off_b, off_a);
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the requests past the end still write LDS
  __syncthreads();

  __shared__ RowStats part[kLossWaves];
  s = block_merge<kLossWaves>(s, part);
  settle(s, xrow, vocab);
  const float lse_d = (s.md + fast_log2(s.zd)) * kLn2;
  const float lse_t = (OP != SPX_LOSS_CE) ? (s.mt + fast_log2(s.zt)) * kLn2 : 0.f;
  float row_loss;
  if (OP == SPX_LOSS_KL) row_loss = s.at / s.zt - lse_t + lse_d;
  else row_loss = lse_d - s.xt;
  if (tid == 0) {
    loss[r] = row_loss;
    lse_draft[r] = lse_d;
    extra[r] = (OP == SPX_LOSS_KL) ? row_loss : 0.f;
    if (argmax_draft) argmax_draft[r] = s.id;
    lse_target[r] = lse_t;
    if (argmax_target) argmax_target[r] = s.it;
    if (sa.counts) {
      const bool m = sa.mask ? mask_value(sa.mask, sa.mask_kind, r) != 0.f : true;
      const bool was = sa.prev ? mask_value(sa.prev, sa.prev_kind, r) != 0.f : true;
      const bool now = was && (s.id == s.it);
      if (m && now) atomicAdd(&sa.counts[0], 1);
      if (m) atomicAdd(&sa.counts[1], 1);
      if (was) atomicAdd(&sa.counts[2], 1);
      if (sa.prev) store_flag(sa.prev, sa.prev_kind, r, now);
    }
  }
}

// ---- backward --------------------------------------------------------------
template <typename T, int OP, bool VEC>
__global__ __launch_bounds__(kLossThreads) void loss_bwd_kernel(
    const T* __restrict__ logits, int64_t ld_logits, const T* __restrict__ targets,
    int64_t ld_targets, int64_t vocab, const float* __restrict__ lse_draft,
    const float* __restrict__ lse_target, const float* __restrict__ extra,
    const int32_t* __restrict__ argmax_target, const float* __restrict__ row_grad,
    const float* __restrict__ scale, T* __restrict__ grad, int64_t ld_grad,
    const int32_t* __restrict__ row_map) {
  const int64_t r = blockIdx.x;
  const int tid = threadIdx.x;
  const int64_t nchunks = (vocab + 7) >> 3;
  // (several workgroups share a row where there are few rows: blockIdx.y)
  const int64_t c_first = (int64_t)blockIdx.y * kLossThreads + tid, c_stride = (int64_t)gridDim.y * kLossThreads;
  // with a row map the gradient of row r goes to row row_map[r] and rows mapped to -1 (zero gradient)
  // are not written: the live rows packed to the front
  int64_t dst = r;
  if (row_map) {
    dst = row_map[r];
    if (dst < 0) return;
  }
  T* grow = grad + dst * ld_grad;
  float g = row_grad[r];
  if (scale) g *= *scale;
  if (g == 0.f) {
    const float z[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    for (int64_t c = c_first; c < nchunks; c += c_stride) store8<T, VEC>(grow, c << 3, vocab, z);
    return;
  }
  const T* xrow = logits + r * ld_logits;
  const T* yrow = (OP != SPX_LOSS_CE) ? targets + r * ld_targets : nullptr;
  const float lse_d = lse_draft[r];
  const float lse_t = (OP != SPX_LOSS_CE) ? lse_target[r] : 0.f;
  const float ex = (OP == SPX_LOSS_RKL || OP == SPX_LOSS_JSD || OP == SPX_LOSS_TV) ? extra[r] : 0.f;
  const int label = (OP == SPX_LOSS_CE) ? argmax_target[r] : -1;
  const float cd = -lse_d * kLog2e, ct = -lse_t * kLog2e;

  for (int64_t c = c_first; c < nchunks; c += c_stride) {
    const int64_t base = c << 3;
    float x[8], y[8];
    load8<T, VEC>(xrow, base, vocab, x);
    if (OP != SPX_LOSS_CE) load8<T, VEC>(yrow, base, vocab, y);
    float o[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      if (OP == SPX_LOSS_CE) {
        float dp = fast_exp2(fmaf(x[i], kLog2e, cd));
        o[i] = g * (dp - (((int)base + i) == label ? 1.f : 0.f));
      } else if (OP == SPX_LOSS_KL) {
        float dp = fast_exp2(fmaf(x[i], kLog2e, cd));
        float tp = fast_exp2(fmaf(y[i], kLog2e, ct));
        o[i] = g * (dp - tp);
      } else {
        if (OP == SPX_LOSS_RKL) {
          o[i] = g * fast_exp2((x[i] - lse_d) * kLog2e) * ((x[i] - lse_d) - (y[i] - lse_t) - ex);
          continue;
        }
        // same expressions as the forward's second walk, so that the
        // q <= p comparison of tv resolves identically in both directions
        const float ldp = x[i] - lse_d, ltp = y[i] - lse_t, dp = fast_exp2(ldp * kLog2e);
        if (OP == SPX_LOSS_JSD) o[i] = g * 0.5f * dp * (mix_logs(ldp, ltp).p - ex);
        else o[i] = -g * dp * ((dp <= fast_exp2(ltp * kLog2e) ? 1.f : 0.f) - ex);
      }
    }
    store8<T, VEC>(grow, base, vocab, o);
  }
}

// ---- gather through the d2t offset table -------------------------------------
template <typename T>
__global__ __launch_bounds__(256) void vocab_gather_kernel(
    const T* __restrict__ full, int64_t ld_full, const int64_t* __restrict__ d2t,
    T* __restrict__ out, int64_t ld_out, int64_t vd, int64_t vt, T neg_inf_bits) {
  const int64_t r = blockIdx.y;
  const T* src = full + r * ld_full;
  T* dst = out + r * ld_out;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < vd; i += (int64_t)gridDim.x * 256) {
    int64_t j = i + d2t[i];
    dst[i] = (j >= 0 && j < vt) ? src[j] : neg_inf_bits;
  }
}

constexpr int kReduceThreads = 1024;

__device__ __forceinline__ float block_sum_f(float v, float* lds) {
  v = wave_sum(v);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) lds[threadIdx.x >> 6] = v;
  __syncthreads();
  float t = 0.f;
  for (int w = 0; w < kReduceThreads / 64; ++w) t += lds[w];
  return t;
}
__device__ __forceinline__ int block_sum_i(int v, int* lds) {
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) v += __shfl_xor(v, m, 64);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) lds[threadIdx.x >> 6] = v;
  __syncthreads();
  int t = 0;
  for (int w = 0; w < kReduceThreads / 64; ++w) t += lds[w];
  return t;
}

__global__ __launch_bounds__(kReduceThreads) void ttt_step_reduce_kernel(
    const float* __restrict__ loss, const int32_t* __restrict__ pred,
    const int32_t* __restrict__ tgt, const void* __restrict__ mask, int mask_kind,
    void* prev, int prev_kind, int64_t rows, float weight, float* __restrict__ out,
    float* __restrict__ row_weight, const int32_t* __restrict__ counts,
    float factor, const float* __restrict__ total_in, float* __restrict__ total_out) {
  __shared__ float fl[kReduceThreads / 64];
  __shared__ int il[kReduceThreads / 64];
  float lsum = 0.f, msum = 0.f;
  int full_total = 0, correct = 0, cond_total = 0;
  // counts != nullptr: the acceptance chain was done row by row in the loss pass (StepArgs);
  // only the masked mean is left here and the counts are copied out
  for (int64_t r = threadIdx.x; r < rows; r += kReduceThreads) {
    float m = mask ? mask_value(mask, mask_kind, r) : 1.f;
    if (!counts) {
      bool was = prev ? (mask_value(prev, prev_kind, r) != 0.f) : true;
      bool hit = pred[r] == tgt[r];
      bool now = was && hit;
      cond_total += was ? 1 : 0;
      if (prev) store_flag(prev, prev_kind, r, now);
      if (m != 0.f) { full_total += 1; correct += now ? 1 : 0; }
    }
    lsum = fmaf(loss[r], m, lsum);
    msum += m;
  }
  lsum = block_sum_f(lsum, fl);
  msum = block_sum_f(msum, fl);
  if (!counts) {
    full_total = block_sum_i(full_total, il);
    correct = block_sum_i(correct, il);
    cond_total = block_sum_i(cond_total, il);
  } else {
    correct = counts[0]; full_total = counts[1]; cond_total = counts[2];
  }
  const float inv = weight / (msum + 1e-5f);
  if (threadIdx.x == 0) {
    out[0] = lsum * inv;
    out[1] = (float)correct;
    out[2] = (float)full_total;
    out[3] = (float)correct;
    out[4] = (prev || counts) ? (float)cond_total : (float)rows;
    out[5] = msum;
    if (total_out) {  // the term in the loss: what a handful of one-element kernels did
      const float part = lsum * inv * factor;
      out[6] = part;
      out[7] = 1.f;
      *total_out = total_in ? *total_in + part : part;
    }
  }
  if (row_weight) {
    for (int64_t r = threadIdx.x; r < rows; r += kReduceThreads) {
      float m = mask ? mask_value(mask, mask_kind, r) : 1.f;
      row_weight[r] = m * inv;
    }
  }
}

// The step's scalars of a loss of several terms, acceptance chain done (spx_ttt_step_terms): one pass over the mask
__global__ __launch_bounds__(kReduceThreads) void ttt_step_terms_kernel(
    const float* __restrict__ loss, LossTerms tm, const void* __restrict__ mask, int mask_kind, int64_t rows,
    float weight, const int32_t* __restrict__ counts, const float* __restrict__ total_in,
    float* __restrict__ total_out, float* __restrict__ out, float* __restrict__ row_weight) {
  __shared__ float fl[kReduceThreads / 64];
  const int n = __popc(tm.mask);
  float sums[5] = {0.f, 0.f, 0.f, 0.f, 0.f}, msum = 0.f;
  for (int64_t r = threadIdx.x; r < rows; r += kReduceThreads) {
    const float m = mask ? mask_value(mask, mask_kind, r) : 1.f;
#pragma unroll
    for (int t = 0; t < 5; ++t)
      if (t < n) sums[t] = fmaf(loss[t * rows + r], m, sums[t]);
    msum += m;
  }
  msum = block_sum_f(msum, fl);
#pragma unroll
  for (int t = 0; t < 5; ++t)
    if (t < n) sums[t] = block_sum_f(sums[t], fl);
  const float inv = weight / (msum + 1e-5f);
  if (threadIdx.x == 0) {
    float total = 0.f;
    int t = 0;
#pragma unroll
    for (int op = 0; op < 5; ++op) {
      float mean = 0.f;
      if (tm.mask >> op & 1) {
#pragma unroll
        for (int u = 0; u < 5; ++u) mean = u == t ? sums[u] * inv : mean;
        total = fmaf(tm.w[op], mean, total);
        ++t;
      }
      out[8 + op] = mean;
      out[13 + op] = 1.f;
    }
    out[0] = out[6] = total;
    out[1] = out[3] = (float)counts[0];
    out[2] = (float)counts[1];
    out[4] = (float)counts[2];
    out[5] = msum;
    out[7] = 1.f;
    *total_out = total_in ? *total_in + total : total;
  }
  for (int64_t r = threadIdx.x; r < rows; r += kReduceThreads)
    row_weight[r] = (mask ? mask_value(mask, mask_kind, r) : 1.f) * inv;
}

// The rows a mask leaves, in order, and three zeroed counters for the loss pass behind it.
__global__ __launch_bounds__(1024) void mask_row_map_kernel(const void* __restrict__ mask, int mask_kind, int rows,
                                                            int32_t* __restrict__ row_map,
                                                            int32_t* __restrict__ count,
                                                            int32_t* __restrict__ row_of, int32_t* __restrict__ zero3) {
  if (zero3 && threadIdx.x < 3) zero3[threadIdx.x] = 0;
  pack_row_map([&](int r) { return mask_value(mask, mask_kind, r) != 0.f; }, rows, row_map, count, row_of);
}

// ---- all steps of a TTT loop at one target row -------------------------------------------------------
// Draft row t of step k meets target row t + k: one workgroup takes target row r and its draft rows (k, r - k), k = 0, 1, ..
// one after the other, the target row in registers throughout: it is read once instead of once a step, and while a
// step's gradient leaves, the next step's row is requested into the registers that it frees, so that the arithmetic of one
// row runs beside the traffic of its neighbour.  Where r < k there is no such draft row, and the workgroup takes row T - k + r
// instead, one of the k last, which have no target: its arg-max is a draft token like any other.  So every
// (step, row) is met once.
//   loss, tokens, hits, row_slot, row_weight: [steps][T] (a loss of several terms: [term][steps][T]), indexed by draft row;
//   grad and slot_row by slot, K a live target: slot = rank of the target among the live ones * K + k (k > r: a row of zeros,
//   of weight zero).
// TERMS: a weighted sum of kl, ce and tv, as loss_terms_grad_kernel takes it (OP: KL if that is one of them, else CE): a second
// walk over the registers where tv is a term, and the gradient of the sum.  (rkl and jsd need registers that are not there.)
// What a step needs of the target row is its probabilities alone (kl: sum p (y - top) once, less sum p (x - top) of each step;
// the difference is taken thread by thread, before it is added up, and from the row's largest logit on, so that no sum of
// large terms cancels: mean error against 64 bits 0.97 - 1.03 of that of sum p (y - x), 0 for equal rows either way).  So they
// are formed once a row and held, in 32 bits: with the draft row's packed chunks 96 of the 128 registers that four waves to a
// SIMD leave, wherefore chunk numbers are formed again each time.
// kl, 7 steps of 4096 rows of 32000, 70 % live: a pass a step 1002 us, exponentials of both rows at each step 724, so 663 (5.2
// TB/s; ce 650, its traffic).  3 steps of 512 rows 52.2 -> 46.0, 7 of 3001 rows of 8192 217 -> 195; 5 of 1999 rows without
// gradient 199 -> 182, 3 of 333 rows of 1000 with it 16.3 -> 15.1; {"ce": 0.1, "tv": 0.9}, 3 steps of 3001 320 -> 298.
// Without gradient it is bound by its instructions (77 % of the issue slots taken).  The waves' results merged by lane moves, and
// the place of a draft row's largest looked for by one thread (kLook), on another box: 5 steps of 1999 rows 204 -> 192, ce 180 -> 170,
// two terms 268 -> 248; with gradients, the moves alone: 3 steps of 512 rows 48.1 -> 45.7, 7 of 3001 rows of 8192 183 -> 155, 7 of 4096
// of 32000 685 -> 681, ce 660 -> 651, two terms 330 -> 333 (its two runs 322 and 344).
struct StepsArgs {
  const uint16_t* logits[SPX_LOSS_STEPS_MAX];  // [T, vocab] each
  int64_t ld;
  const uint16_t* targets;  // null: argmax_target is known (ce)
  int64_t ld_targets;
  const int32_t* argmax_target;
  int T, vocab, steps, k0, k1;  // this launch: steps k0 .. k1 - 1 of `steps`
  int masked_first;             // GRAD: the first step's masked rows are formed, too
  LossTerms tm;                 // TERMS
  const void* mask;
  int mask_kind;
  const float* inv;             // [steps]: weight of a step's masked mean over the sum of its mask
  const int32_t* row_map;       // [T]: rank of a live target, -1
  const int32_t* live;          // live targets
  float* loss;
  int64_t* tokens;
  uint8_t* hits;
  int32_t* row_slot;            // GRAD ...
  int32_t* slot_row;
  int32_t* slots;
  float* row_weight;
  uint16_t* grad;
  int64_t ld_grad;
};

template <int OP, bool GRAD, bool TERMS = false>
__global__ __launch_bounds__(kFgThreads) __attribute__((amdgpu_waves_per_eu(4, 4))) void loss_steps_kernel(StepsArgs a) {
  constexpr bool kY = OP == SPX_LOSS_KL || TERMS;  // the target's probabilities are needed at every step
  // Which chunk of a draft row holds its largest, and where in it only that chunk's thread looks, in memory, instead of every thread
  // in every chunk (12 % of a step's instructions).  Not where gradients are: its wait is for their stores, too.
  constexpr bool kLook = !GRAD;
  const int r = blockIdx.x, tid = threadIdx.x, T = a.T;
  const int nchunks = a.vocab >> 3;
  const int rank = GRAD ? a.row_map[r] : -1;
  const bool live = rank >= 0;
  auto row_of = [&](int k) __attribute__((always_inline)) { return r >= k ? r - k : T - k + r; };
  auto chunk = [&](int j) __attribute__((always_inline)) {  // (formed again each time: held, they would be eight registers)
    int first = tid;
    if (kY) asm volatile("" : "+v"(first));
    return first + j * kFgThreads;
  };
  auto at8 = [](const uint16_t* row, int c) __attribute__((always_inline)) {
    return reinterpret_cast<const uint16_t*>(reinterpret_cast<const char*>(row) + ((uint32_t)c << 4));
  };
  auto unpack = [](u32x4 raw, float (&v)[8]) __attribute__((always_inline)) {
    v[0] = bf16_lo(raw.x); v[1] = bf16_hi(raw.x); v[2] = bf16_lo(raw.y); v[3] = bf16_hi(raw.y);
    v[4] = bf16_lo(raw.z); v[5] = bf16_hi(raw.z); v[6] = bf16_lo(raw.w); v[7] = bf16_hi(raw.w);
  };
  u32x4 xr[kFgChunks], yr[kFgChunks];
  float p[kFgChunks][8];
  const uint16_t* xrow = a.logits[a.k0] + (int64_t)row_of(a.k0) * a.ld;
  const uint16_t* const yrow = a.targets ? a.targets + (int64_t)r * a.ld_targets : nullptr;
  if (a.targets) {
#pragma unroll
    for (int j = 0; j < kFgChunks; ++j) {
      if (j * kFgThreads >= nchunks) break;
      const int c = chunk(j);
      if (c < nchunks) yr[j] = ld16(at8(yrow, c));
    }
  }
#pragma unroll
  for (int j = 0; j < kFgChunks; ++j) {
    if (j * kFgThreads >= nchunks) break;
    const int c = chunk(j);
    if (c < nchunks) xr[j] = ld16(at8(xrow, c));
  }
  struct Part { float z, a, b; int i; };
  __shared__ __attribute__((aligned(16))) Part part[2][kFgWaves];
  __shared__ float second[2][kFgWaves], of_target[kFgThreads];
  int turn = 0;
  // every thread's (maximum, first place of it, sum of 2^(x' - max x'), sum) -> the workgroup's: by lane moves in a wave, then among
  // eight lanes that hold a wave's each (one after the other, an exponential each, the waves' results took 15 % of a step)
  static_assert(kFgWaves == 8, "a wave's results in each lane of eight");
  const auto add = [](float x, float y) { return x + y; };
  const auto higher = [](float x, float y) { return fmaxf(x, y); };
  const auto lower = [](int x, int y) { return min(x, y); };
  auto scale_of = [](float b) __attribute__((always_inline)) { return fmaxf(b * kLog2e, kNegBig); };
  auto reduce = [&](float& best, int& at, float& z, float& sum, bool soft) __attribute__((always_inline)) {
    const float wb = wave_all(best, higher);
    const int i = wave_all(best == wb ? at : 0x7fffffff, lower);
    if (soft) {
      z = wave_all(z * fast_exp2(scale_of(best) - scale_of(wb)), add);
      sum = wave_all(sum, add);
    }
    if ((tid & 63) == 0) part[turn][tid >> 6] = Part{z, sum, wb, i};
    __syncthreads();
    const Part o = part[turn][tid & 7];
    best = eight_all(o.b, higher);
    at = eight_all(o.b == best ? o.i : 0x7fffffff, lower);
    if (soft) {
      const float m = scale_of(best);
      z = m + fast_log2(eight_all(o.z * fast_exp2(scale_of(o.b) - m), add));
      sum = eight_all(o.a, add);
    }
    turn ^= 1;
  };
  auto at_most = [&](int i) __attribute__((always_inline)) { return (uint32_t)i < (uint32_t)a.vocab ? i : 0; };
  auto place_in = [](const float (&x)[8], float of) __attribute__((always_inline)) {
    int k = 7;
#pragma unroll
    for (int i = 6; i >= 0; --i) k = (x[i] == of) ? i : k;
    return k;
  };
  auto largest = [&](const float (&x)[8], int c, float& best, int& at, auto look) __attribute__((always_inline)) {
    float cx = x[0];
#pragma unroll
    for (int i = 1; i < 8; ++i) cx = fmaxf(cx, x[i]);
    if (cx > best) {  // strict: an earlier chunk of this thread keeps a tie
      best = cx;
      at = decltype(look)::value ? c : (c << 3) + place_in(x, cx);
    }
    return cx;
  };
  // max and sum of exponentials of a chunk into a thread's
  auto soften = [&](const float (&x)[8], float cx, float& m, float& z) __attribute__((always_inline)) {
    const float cs = cx * kLog2e;
    if (cs > m) {
      z *= fast_exp2(m - cs);
      m = cs;
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) z += fast_exp2(fmaf(x[i], kLog2e, -m));
  };

  float top = 0.f;  // the target row's largest, see below
  float lt2 = 0.f;  // base-2 log-sum-exp of the target row
  int label;
  if (a.targets) {
    float best = -INFINITY, m = kNegBig, z = 0.f, none = 0.f;
    label = 0x7fffffff;
#pragma unroll
    for (int j = 0; j < kFgChunks; ++j) {
      if (j * kFgThreads >= nchunks) break;
      const int c = chunk(j);
      if (c >= nchunks) continue;
      float y[8];
      unpack(yr[j], y);
      const float cy = largest(y, c, best, label, std::false_type{});
      if (kY) soften(y, cy, m, z);
    }
    reduce(best, label, z, none, kY);
    label = at_most(label);
    lt2 = z;
    // (within 2^119: from a larger one the difference to the type's lowest value would overflow, and times p = 0 be NaN)
    top = fminf(fmaxf(best, -0x1p119f), 0x1p119f);
    if (kY) {
      float sum = 0.f;
#pragma unroll
      for (int j = 0; j < kFgChunks; ++j) {
        if (j * kFgThreads >= nchunks) break;
        if (chunk(j) >= nchunks) continue;
        asm volatile("" : "+v"(yr[j].x), "+v"(yr[j].y), "+v"(yr[j].z), "+v"(yr[j].w));
        float y[8];
        unpack(yr[j], y);
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          p[j][i] = fast_exp2(fmaf(y[i], kLog2e, -lt2));
          sum = fmaf(p[j][i], y[i] - top, sum);
        }
      }
      if (OP == SPX_LOSS_KL) of_target[tid] = sum;
    }
  } else {
    label = a.argmax_target[r];
    if ((uint32_t)label >= (uint32_t)a.vocab) label = 0;
  }
  if (GRAD && r == 0 && tid == 0 && a.k0 == 0) *a.slots = *a.live * a.steps;
  const float mask = mask_value(a.mask, a.mask_kind, r);

  for (int k = a.k0; k < a.k1; ++k) {
    const bool tail = r < k;
    const int t = row_of(k);
    asm volatile("" : "+v"(label));
    // (a masked row's loss enters no mean: behind the first step it is not formed where gradients are)
    const bool soft = !tail && (!GRAD || live || (k == 0 && a.masked_first));
    const bool more = k + 1 < a.k1;
    const uint16_t* const nrow = more ? a.logits[k + 1] + (int64_t)row_of(k + 1) * a.ld : nullptr;
    const int tm = TERMS ? a.tm.mask : 0;
    const bool has_tv = tm >> SPX_LOSS_TV & 1, walk2 = TERMS && soft && has_tv;
    const bool early = more && !(GRAD && live) && !walk2;  // the row is read once: its registers are free chunk by chunk
    float best = -INFINITY, m = kNegBig, z = 0.f, sum = 0.f;
    int at = 0x7fffffff;
    float xt = 0.f;
    if ((OP == SPX_LOSS_CE || TERMS) && tid == 0) xt = load1(xrow + label);
#pragma unroll
    for (int j = 0; j < kFgChunks; ++j) {
      if (j * kFgThreads >= nchunks) break;
      const int c = chunk(j);
      if (c >= nchunks) continue;
      float x[8];
      unpack(xr[j], x);
      if (early) xr[j] = ld16(at8(nrow, c));
      const float cx = largest(x, c, best, at, std::bool_constant<kLook>{});
      if (soft) {
        soften(x, cx, m, z);
        if (OP == SPX_LOSS_KL) {
#pragma unroll
          for (int i = 0; i < 8; ++i) sum = fmaf(p[j][i], x[i] - top, sum);
        }
      }
    }
    if (OP == SPX_LOSS_KL) sum = of_target[tid] - sum;
    reduce(best, at, z, sum, soft);
    float sum_v = 0.f, ext_v = 0.f;
    if (walk2) {
#pragma unroll
      for (int j = 0; j < kFgChunks; ++j) {
        asm volatile("" : "+v"(xr[j].x), "+v"(xr[j].y), "+v"(xr[j].z), "+v"(xr[j].w));
      }
#pragma unroll
      for (int j = 0; j < kFgChunks; ++j) {
        if (j * kFgThreads >= nchunks) break;
        const int c = chunk(j);
        if (c >= nchunks) continue;
        float x[8];
        unpack(xr[j], x);
        if (more && !(GRAD && live)) xr[j] = ld16(at8(nrow, c));
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const float dp = fast_exp2(fmaf(x[i], kLog2e, -z)), tp = p[j][i];
          sum_v += fminf(dp, tp);
          ext_v += dp <= tp ? dp : 0.f;
        }
      }
      sum_v = wave_all(sum_v, add);
      ext_v = wave_all(ext_v, add);
      if ((tid & 63) == 0) { second[0][tid >> 6] = sum_v; second[1][tid >> 6] = ext_v; }
      __syncthreads();  // (the next writes come behind the next step's reduction, its barrier behind these reads)
      sum_v = ext_v = 0.f;
#pragma unroll
      for (int w = 0; w < kFgWaves; ++w) { sum_v += second[0][w]; ext_v += second[1][w]; }
    }
    const int64_t g = (int64_t)k * T + t;
    const bool none = !kLook || (uint32_t)at >= (uint32_t)nchunks;  // (nothing above -inf)
    if (none ? tid == 0 : (at & (kFgThreads - 1)) == tid) {
      int token = kLook ? 0 : at_most(at);
      if (!none) {
        float x[8];
        unpack(ld16(at8(xrow, at)), x);
        token = (at << 3) + place_in(x, best);
      }
      a.tokens[g] = token;
      a.hits[g] = token == label;
    }
    if (tid == 0) {
      const float kl = sum - lt2 * kLn2 + z * kLn2, ce = z * kLn2 - xt;
      if (TERMS) {
        int64_t at_term = g;
        auto put = [&](int op, float v) {
          if (!(tm >> op & 1)) return;
          a.loss[at_term] = soft ? v : 0.f;
          at_term += (int64_t)a.steps * T;
        };
        put(SPX_LOSS_KL, kl);
        put(SPX_LOSS_CE, ce);
        put(SPX_LOSS_TV, 1.f - sum_v);
      } else {
        a.loss[g] = soft ? (OP == SPX_LOSS_KL ? kl : ce) : 0.f;
      }
      if (GRAD) {
        const int slot = live ? rank * a.steps + k : -1;
        a.row_slot[g] = tail ? -1 : slot;
        if (live) a.slot_row[slot] = (int)g;
        a.row_weight[g] = tail ? 0.f : mask * a.inv[k];
      }
    }
    if (GRAD && live) {
      uint16_t* const grow = a.grad + ((int64_t)rank * a.steps + k) * a.ld_grad;
      const float cd = -z;
#pragma unroll
      for (int j = 0; j < kFgChunks; ++j) {  // (the packed chunks are what stays in registers between the passes)
        asm volatile("" : "+v"(xr[j].x), "+v"(xr[j].y), "+v"(xr[j].z), "+v"(xr[j].w));
      }
      // TERMS: every term's gradient is the draft probability times a factor, less w_kl times the target's and w_ce at the label
      const float w_ce = TERMS ? a.tm.w[SPX_LOSS_CE] : 0.f, w_kl = TERMS ? a.tm.w[SPX_LOSS_KL] : 0.f;
      const float w_tv = TERMS && has_tv ? a.tm.w[SPX_LOSS_TV] : 0.f;
      const float base_f = w_ce + (OP == SPX_LOSS_KL ? w_kl : 0.f), above = fmaf(w_tv, ext_v, base_f), below = above - w_tv;
#pragma unroll
      for (int j = 0; j < kFgChunks; ++j) {
        if (OP == SPX_LOSS_KL && !TERMS && j * kFgThreads >= nchunks) break;
        const int c = chunk(j);
        if (c >= nchunks) continue;
        const int base = c << 3;
        float x[8], o[8];
        unpack(xr[j], x);
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const float dp = fast_exp2(fmaf(x[i], kLog2e, cd));
          if (TERMS) {
            const float tp = p[j][i];
            o[i] = dp * (dp <= tp ? below : above);
            if (OP == SPX_LOSS_KL) o[i] = fmaf(-w_kl, tp, o[i]);
          } else if (OP == SPX_LOSS_CE) {
            o[i] = dp - ((base + i) == label ? 1.f : 0.f);
          } else {
            o[i] = dp - p[j][i];
          }
        }
        if (TERMS && c == label >> 3) {
#pragma unroll
          for (int i = 0; i < 8; ++i) o[i] -= i == (label & 7) ? w_ce : 0.f;
        }
        if (tail) {
#pragma unroll
          for (int i = 0; i < 8; ++i) o[i] = 0.f;
        }
        store8_vec<uint16_t>(const_cast<uint16_t*>(at8(grow, c)), o);
        if (more) xr[j] = ld16(at8(nrow, c));
      }
    }
    xrow = nrow;
  }
}

// What the passes of loss_steps_kernel need of the mask: the live targets in order, and for every step the weight of its
// mean over the sum of the mask of its targets (k, k + 1, ..), how many of them are live, and that sum.  One workgroup.
struct StepWeights { float w[SPX_LOSS_STEPS_MAX]; };
__global__ __launch_bounds__(1024) void steps_mask_kernel(const void* __restrict__ mask, int mask_kind, int T, int steps,
                                                          StepWeights weights, int32_t* __restrict__ row_map,
                                                          int32_t* __restrict__ live, float* __restrict__ inv,
                                                          float* __restrict__ msum, int32_t* __restrict__ full,
                                                          int32_t* __restrict__ ticket) {
  __shared__ float fl[16];
  __shared__ int il[16];
  pack_row_map([&](int r) { return mask_value(mask, mask_kind, r) != 0.f; }, T, row_map, live);
  float s = 0.f;
  int n = 0;
  for (int r = steps - 1 + threadIdx.x; r < T; r += 1024) {  // (steps <= T)
    const float v = mask_value(mask, mask_kind, r);
    s += v;
    n += v != 0.f;
  }
  s = block_sum_f(s, fl);
  n = block_sum_i(n, il);
  if (threadIdx.x == 0) {
    *ticket = 0;
    for (int k = steps - 1; k >= 0; --k) {
      if (k < steps - 1) {
        const float v = mask_value(mask, mask_kind, k);
        s += v;
        n += v != 0.f;
      }
      msum[k] = s;
      full[k] = n;
      inv[k] = weights.w[k] / (s + 1e-5f);
    }
  }
}

// Behind the row passes: the acceptance chain along a draft row's steps, every step's masked mean and counts (as
// ttt_step_reduce_kernel leaves them in out[k][8], for several terms ttt_step_terms_kernel in out[k][18]) and the loss.  A thread owns a draft row; the workgroups' partial sums are
// added in their order by the one that arrives last, which resets nothing and waits for nothing.
constexpr int kStepsRows = 256;
__global__ __launch_bounds__(kStepsRows) void steps_total_kernel(
    const float* __restrict__ loss, const uint8_t* __restrict__ hits, const void* __restrict__ mask, int mask_kind,
    void* prev, int prev_kind, int T, int steps, float factor, LossTerms tm, const float* __restrict__ inv, const float* __restrict__ msum,
    const int32_t* __restrict__ full, float* __restrict__ partial, int32_t* __restrict__ ticket, float* __restrict__ out,
    float* __restrict__ total) {
  __shared__ float ls[kStepsRows / 64][SPX_LOSS_STEPS_MAX][5];
  __shared__ int cs[kStepsRows / 64][SPX_LOSS_STEPS_MAX][2];
  __shared__ int last;
  __shared__ float parts[SPX_LOSS_STEPS_MAX];
  const int t = blockIdx.x * kStepsRows + threadIdx.x, wave = threadIdx.x >> 6;
  const int n = tm.mask ? __popc(tm.mask) : 1, values = n + 2;
  bool was = t < T && (!prev || mask_value(prev, prev_kind, t) != 0.f);
  for (int k = 0; k < steps; ++k) {
    float l[5] = {0.f, 0.f, 0.f, 0.f, 0.f};
    bool good = false, chained = false;
    if (t < T - k) {
      const float m = mask_value(mask, mask_kind, t + k);
#pragma unroll
      for (int u = 0; u < 5; ++u)
        if (u < n) l[u] = loss[((int64_t)u * steps + k) * T + t] * m;
      chained = was;
      was = was && hits[(int64_t)k * T + t];
      good = was && m != 0.f;
    }
#pragma unroll
    for (int u = 0; u < 5; ++u)
      if (u < n) {
        l[u] = wave_sum(l[u]);
        if ((threadIdx.x & 63) == 0) ls[wave][k][u] = l[u];
      }
    const int correct = __popcll(__ballot(good)), cond = __popcll(__ballot(chained));
    if ((threadIdx.x & 63) == 0) { cs[wave][k][0] = correct; cs[wave][k][1] = cond; }
  }
  if (prev && t < T) store_flag(prev, prev_kind, t, was);
  __syncthreads();
  if ((int)threadIdx.x < steps) {
    const int k = threadIdx.x;
    int c = 0, d = 0;
    for (int w = 0; w < kStepsRows / 64; ++w) { c += cs[w][k][0]; d += cs[w][k][1]; }
    float* const p = partial + ((int64_t)blockIdx.x * steps + k) * values;
    __hip_atomic_store(p, __int_as_float(c), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(p + 1, __int_as_float(d), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    for (int u = 0; u < n; ++u) {
      float l = 0.f;
      for (int w = 0; w < kStepsRows / 64; ++w) l += ls[w][k][u];
      __hip_atomic_store(p + 2 + u, l, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
  }
  __threadfence();
  __syncthreads();
  if (threadIdx.x == 0)
    last = __hip_atomic_fetch_add(ticket, 1, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT) == (int)gridDim.x - 1;
  __syncthreads();
  if (!last) return;
  if ((int)threadIdx.x < steps) {
    const int k = threadIdx.x;
    float l[5] = {0.f, 0.f, 0.f, 0.f, 0.f};
    int c = 0, d = 0;
    for (int b = 0; b < (int)gridDim.x; ++b) {
      const float* const p = partial + ((int64_t)b * steps + k) * values;
      c += __float_as_int(__hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
      d += __float_as_int(__hip_atomic_load(p + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
#pragma unroll
      for (int u = 0; u < 5; ++u)
        if (u < n) l[u] += __hip_atomic_load(p + 2 + u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    float* const o = out + (tm.mask ? 18 : 8) * k;
    float sum = l[0] * inv[k];
    if (tm.mask) {
      sum = 0.f;
      int u = 0;
#pragma unroll
      for (int op = 0; op < 5; ++op) {
        float mean = 0.f;
        if (tm.mask >> op & 1) {
#pragma unroll
          for (int v = 0; v < 5; ++v) mean = v == u ? l[v] * inv[k] : mean;
          sum = fmaf(tm.w[op], mean, sum);
          ++u;
        }
        o[8 + op] = mean;
        o[13 + op] = 1.f;
      }
    }
    o[0] = sum;
    o[1] = o[3] = (float)c;
    o[2] = (float)full[k];
    o[4] = (float)d;
    o[5] = msum[k];
    o[6] = parts[k] = sum * factor;
    o[7] = 1.f;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    float sum = parts[0];
    for (int k = 1; k < steps; ++k) sum += parts[k];
    *total = sum;
  }
}

// Draft tokens (int64): the known arg-maxes of the first n rows widened, the arg-max (first index of the
// maximum) of the rows behind them, one workgroup each.  One launch for a conversion, an arg-max pass over few
// rows, another conversion and a concatenation.  A handful of rows is a chain of loads: with 1024 threads to a row
// of 32000 it is four long instead of sixteen (four rows behind 1995, cold: 11.5 -> 8.8 us); rows that fill the chip take 256.
template <typename T, bool VEC, int NT>
__global__ __launch_bounds__(NT) void row_tokens_kernel(const int32_t* __restrict__ known, int n,
                                                                  const T* __restrict__ rows, int64_t ld,
                                                                  int64_t vocab, int tail, int64_t* __restrict__ out) {
  if ((int)blockIdx.x >= tail) {
    const int i = ((int)blockIdx.x - tail) * NT + threadIdx.x;
    if (i < n) out[i] = known[i];
    return;
  }
  const T* row = rows + (int64_t)blockIdx.x * ld;
  float best = -INFINITY;
  int at = 0x7fffffff;
  constexpr int kAhead = NT > 256 ? 4 : 1;
#pragma unroll kAhead
  for (int64_t base = (int64_t)threadIdx.x * 8; base < vocab; base += NT * 8) {
    float x[8];
    load8<T, VEC>(row, base, vocab, x);
#pragma unroll
    for (int i = 0; i < 8; ++i)
      if (x[i] > best && base + i < vocab) { best = x[i]; at = (int)(base + i); }
  }
  auto take = [&](float b, int a) { if (b > best || (b == best && a < at)) { best = b; at = a; } };
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) take(__shfl_xor(best, m, 64), __shfl_xor(at, m, 64));
  __shared__ float bl[NT / 64];
  __shared__ int al[NT / 64];
  if ((threadIdx.x & 63) == 0) { bl[threadIdx.x >> 6] = best; al[threadIdx.x >> 6] = at; }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < NT / 64; ++w) take(bl[w], al[w]);
    out[n + (int64_t)blockIdx.x] = at < vocab ? at : 0;  // (no value above -infinity: see settle)
  }
}

// spx_block_total.  pos_weight == nullptr: the weight of slot s is exp(-max(s - 1, 0) / gamma), 0 at s = 0; from_anchor:
// exp(-s / gamma).
__global__ __launch_bounds__(kReduceThreads) void block_reduce_kernel(
    const float* __restrict__ loss, const int32_t* __restrict__ pred, const int32_t* __restrict__ tgt,
    const void* __restrict__ mask, int mask_kind, const float* __restrict__ pos_weight, float gamma, int from_anchor,
    int64_t rows, int block_size, float factor, const float* total_in, float* total_out, float* __restrict__ out,
    float* __restrict__ row_weight) {
  __shared__ float fl[kReduceThreads / 64];
  extern __shared__ int slots[];  // [2 * block_size], and a weight per slot behind them
  float* const decay = reinterpret_cast<float*>(slots + 2 * block_size);
  for (int i = threadIdx.x; i < 2 * block_size; i += kReduceThreads) slots[i] = 0;
  if (!pos_weight)
    for (int i = threadIdx.x; i < block_size; i += kReduceThreads)
      decay[i] = from_anchor ? expf(-(float)i / gamma) : i == 0 ? 0.f : expf(-(float)(i - 1) / gamma);
  __syncthreads();
  auto weight = [&](int64_t r) { return pos_weight ? pos_weight[r] : decay[r % block_size]; };
  float lsum = 0.f, msum = 0.f;
  for (int64_t r = threadIdx.x; r < rows; r += kReduceThreads) {
    float m = mask ? mask_value(mask, mask_kind, r) : 1.f;
    float w = weight(r);
    if (m != 0.f) {
      int s = (int)(r % block_size);
      atomicAdd(&slots[block_size + s], 1);
      if (pred[r] == tgt[r]) atomicAdd(&slots[s], 1);
    }
    lsum = fmaf(loss[r] * m, w, lsum);
    msum += m;
  }
  lsum = block_sum_f(lsum, fl);
  msum = block_sum_f(msum, fl);
  const float inv = 1.f / (msum + 1e-5f);
  __syncthreads();
  for (int i = threadIdx.x; i < 2 * block_size; i += kReduceThreads) out[9 + i] = (float)slots[i];
  if (threadIdx.x == 0) {
    const float part = factor * (lsum * inv), sum = total_in ? *total_in + part : part;
    *total_out = sum;
    // the step's metrics: what a dozen one-element kernels did
    float hits = 0.f, rows_in = 0.f, run = 1.f, eal = 0.f;
    for (int i = from_anchor ? 0 : 1; i < block_size; ++i) {
      const float c = (float)slots[i], t = (float)slots[block_size + i];
      hits += c;
      rows_in += t;
      run *= c / fmaxf(t, 1.f);
      eal += run;
    }
    out[0] = lsum * inv;
    out[1] = msum;
    out[2] = sum;
    out[3] = hits;
    out[4] = rows_in;
    out[5] = eal;
    out[6] = out[7] = out[8] = 1.f;
  }
  for (int64_t r = threadIdx.x; r < rows; r += kReduceThreads) {
    const float m = mask ? mask_value(mask, mask_kind, r) : 1.f;
    row_weight[r] = m * weight(r) * inv;
  }
}

// One thread per row of the draft: the inputs of an anchored-block step (models/dflash/core.py:264-271,330-439)
__global__ __launch_bounds__(256) void dflash_inputs_kernel(
    const int64_t* __restrict__ anchors, const uint8_t* __restrict__ valid, int n_q, int block_size, int64_t T,
    int64_t mask_token, const int64_t* __restrict__ input_ids, const int64_t* __restrict__ positions,
    const void* __restrict__ loss_mask, int mask_kind, int from_anchor, int64_t* __restrict__ ids,
    int64_t* __restrict__ kv_pos, int64_t* __restrict__ target_row, float* __restrict__ aligned,
    int32_t* __restrict__ outside) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i < T) {
    kv_pos[i] = positions[i];
    return;
  }
  const int64_t r = i - T;
  if (r >= n_q) return;
  const int j = (int)(r / block_size), s = (int)(r % block_size);
  int64_t a = anchors[j], row = a + s;
  const bool inside = a >= -T && row < T;
  if (!inside && outside) *outside = 1;
  if (row < 0) row += T;  // (counted from the end row by row: a block that begins in front of the end goes on at the start)
  if (a < 0) a += T;
  a = min(max(a, (int64_t)0), T - 1);
  row = min(max(row, (int64_t)0), T - 1);
  ids[r] = s == 0 ? input_ids[a] : mask_token;
  kv_pos[i] = positions[a] + s;
  target_row[r] = from_anchor ? row : row > 0 ? row - 1 : T - 1;
  // (a block that leaves the sequence shows in the loss)
  const float m = mask_value(loss_mask, mask_kind, row) * (valid[j] ? 1.f : 0.f);
  aligned[r] = !inside && valid[j] ? __uint_as_float(0x7fc00000u) : (!from_anchor && s == 0) ? 0.f : m;
}

// ---- dispatch ----------------------------------------------------------------
static bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

// Threads per row: enough that few rows fill the chip (2048 threads per compute unit), not so many that a compute unit holds
// one row only and waits between them.  It depends on the call's sizes alone: the gathering form of a call adds in the same order
// and gives the same bits, except that above 64 rows its KL / CE form stays with the pipelined kernel of 256 threads, and above 256
// its fp32 form of jsd and tv with 512 where the plain one has 1024.
// Measured with 256 threads, a load at a time -> these and one wave's sums by lane moves (us), bf16: KL 64 rows of 128256 76 -> 24,
// 333 rows of 128256 92 -> 45, of 32000 27 -> 17, 1024 of 32000 33 -> 30; backward (columns over several workgroups) 64 rows of
// 128256 66 -> 7.
static int threads_per_row(int64_t rows) { return rows <= 256 ? 1024 : rows <= 512 ? 512 : kLossThreads; }
// jsd and tv walk a row twice.  Of some columns on, up to 32768, the pair stays in a workgroup's registers between the walks: 512 threads
// a row, two rows a compute unit (bf16), or 1024 and one (fp32, and where there are no more rows than compute units).  256 threads that
// read twice / held, forward + backward, us: jsd bf16 3000 rows of 32000 242 / 231, of 24000 179 / 177, of 16000 125 / 125 (1024 rows
// 50.3 / 46.8), of 12000 98 / 103; tv 236 / 200, 174 / 156, 121 / 112, 91 / 93; fp32 jsd 453 / 438, 344 / 337, 231 / 243, 169 / 187, tv
// 448 / 418, 338 / 321, 227 / 230, 166 / 178; forward alone, 3000 rows of 1000 18 / 27 (bf16), 18 / 59 (fp32).  Rows that do not begin
// at 16 bytes, and the gathering form, have nothing to hold, but the same threads (256 / so, forward: bf16 3000 rows of 32003 485 / 368,
// gathered 1024 of 32000 154 / 149; gathered fp32 253 with 1024 threads, 247 with 256, 238 with 512).
static bool walked_twice(int op) { return op == SPX_LOSS_JSD || op == SPX_LOSS_TV; }
static bool held_vocab(int64_t vocab, bool wide) {
  return vocab > (wide ? 18432 : 14336) && vocab <= 32768 + 7;  // (columns behind the last whole chunk are read again)
}
static int threads_per_row(int64_t rows, int64_t vocab, int op, bool wide, bool gather) {
  if (!walked_twice(op) || !held_vocab(vocab, wide)) return threads_per_row(rows);
  return rows <= 256 || (wide && !gather) ? 1024 : 512;
}

// Rows that the 256 MB cache can hold a good part of are left in it for the backward; ce's target rows never, which its backward does
// not read.  Forward + backward past the caches / through them, us, other rows read before, and the rows themselves just written: kl bf16
// 333 x 32000 (41 MiB a pair) 32 / 28 and 32 / 27, 1500 x 60000 (343) 182 / 164 and 193 / 188, 3000 x 32000 (366) 182 / 159 and 191 / 191,
// ce 140 / 120 and 151 / 128; fp32 333 x 32000 52 / 43 and 60 / 40, 333 x 128256 (326) 183 / 165 and 195 / 178, ce 150 / 142 and 164 / 149, but
// 3000 x 16000 (366) 172 / 168 and 181 / 195, ce 139 / 132 and 146 / 148.
template <typename T>
constexpr int64_t kKeptBytes = (sizeof(T) == 4 ? 340ll : 400ll) << 20;

template <typename T, bool VEC, bool KNOWN, bool GATHER, int NT>
static int launch_fwd(const char* fname, int op, const T* lg, int64_t ldl, const T* tg, int64_t ldt, int64_t rows,
                      int64_t vocab, float* loss, float* lsd, float* lst, float* ex, int32_t* ad,
                      int32_t* at, const StepArgs& sa, hipStream_t st) {
  const dim3 grid((unsigned)rows), block(NT);
  constexpr int lds = GATHER ? gather_stage_bytes(NT) : 0;
  const bool keep = rows * vocab * 2 * (int64_t)sizeof(T) <= kKeptBytes<T>;
#define SPX_FWD(OPV)                                                                                               \
  case OPV: if constexpr (!KNOWN || OPV == SPX_LOSS_KL || OPV == SPX_LOSS_CE) {                                    \
    if constexpr (lds > 65536) {                                                                                   \
      static std::atomic<uint64_t> lds_set;                                                                        \
      if (int rc = ensure_dynamic_lds(reinterpret_cast<const void*>(&loss_fwd_kernel<T, OPV, VEC, KNOWN, GATHER, NT, 0>), \
                                      lds, lds_set, fname))                                                        \
        return rc;                                                                                                 \
    }                                                                                                              \
    constexpr bool held = VEC && !KNOWN && !GATHER && (NT == 1024 || (NT == 512 && sizeof(T) == 2)) &&              \
                          (OPV == SPX_LOSS_JSD || OPV == SPX_LOSS_TV);                                             \
    if (held && held_vocab(vocab, sizeof(T) == 4))                                                                 \
      hipLaunchKernelGGL((loss_fwd_kernel<T, OPV, VEC, KNOWN, GATHER, NT, held ? 4096 / NT : 0>), grid, block, lds, \
                         st, lg, ldl, tg, ldt, vocab, loss, lsd, lst, ex, ad, at, sa, keep);                       \
    else                                                                                                           \
      hipLaunchKernelGGL((loss_fwd_kernel<T, OPV, VEC, KNOWN, GATHER, NT, 0>), grid, block, lds, st, lg, ldl, tg,  \
                         ldt, vocab, loss, lsd, lst, ex, ad, at, sa, keep);                                        \
  }                                                                                                                \
  break;
  switch (op) {
    SPX_FWD(SPX_LOSS_KL) SPX_FWD(SPX_LOSS_RKL) SPX_FWD(SPX_LOSS_JSD) SPX_FWD(SPX_LOSS_CE)
    SPX_FWD(SPX_LOSS_TV)
  }
#undef SPX_FWD
  return check_launch(fname);
}

template <typename T, bool VEC>
static void launch_bwd(int op, const T* lg, int64_t ldl, const T* tg, int64_t ldt, int64_t rows,
                       int64_t vocab, const float* lsd, const float* lst, const float* ex,
                       const int32_t* at, const float* rg, const float* sc, T* grad, int64_t ldg,
                       const int32_t* row_map, hipStream_t st) {
  // at least 2048 workgroups, each with a chunk per thread
  const int64_t parts = std::max<int64_t>(1, std::min((2048 + rows - 1) / rows, (vocab / 8 + kLossThreads - 1) / kLossThreads));
  dim3 grid((unsigned)rows, (unsigned)parts), block(kLossThreads);
#define SPX_BWD(OPV)                                                                         \
  case OPV:                                                                                  \
    hipLaunchKernelGGL((loss_bwd_kernel<T, OPV, VEC>), grid, block, 0, st, lg, ldl, tg, ldt, \
                       vocab, lsd, lst, ex, at, rg, sc, grad, ldg, row_map);                 \
    break;
  switch (op) {
    SPX_BWD(SPX_LOSS_KL) SPX_BWD(SPX_LOSS_RKL) SPX_BWD(SPX_LOSS_JSD) SPX_BWD(SPX_LOSS_CE)
    SPX_BWD(SPX_LOSS_TV)
  }
#undef SPX_BWD
}

}  // namespace spx

using namespace spx;

static bool kind_ok(int k) { return k >= SPX_KIND_U8 && k <= SPX_KIND_BF16; }

#define SPX_REQ_FN(cond, what) do { if (!(cond)) return spx::fail_arg(fname, what); } while (0)
static int loss_fwd_impl(const char* fname, int op, const void* logits, int64_t ld_logits,
                         const void* targets, int64_t ld_targets, int64_t rows, int64_t vocab,
                         int dtype, float* loss, float* lse_draft, float* lse_target, float* extra,
                         int32_t* argmax_draft, int32_t* argmax_target, int reuse_target_stats,
                         const StepArgs& sa, void* stream) {
  SPX_REQ_FN(op >= SPX_LOSS_KL && op <= SPX_LOSS_TV, "unknown loss op");
  SPX_REQ_FN(dtype == SPX_DTYPE_BF16 || dtype == SPX_DTYPE_F32, "dtype must be bf16 or f32");
  SPX_REQ_FN(rows >= 0 && vocab > 0 && vocab < (1ll << 31), "rows >= 0 and 0 < vocab < 2^31");
  const bool gather = sa.d2t != nullptr;
  // cross-entropy with the target rows' arg-max handed in reads no target element: the rows may be absent
  const bool no_targets = !targets && reuse_target_stats && op == SPX_LOSS_CE && !gather;
  SPX_REQ_FN(ld_logits >= vocab && (no_targets || ld_targets >= (gather ? sa.vt : vocab)),
             "row stride smaller than vocab");
  SPX_REQ_FN(rows < (1ll << 31), "too many rows");
  if (gather) {
    SPX_REQ_FN(sa.vt > 0 && sa.vt < (1ll << 31), "0 < vt < 2^31");
    SPX_REQ_FN(!reuse_target_stats, "the gather form computes the target statistics itself");
    SPX_REQ_FN(!sa.gathered || sa.ld_gathered >= vocab, "gathered row stride smaller than vocab");
  }
  if (sa.counts) {
    SPX_REQ_FN(argmax_draft && argmax_target, "the acceptance chain needs both arg-max outputs");
    SPX_REQ_FN(!sa.mask || kind_ok(sa.mask_kind), "unknown mask element kind");
    SPX_REQ_FN(!sa.prev || kind_ok(sa.prev_kind), "unknown prev_correct element kind");
  }
  if (rows == 0) return SPX_OK;
  SPX_REQ_FN(logits && (targets || no_targets) && loss && lse_draft && lse_target && extra, "null buffer");
  // the second-pass reductions (rkl, jsd, tv) recompute from both rows anyway
  const bool known = reuse_target_stats && (op == SPX_LOSS_KL || op == SPX_LOSS_CE);
  if (known && op == SPX_LOSS_CE) SPX_REQ_FN(argmax_target, "ce with reused statistics needs argmax_target");
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  const int64_t per16 = dtype == SPX_DTYPE_BF16 ? 8 : 4;
  const bool vec = aligned16(logits) && ld_logits % per16 == 0 &&
                   (gather ? (!sa.gathered || (aligned16(sa.gathered) && sa.ld_gathered % per16 == 0))
                           : (no_targets || (aligned16(targets) && ld_targets % per16 == 0)));
  // the first step of the verifier-logits entry in its common form: the pipelined kernel
  const int nt = threads_per_row(rows, vocab, op, dtype == SPX_DTYPE_F32, gather);
  if (gather && vec && (nt == kLossThreads || rows > 64) && dtype == SPX_DTYPE_BF16 && (op == SPX_LOSS_KL || op == SPX_LOSS_CE) &&
      aligned16(targets) && ld_targets % 8 == 0 && vocab <= (int64_t)kPipeMaxTiles * kPipeTileIds &&
      sa.vt < (1ll << 30)) {
    static std::atomic<uint64_t> lds_set[2];  // per instantiation, one bit per device
    const bool kl = op == SPX_LOSS_KL;
    const void* fn = kl ? reinterpret_cast<const void*>(&loss_fwd_gather_pipe_kernel<SPX_LOSS_KL>)
                        : reinterpret_cast<const void*>(&loss_fwd_gather_pipe_kernel<SPX_LOSS_CE>);
    if (int rc = ensure_dynamic_lds(fn, kPipeSmem, lds_set[kl], fname)) return rc;
    const dim3 grid((unsigned)rows), block(kLossThreads);
    auto lg = reinterpret_cast<const uint16_t*>(logits);
    auto tg = reinterpret_cast<const uint16_t*>(targets);
    if (kl)
      hipLaunchKernelGGL(loss_fwd_gather_pipe_kernel<SPX_LOSS_KL>, grid, block, kPipeSmem, st, lg, ld_logits, tg,
                         ld_targets, vocab, loss, lse_draft, lse_target, extra, argmax_draft, argmax_target, sa);
    else
      hipLaunchKernelGGL(loss_fwd_gather_pipe_kernel<SPX_LOSS_CE>, grid, block, kPipeSmem, st, lg, ld_logits, tg,
                         ld_targets, vocab, loss, lse_draft, lse_target, extra, argmax_draft, argmax_target, sa);
    return check_launch(fname);
  }
#define SPX_GO_N(TT, VV, KK, GG, NN)                                                                        \
  return launch_fwd<TT, VV, KK, GG, NN>(fname, op, reinterpret_cast<const TT*>(logits), ld_logits,           \
                                        reinterpret_cast<const TT*>(targets), ld_targets, rows, vocab, loss, \
                                        lse_draft, lse_target, extra, argmax_draft, argmax_target, sa, st)
#define SPX_GO(TT, VV, KK, GG)                                                                        \
  do {                                                                                                \
    if (nt == 1024) SPX_GO_N(TT, VV, KK, GG, 1024);                                                   \
    else if (nt == 512) SPX_GO_N(TT, VV, KK, GG, 512);                                                \
    else SPX_GO_N(TT, VV, KK, GG, kLossThreads);                                                      \
  } while (0)
#define SPX_GO_T(TT)                                                                   \
  do {                                                                                 \
    if (gather) { if (vec) SPX_GO(TT, true, false, true); else SPX_GO(TT, false, false, true); } \
    else if (vec) { if (known) SPX_GO(TT, true, true, false); else SPX_GO(TT, true, false, false); } \
    else { if (known) SPX_GO(TT, false, true, false); else SPX_GO(TT, false, false, false); } \
  } while (0)
  if (dtype == SPX_DTYPE_BF16) SPX_GO_T(uint16_t);
  else SPX_GO_T(float);
#undef SPX_GO_T
#undef SPX_GO
#undef SPX_GO_N
}

extern "C" int spx_fused_vocab_loss_fwd(int op, const void* logits, int64_t ld_logits,
                                        const void* targets, int64_t ld_targets, int64_t rows,
                                        int64_t vocab, int dtype, float* loss, float* lse_draft,
                                        float* lse_target, float* extra, int32_t* argmax_draft,
                                        int32_t* argmax_target, int reuse_target_stats,
                                        void* stream) {
  const StepArgs none = {nullptr, 0, nullptr, 0, nullptr, 0, nullptr, 0, nullptr};
  return loss_fwd_impl(__func__, op, logits, ld_logits, targets, ld_targets, rows, vocab, dtype, loss,
                       lse_draft, lse_target, extra, argmax_draft, argmax_target, reuse_target_stats,
                       none, stream);
}

extern "C" int spx_vocab_loss_step_fwd(int op, const void* logits, int64_t ld_logits,
                                       const void* targets, int64_t ld_targets, const int64_t* d2t,
                                       int64_t vt, void* gathered, int64_t ld_gathered, int64_t rows,
                                       int64_t vocab, int dtype, float* loss, float* lse_draft,
                                       float* lse_target, float* extra, int32_t* argmax_draft,
                                       int32_t* argmax_target, int reuse_target_stats,
                                       const void* mask, int mask_kind, void* prev_correct,
                                       int prev_kind, int32_t* counts, void* stream) {
  const StepArgs sa = {d2t, vt, gathered, ld_gathered, mask, mask_kind, prev_correct, prev_kind, counts};
  return loss_fwd_impl(__func__, op, logits, ld_logits, targets, ld_targets, rows, vocab, dtype, loss,
                       lse_draft, lse_target, extra, argmax_draft, argmax_target, reuse_target_stats,
                       sa, stream);
}

extern "C" int spx_vocab_loss_step_fwd_grad(int op, const void* logits, int64_t ld_logits,
                                            const void* targets, int64_t ld_targets, int64_t rows,
                                            int64_t vocab, float* loss, float* lse_draft,
                                            float* lse_target, float* extra, int32_t* argmax_draft,
                                            int32_t* argmax_target, int reuse_target_stats,
                                            const void* mask, int mask_kind, void* prev_correct,
                                            int prev_kind, int32_t* counts, const int32_t* row_map,
                                            void* grad_logits, int64_t ld_grad, void* stream) {
  const char* fname = __func__;
  SPX_REQ_FN(op == SPX_LOSS_KL || op == SPX_LOSS_CE, "the one-pass form is built for kl and ce");
  SPX_REQ_FN(rows >= 0 && rows < (1ll << 31), "bad row count");
  SPX_REQ_FN(vocab > 0 && vocab % 8 == 0 && vocab <= (int64_t)kFgThreads * kFgChunks * 8,
             "vocab must be a multiple of 8, at most 32768");
  const bool known = reuse_target_stats != 0;
  const bool no_targets = known && op == SPX_LOSS_CE;
  SPX_REQ_FN(ld_logits >= vocab && ld_grad >= vocab && (no_targets || ld_targets >= vocab),
             "row stride smaller than vocab");
  SPX_REQ_FN(ld_logits % 8 == 0 && ld_grad % 8 == 0 && (no_targets || ld_targets % 8 == 0),
             "row strides must be multiples of 8 elements");
  if (counts) {
    SPX_REQ_FN(!mask || kind_ok(mask_kind), "unknown mask element kind");
    SPX_REQ_FN(!prev_correct || kind_ok(prev_kind), "unknown prev_correct element kind");
  }
  if (rows == 0) return SPX_OK;
  SPX_REQ_FN(logits && (targets || no_targets) && loss && lse_draft && lse_target && extra && argmax_target &&
                 row_map && grad_logits, "null buffer");
  SPX_REQ_FN(!counts || argmax_draft, "the acceptance chain needs both arg-max outputs");
  SPX_REQ_FN(aligned16(logits) && aligned16(grad_logits) && (no_targets || aligned16(targets)),
             "rows must be 16-byte aligned");
  const StepArgs sa = {nullptr, 0, nullptr, 0, mask, mask_kind, prev_correct, prev_kind, counts};
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  const dim3 grid((unsigned)rows), block(kFgThreads);
  auto lg = reinterpret_cast<const uint16_t*>(logits);
  auto tg = reinterpret_cast<const uint16_t*>(targets);
  auto gr = reinterpret_cast<uint16_t*>(grad_logits);
#define SPX_FG(OPV, KN)                                                                                     \
  hipLaunchKernelGGL((loss_fwd_grad_kernel<OPV, KN>), grid, block, 0, st, lg, ld_logits, tg, ld_targets, vocab, \
                     loss, lse_draft, lse_target, extra, argmax_draft, argmax_target, sa, row_map, gr, ld_grad)
  if (op == SPX_LOSS_KL) { if (known) SPX_FG(SPX_LOSS_KL, true); else SPX_FG(SPX_LOSS_KL, false); }
  else { if (known) SPX_FG(SPX_LOSS_CE, true); else SPX_FG(SPX_LOSS_CE, false); }
#undef SPX_FG
  return check_launch(fname);
}

static bool terms_ok(int32_t terms, const float* w) { return terms > 0 && terms < 32 && w; }
static LossTerms loss_terms(int32_t terms, const float* w) {
  LossTerms t{terms, {}};
  for (int op = 0; op < 5; ++op) t.w[op] = terms >> op & 1 ? w[op] : 0.f;
  return t;
}

extern "C" int spx_vocab_loss_terms_fwd_grad(int32_t terms, const float* term_weights, const void* logits,
                                             int64_t ld_logits, const void* targets, int64_t ld_targets, int64_t rows,
                                             int64_t vocab, float* loss, float* lse_draft, float* lse_target,
                                             int32_t* argmax_draft, int32_t* argmax_target, int reuse_target_stats,
                                             const void* mask, int mask_kind, void* prev_correct, int prev_kind,
                                             int32_t* counts, const int32_t* row_map, void* grad_logits,
                                             int64_t ld_grad, void* stream) {
  SPX_REQUIRE(terms_ok(terms, term_weights), "terms must be a set of loss ops with their weights");
  SPX_REQUIRE(rows >= 0 && rows < (1ll << 31), "bad row count");
  SPX_REQUIRE(vocab > 0 && vocab % 8 == 0 && vocab <= (int64_t)kFgThreads * kFgChunks * 8,
              "vocab must be a multiple of 8, at most 32768");
  SPX_REQUIRE(ld_logits >= vocab && ld_grad >= vocab && ld_targets >= vocab, "row stride smaller than vocab");
  SPX_REQUIRE(ld_logits % 8 == 0 && ld_grad % 8 == 0 && ld_targets % 8 == 0,
              "row strides must be multiples of 8 elements");
  SPX_REQUIRE(!mask || kind_ok(mask_kind), "unknown mask element kind");
  SPX_REQUIRE(!prev_correct || kind_ok(prev_kind), "unknown prev_correct element kind");
  if (rows == 0) return SPX_OK;
  SPX_REQUIRE(logits && targets && loss && lse_draft && lse_target && argmax_draft && argmax_target && row_map &&
                  grad_logits, "null buffer");
  SPX_REQUIRE(aligned16(logits) && aligned16(grad_logits) && aligned16(targets), "rows must be 16-byte aligned");
  const StepArgs sa = {nullptr, 0, nullptr, 0, mask, mask_kind, prev_correct, prev_kind, counts};
  const LossTerms tm = loss_terms(terms, term_weights);
#define SPX_TG(KN, KLV)                                                                                              \
  hipLaunchKernelGGL((loss_terms_grad_kernel<KN, KLV>), dim3((unsigned)rows), dim3(kFgThreads), 0,                   \
                     reinterpret_cast<hipStream_t>(stream), reinterpret_cast<const uint16_t*>(logits), ld_logits,    \
                     reinterpret_cast<const uint16_t*>(targets), ld_targets, rows, vocab, loss, lse_draft, lse_target, \
                     argmax_draft, argmax_target, sa, tm, row_map, reinterpret_cast<uint16_t*>(grad_logits), ld_grad)
  if (terms >> SPX_LOSS_KL & 1) { if (reuse_target_stats) SPX_TG(true, true); else SPX_TG(false, true); }
  else { if (reuse_target_stats) SPX_TG(true, false); else SPX_TG(false, false); }
#undef SPX_TG
  return check_launch(__func__);
}

static int loss_bwd_impl(const char* fname, int op, const void* logits, int64_t ld_logits,
                         const void* targets, int64_t ld_targets, int64_t rows,
                         int64_t vocab, int dtype, const float* lse_draft,
                         const float* lse_target, const float* extra,
                         const int32_t* argmax_target, const float* row_grad,
                         const float* scale, void* grad_logits, int64_t ld_grad,
                         const int32_t* row_map, void* stream) {
  SPX_REQ_FN(op >= SPX_LOSS_KL && op <= SPX_LOSS_TV, "unknown loss op");
  SPX_REQ_FN(dtype == SPX_DTYPE_BF16 || dtype == SPX_DTYPE_F32, "dtype must be bf16 or f32");
  SPX_REQ_FN(rows >= 0 && vocab > 0 && vocab < (1ll << 31), "rows >= 0 and 0 < vocab < 2^31");
  SPX_REQ_FN(ld_logits >= vocab && ld_grad >= vocab, "row stride smaller than vocab");
  SPX_REQ_FN(rows < (1ll << 31), "too many rows");
  if (rows == 0) return SPX_OK;
  SPX_REQ_FN(logits && grad_logits && lse_draft && row_grad, "null buffer");
  if (op == SPX_LOSS_CE) SPX_REQ_FN(argmax_target, "ce needs argmax_target");
  else SPX_REQ_FN(targets && lse_target && ld_targets >= vocab, "targets / lse_target missing");
  if (op == SPX_LOSS_RKL || op == SPX_LOSS_JSD || op == SPX_LOSS_TV) SPX_REQ_FN(extra, "extra missing");
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  const int64_t per16 = dtype == SPX_DTYPE_BF16 ? 8 : 4;
  const bool vec = aligned16(logits) && (op == SPX_LOSS_CE || (aligned16(targets) && ld_targets % per16 == 0)) &&
                   aligned16(grad_logits) && ld_logits % per16 == 0 && ld_grad % per16 == 0;
  if (dtype == SPX_DTYPE_BF16) {
    auto lg = reinterpret_cast<const uint16_t*>(logits);
    auto tg = reinterpret_cast<const uint16_t*>(targets);
    auto gr = reinterpret_cast<uint16_t*>(grad_logits);
    if (vec) launch_bwd<uint16_t, true>(op, lg, ld_logits, tg, ld_targets, rows, vocab, lse_draft, lse_target, extra, argmax_target, row_grad, scale, gr, ld_grad, row_map, st);
    else launch_bwd<uint16_t, false>(op, lg, ld_logits, tg, ld_targets, rows, vocab, lse_draft, lse_target, extra, argmax_target, row_grad, scale, gr, ld_grad, row_map, st);
  } else {
    auto lg = reinterpret_cast<const float*>(logits);
    auto tg = reinterpret_cast<const float*>(targets);
    auto gr = reinterpret_cast<float*>(grad_logits);
    if (vec) launch_bwd<float, true>(op, lg, ld_logits, tg, ld_targets, rows, vocab, lse_draft, lse_target, extra, argmax_target, row_grad, scale, gr, ld_grad, row_map, st);
    else launch_bwd<float, false>(op, lg, ld_logits, tg, ld_targets, rows, vocab, lse_draft, lse_target, extra, argmax_target, row_grad, scale, gr, ld_grad, row_map, st);
  }
  return check_launch(fname);
}
#undef SPX_REQ_FN

extern "C" int spx_fused_vocab_loss_bwd(int op, const void* logits, int64_t ld_logits,
                                        const void* targets, int64_t ld_targets, int64_t rows,
                                        int64_t vocab, int dtype, const float* lse_draft,
                                        const float* lse_target, const float* extra,
                                        const int32_t* argmax_target, const float* row_grad,
                                        const float* scale, void* grad_logits, int64_t ld_grad,
                                        void* stream) {
  return loss_bwd_impl(__func__, op, logits, ld_logits, targets, ld_targets, rows, vocab, dtype, lse_draft,
                       lse_target, extra, argmax_target, row_grad, scale, grad_logits, ld_grad, nullptr, stream);
}

extern "C" int spx_fused_vocab_loss_bwd_packed(int op, const void* logits, int64_t ld_logits,
                                               const void* targets, int64_t ld_targets, int64_t rows,
                                               int64_t vocab, int dtype, const float* lse_draft,
                                               const float* lse_target, const float* extra,
                                               const int32_t* argmax_target, const float* row_grad,
                                               const float* scale, const int32_t* row_map,
                                               void* grad_logits, int64_t ld_grad, void* stream) {
  if (!row_map) return spx::fail_arg(__func__, "null row map");
  return loss_bwd_impl(__func__, op, logits, ld_logits, targets, ld_targets, rows, vocab, dtype, lse_draft,
                       lse_target, extra, argmax_target, row_grad, scale, grad_logits, ld_grad, row_map, stream);
}

extern "C" int spx_vocab_gather(const void* full, int64_t ld_full, const int64_t* d2t, void* out,
                                int64_t ld_out, int64_t rows, int64_t vd, int64_t vt, int dtype,
                                void* stream) {
  SPX_REQUIRE(dtype == SPX_DTYPE_BF16 || dtype == SPX_DTYPE_F32, "dtype must be bf16 or f32");
  SPX_REQUIRE(rows >= 0 && vd > 0 && vt > 0, "rows >= 0, vd > 0, vt > 0");
  SPX_REQUIRE(ld_full >= vt && ld_out >= vd, "row stride smaller than the row");
  SPX_REQUIRE(rows < 65536, "at most 65535 rows per call");
  if (rows == 0) return SPX_OK;
  SPX_REQUIRE(full && d2t && out, "null buffer");
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  unsigned gx = (unsigned)((vd + 256 * 4 - 1) / (256 * 4));
  dim3 grid(gx, (unsigned)rows), block(256);
  if (dtype == SPX_DTYPE_BF16)
    hipLaunchKernelGGL(vocab_gather_kernel<uint16_t>, grid, block, 0, st,
                       reinterpret_cast<const uint16_t*>(full), ld_full, d2t,
                       reinterpret_cast<uint16_t*>(out), ld_out, vd, vt, (uint16_t)0xff80);
  else
    hipLaunchKernelGGL(vocab_gather_kernel<float>, grid, block, 0, st,
                       reinterpret_cast<const float*>(full), ld_full, d2t,
                       reinterpret_cast<float*>(out), ld_out, vd, vt, -INFINITY);
  return check_launch(__func__);
}

extern "C" int spx_ttt_step_reduce(const float* loss, const int32_t* argmax_draft,
                                   const int32_t* argmax_target, const void* mask, int mask_kind,
                                   void* prev_correct, int prev_kind, int64_t rows, float weight,
                                   float* out, float* row_weight, void* stream) {
  SPX_REQUIRE(rows >= 0 && rows < (1ll << 24), "0 <= rows < 2^24");
  SPX_REQUIRE(loss && argmax_draft && argmax_target && out, "null buffer");
  SPX_REQUIRE(!mask || kind_ok(mask_kind), "unknown mask element kind");
  SPX_REQUIRE(!prev_correct || kind_ok(prev_kind), "unknown prev_correct element kind");
  hipLaunchKernelGGL(ttt_step_reduce_kernel, dim3(1), dim3(kReduceThreads), 0,
                     reinterpret_cast<hipStream_t>(stream), loss, argmax_draft, argmax_target, mask,
                     mask_kind, prev_correct, prev_kind, rows, weight, out, row_weight, nullptr, 1.f, nullptr,
                     nullptr);
  return check_launch(__func__);
}

extern "C" int spx_ttt_step_mean(const float* loss, const void* mask, int mask_kind, int64_t rows,
                                 float weight, const int32_t* counts, float* out, float* row_weight,
                                 void* stream) {
  SPX_REQUIRE(rows >= 0 && rows < (1ll << 24), "0 <= rows < 2^24");
  SPX_REQUIRE(loss && counts && out, "null buffer");
  SPX_REQUIRE(!mask || kind_ok(mask_kind), "unknown mask element kind");
  hipLaunchKernelGGL(ttt_step_reduce_kernel, dim3(1), dim3(kReduceThreads), 0,
                     reinterpret_cast<hipStream_t>(stream), loss, nullptr, nullptr, mask, mask_kind,
                     nullptr, 0, rows, weight, out, row_weight, counts, 1.f, nullptr, nullptr);
  return check_launch(__func__);
}

extern "C" int spx_ttt_step_total(const float* loss, const int32_t* argmax_draft, const int32_t* argmax_target,
                                  const void* mask, int mask_kind, void* prev_correct, int prev_kind, int64_t rows,
                                  float weight, const int32_t* counts, float factor, const float* total_in,
                                  float* total_out, float* out, float* row_weight, void* stream) {
  SPX_REQUIRE(rows >= 0 && rows < (1ll << 24), "0 <= rows < 2^24");
  SPX_REQUIRE(loss && out && total_out && (counts || (argmax_draft && argmax_target)), "null buffer");
  SPX_REQUIRE(!mask || kind_ok(mask_kind), "unknown mask element kind");
  SPX_REQUIRE(!prev_correct || kind_ok(prev_kind), "unknown prev_correct element kind");
  hipLaunchKernelGGL(ttt_step_reduce_kernel, dim3(1), dim3(kReduceThreads), 0,
                     reinterpret_cast<hipStream_t>(stream), loss, argmax_draft, argmax_target, mask, mask_kind,
                     prev_correct, prev_kind, rows, weight, out, row_weight, counts, factor, total_in, total_out);
  return check_launch(__func__);
}

extern "C" int spx_ttt_step_terms(int32_t terms, const float* term_weights, const float* loss, const void* mask,
                                  int mask_kind, int64_t rows, float weight, const int32_t* counts,
                                  const float* total_in, float* total_out, float* out, float* row_weight,
                                  void* stream) {
  SPX_REQUIRE(terms_ok(terms, term_weights), "terms must be a set of loss ops with their weights");
  SPX_REQUIRE(rows >= 0 && rows < (1ll << 24), "0 <= rows < 2^24");
  SPX_REQUIRE(loss && counts && total_out && out && row_weight, "null buffer");
  SPX_REQUIRE(!mask || kind_ok(mask_kind), "unknown mask element kind");
  hipLaunchKernelGGL(ttt_step_terms_kernel, dim3(1), dim3(kReduceThreads), 0, reinterpret_cast<hipStream_t>(stream),
                     loss, loss_terms(terms, term_weights), mask, mask_kind, rows, weight, counts, total_in, total_out,
                     out, row_weight);
  return check_launch(__func__);
}

extern "C" int spx_mask_row_lists(const void* mask, int mask_kind, int64_t rows, int32_t* row_map, int32_t* count,
                                  int32_t* row_of, int32_t* zero3, void* stream) {
  SPX_REQUIRE(rows > 0 && rows < (1ll << 31), "rows out of range");
  SPX_REQUIRE(mask && row_map && count && kind_ok(mask_kind), "null buffer or unknown mask element kind");
  hipLaunchKernelGGL(mask_row_map_kernel, dim3(1), dim3(1024), 0, reinterpret_cast<hipStream_t>(stream), mask,
                     mask_kind, (int)rows, row_map, count, row_of, zero3);
  return check_launch(__func__);
}

extern "C" int spx_mask_row_map(const void* mask, int mask_kind, int64_t rows, int32_t* row_map, int32_t* count,
                                int32_t* zero3, void* stream) {
  return spx_mask_row_lists(mask, mask_kind, rows, row_map, count, nullptr, zero3, stream);
}

static bool steps_ok(int64_t T, int32_t steps) {
  return steps > 0 && steps <= SPX_LOSS_STEPS_MAX && T >= steps && T * steps < (1ll << 31);
}

extern "C" int spx_loss_steps_mask(const void* mask, int mask_kind, int64_t T, int32_t steps, const float* step_weights,
                                   int32_t* row_map, int32_t* live, float* inv, float* mask_sum, int32_t* full,
                                   int32_t* ticket, void* stream) {
  SPX_REQUIRE(steps_ok(T, steps), "1 .. 32 steps, no more than rows");
  SPX_REQUIRE(mask && step_weights && row_map && live && inv && mask_sum && full && ticket, "null buffer");
  SPX_REQUIRE(kind_ok(mask_kind), "unknown mask element kind");
  StepWeights w{};
  for (int k = 0; k < steps; ++k) w.w[k] = step_weights[k];
  hipLaunchKernelGGL(steps_mask_kernel, dim3(1), dim3(1024), 0, reinterpret_cast<hipStream_t>(stream), mask, mask_kind,
                     (int)T, steps, w, row_map, live, inv, mask_sum, full, ticket);
  return check_launch(__func__);
}

extern "C" int spx_loss_steps_pass(int op, int32_t terms, const float* term_weights, const void* const* logits, int64_t ld_logits, const void* targets,
                                   int64_t ld_targets, const int32_t* argmax_target, int64_t T, int64_t vocab,
                                   int32_t steps, int32_t first, int32_t end, int32_t masked_first, const void* mask,
                                   int mask_kind, const float* inv, const int32_t* row_map, const int32_t* live, float* loss,
                                   int64_t* tokens, uint8_t* hits, int32_t* row_slot, int32_t* slot_row, int32_t* slots,
                                   float* row_weight, void* grad_logits, int64_t ld_grad, void* stream) {
  constexpr int kTerms = 1 << SPX_LOSS_KL | 1 << SPX_LOSS_CE | 1 << SPX_LOSS_TV;
  SPX_REQUIRE(terms ? terms_ok(terms, term_weights) && !(terms & ~kTerms) : op == SPX_LOSS_KL || op == SPX_LOSS_CE,
              "kl, ce or a set of kl, ce and tv with their weights");
  SPX_REQUIRE(steps_ok(T, steps) && first >= 0 && first < end && end <= steps, "1 .. 32 steps, no more than rows");
  SPX_REQUIRE(vocab > 0 && vocab % 8 == 0 && vocab <= (int64_t)kFgThreads * kFgChunks * 8,
              "vocab must be a multiple of 8, at most 32768");
  SPX_REQUIRE(targets || (!terms && op == SPX_LOSS_CE && argmax_target), "no targets");
  SPX_REQUIRE(ld_logits >= vocab && ld_logits % 8 == 0 && (!targets || (ld_targets >= vocab && ld_targets % 8 == 0)) &&
                  (!grad_logits || (ld_grad >= vocab && ld_grad % 8 == 0)),
              "row strides must be multiples of 8 elements, at least vocab");
  SPX_REQUIRE(logits && mask && inv && loss && tokens && hits, "null buffer");
  SPX_REQUIRE(kind_ok(mask_kind), "unknown mask element kind");
  SPX_REQUIRE(!grad_logits || (row_map && live && row_slot && slot_row && slots && row_weight), "null buffer");
  SPX_REQUIRE((!targets || aligned16(targets)) && (!grad_logits || aligned16(grad_logits)), "rows must be 16-byte aligned");
  StepsArgs a{};
  for (int k = first; k < end; ++k) {
    SPX_REQUIRE(logits[k - first] && aligned16(logits[k - first]), "null or unaligned logits");
    a.logits[k] = reinterpret_cast<const uint16_t*>(logits[k - first]);
  }
  a.ld = ld_logits;
  a.targets = reinterpret_cast<const uint16_t*>(targets);
  a.ld_targets = ld_targets;
  a.argmax_target = argmax_target;
  a.T = (int)T; a.vocab = (int)vocab; a.steps = steps; a.k0 = first; a.k1 = end;
  a.masked_first = masked_first;
  a.tm = terms ? loss_terms(terms, term_weights) : LossTerms{};
  a.mask = mask; a.mask_kind = mask_kind; a.inv = inv;
  a.row_map = row_map; a.live = live;
  a.loss = loss; a.tokens = tokens; a.hits = hits;
  a.row_slot = row_slot; a.slot_row = slot_row; a.slots = slots; a.row_weight = row_weight;
  a.grad = reinterpret_cast<uint16_t*>(grad_logits);
  a.ld_grad = ld_grad;
  const dim3 grid((unsigned)T), block(kFgThreads);
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
#define SPX_SP(...) hipLaunchKernelGGL((loss_steps_kernel<__VA_ARGS__>), grid, block, 0, st, a)
  if (terms >> SPX_LOSS_KL & 1) { if (grad_logits) SPX_SP(SPX_LOSS_KL, true, true); else SPX_SP(SPX_LOSS_KL, false, true); }
  else if (terms) { if (grad_logits) SPX_SP(SPX_LOSS_CE, true, true); else SPX_SP(SPX_LOSS_CE, false, true); }
  else if (op == SPX_LOSS_KL) { if (grad_logits) SPX_SP(SPX_LOSS_KL, true); else SPX_SP(SPX_LOSS_KL, false); }
  else { if (grad_logits) SPX_SP(SPX_LOSS_CE, true); else SPX_SP(SPX_LOSS_CE, false); }
#undef SPX_SP
  return check_launch(__func__);
}

extern "C" int64_t spx_loss_steps_partials(int64_t T, int32_t steps, int32_t terms) {
  return T <= 0 || steps <= 0 ? 0 : (T + kStepsRows - 1) / kStepsRows * steps * (2 + (terms > 0 ? __builtin_popcount(terms) : 1));
}

extern "C" int spx_loss_steps_total(const float* loss, const uint8_t* hits, const void* mask, int mask_kind,
                                    void* prev_correct, int prev_kind, int64_t T, int32_t steps, float factor,
                                    int32_t terms, const float* term_weights, const float* inv, const float* mask_sum, const int32_t* full, float* partials,
                                    int32_t* ticket, float* out, float* total, void* stream) {
  SPX_REQUIRE(steps_ok(T, steps), "1 .. 32 steps, no more than rows");
  SPX_REQUIRE(!terms || terms_ok(terms, term_weights), "terms must be a set of loss ops with their weights");
  SPX_REQUIRE(loss && hits && mask && inv && mask_sum && full && partials && ticket && out && total, "null buffer");
  SPX_REQUIRE(kind_ok(mask_kind) && (!prev_correct || kind_ok(prev_kind)), "unknown element kind");
  hipLaunchKernelGGL(steps_total_kernel, dim3((unsigned)((T + kStepsRows - 1) / kStepsRows)), dim3(kStepsRows), 0,
                     reinterpret_cast<hipStream_t>(stream), loss, hits, mask, mask_kind, prev_correct, prev_kind, (int)T,
                     steps, factor, terms ? loss_terms(terms, term_weights) : LossTerms{}, inv, mask_sum, full, partials, ticket,
                     out, total);
  return check_launch(__func__);
}

extern "C" int spx_row_tokens(const int32_t* known, int64_t n, const void* rows, int64_t ld, int64_t tail,
                              int64_t vocab, int dtype, int64_t* out, void* stream) {
  SPX_REQUIRE(dtype == SPX_DTYPE_BF16 || dtype == SPX_DTYPE_F32, "dtype must be bf16 or f32");
  SPX_REQUIRE(n >= 0 && tail >= 0 && n + tail < (1ll << 31) && vocab > 0 && vocab < (1ll << 31), "sizes out of range");
  if (n + tail == 0) return SPX_OK;
  SPX_REQUIRE(out && (n == 0 || known) && (tail == 0 || (rows && ld >= vocab)), "null buffer or short row stride");
  const bool few = tail <= 256;  // one row per compute unit
  const int nt = few ? 1024 : kLossThreads;
  const dim3 grid((unsigned)(tail + (n + nt - 1) / nt));
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  const bool vec = aligned16(rows) && ld % (dtype == SPX_DTYPE_BF16 ? 8 : 4) == 0;
#define SPX_TOKENS_AS(T, VEC, NT)                                                                             \
  hipLaunchKernelGGL((row_tokens_kernel<T, VEC, NT>), grid, dim3(NT), 0, st, known, (int)n,                  \
                     reinterpret_cast<const T*>(rows), ld, vocab, (int)tail, out)
#define SPX_TOKENS(T, VEC) do { if (few) SPX_TOKENS_AS(T, VEC, 1024); else SPX_TOKENS_AS(T, VEC, kLossThreads); } while (0)
  if (dtype == SPX_DTYPE_BF16) { if (vec) SPX_TOKENS(uint16_t, true); else SPX_TOKENS(uint16_t, false); }
  else { if (vec) SPX_TOKENS(float, true); else SPX_TOKENS(float, false); }
#undef SPX_TOKENS
#undef SPX_TOKENS_AS
  return check_launch(__func__);
}

extern "C" int spx_block_total(const float* loss, const int32_t* argmax_draft, const int32_t* argmax_target,
                               const void* mask, int mask_kind, const float* pos_weight, float gamma, int from_anchor,
                               int64_t rows, int32_t block_size, float factor, const float* total_in,
                               float* total_out, float* out, float* row_weight, void* stream) {
  SPX_REQUIRE(total_out && out && row_weight, "null buffer");
  SPX_REQUIRE(rows >= 0 && rows < (1ll << 24), "0 <= rows < 2^24");
  SPX_REQUIRE(block_size > 0 && block_size <= 4096, "0 < block_size <= 4096");
  SPX_REQUIRE(loss && argmax_draft && argmax_target, "null buffer");
  SPX_REQUIRE(!mask || kind_ok(mask_kind), "unknown mask element kind");
  hipLaunchKernelGGL(block_reduce_kernel, dim3(1), dim3(kReduceThreads),
                     (2 * sizeof(int) + sizeof(float)) * block_size, reinterpret_cast<hipStream_t>(stream), loss,
                     argmax_draft, argmax_target, mask, mask_kind, pos_weight, gamma, from_anchor, rows, block_size,
                     factor, total_in, total_out, out, row_weight);
  return check_launch(__func__);
}

extern "C" int spx_dflash_inputs_checked(const int64_t* anchors, const uint8_t* valid, int64_t n_anchors,
                                         int32_t block_size, int64_t T, int64_t mask_token, const int64_t* input_ids,
                                         const int64_t* positions, const void* loss_mask, int mask_kind, int from_anchor,
                                         int64_t* ids, int64_t* kv_pos, int64_t* target_row, float* aligned,
                                         int32_t* outside, void* stream) {
  SPX_REQUIRE(T > 0 && T < (1ll << 30) && n_anchors >= 0 && block_size > 0 && n_anchors * block_size < (1ll << 30),
              "sizes out of range");
  SPX_REQUIRE(input_ids && positions && loss_mask && kv_pos && kind_ok(mask_kind), "null buffer or unknown mask kind");
  SPX_REQUIRE(n_anchors == 0 || (anchors && valid && ids && target_row && aligned), "null buffer");
  const int64_t n_q = n_anchors * block_size;
  hipLaunchKernelGGL(dflash_inputs_kernel, dim3((unsigned)((T + n_q + 255) / 256)), dim3(256), 0,
                     reinterpret_cast<hipStream_t>(stream), anchors, valid, (int)n_q, block_size, T, mask_token,
                     input_ids, positions, loss_mask, mask_kind, from_anchor, ids, kv_pos, target_row, aligned, outside);
  return check_launch(__func__);
}

extern "C" int spx_dflash_inputs(const int64_t* anchors, const uint8_t* valid, int64_t n_anchors, int32_t block_size,
                                 int64_t T, int64_t mask_token, const int64_t* input_ids, const int64_t* positions,
                                 const void* loss_mask, int mask_kind, int from_anchor, int64_t* ids, int64_t* kv_pos,
                                 int64_t* target_row, float* aligned, void* stream) {
  return spx_dflash_inputs_checked(anchors, valid, n_anchors, block_size, T, mask_token, input_ids, positions, loss_mask,
                                   mask_kind, from_anchor, ids, kv_pos, target_row, aligned, nullptr, stream);
}
