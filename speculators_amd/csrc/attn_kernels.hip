// Draft-model attention for gfx950: EAGLE3 test-time-training (TTT) attention
// and DFlash anchored-block attention, forward and backward, from one family
// of interval-masked flash-attention kernels.
//
// Every query row r sees up to two key INTERVALS of the K/V rows, plus (TTT
// only) a few single keys:
//   * context keys      a1[r] <= c < b1[r]          (rows [0, T) of K/V)
//   * block keys    T + a2[r] <= c < T + b2[r]      (rows [T, T+NQ): DFlash's own
//                                                    mask-token block)
//   * TTT diagonal keys: rows j*T + r, j = 1..n_extra -- ONE key per earlier
//     step, handled as n_extra dot products per row instead of 128x128 tiles.
// TTT:    a1 = row_lo (document start / window / the row itself for padding),
//         b1 = r + 1, no block interval.
// DFlash: a1 = max(doc start, anchor - W), b1 = anchor, a2/b2 = the query's own
//         block (all of it, or up to the query under a causal window layer).
// Key tiles that no row of a workgroup can see are skipped analytically; no
// dense mask or BlockMask exists anywhere.

#include <algorithm>
#include <mutex>
#include <type_traits>

#include "attn_common.h"
#include "../../include/spx.h"

namespace spx {

struct AttnParams {
  const uint16_t* Q; int64_t q_hs;   // [Hq][NQ][D]
  const uint16_t* K; int64_t k_hs;   // [Hkv][>= NKV (+ n_extra*T)][D]
  const uint16_t* V; int64_t v_hs;
  const int32_t* a1; const int32_t* b1;  // b1 == nullptr: b1[r] = r + 1
  const int32_t* a2; const int32_t* b2;  // nullptr: no block interval
  int NQ, T, NKV, NKVp;  // NKVp: row length of the transposed operands (multiple of 128)
  int n_extra, Hq, Hkv;
  float scale_log2e, scaling;
};

// ---------------------------------------------------------------- mask descriptors
// largest value of the lower threads of a workgroup of 1024 (-1: none)
__device__ __forceinline__ int lower_max(int v) {
  __shared__ int wave_top[16];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const int o = __shfl_up(v, d, 64);
    if (lane >= d) v = max(v, o);
  }
  if (lane == 63) wave_top[wave] = v;
  __syncthreads();
  const int up = __shfl_up(v, 1, 64);
  int carry = lane > 0 ? up : -1;
  for (int w = 0; w < wave; ++w) carry = max(carry, wave_top[w]);
  return carry;
}

// (one workgroup: a walk over the run starts of up to 1023 lower threads in LDS made this 8.5 us at any length)
template <typename I>
__global__ __launch_bounds__(1024) void ttt_row_lo_kernel(const I* __restrict__ doc, int64_t T,
                                                          int64_t window, int32_t* __restrict__ lo) {
  const int t = threadIdx.x;
  const int64_t len = (T + 1023) / 1024;
  const int64_t b = t * len, e = (b + len < T) ? b + len : T;
  int run = -1;
  for (int64_t i = b; i < e; ++i)
    if (i == 0 || doc[i] != doc[i - 1]) run = (int)i;
  run = lower_max(run);
  for (int64_t i = b; i < e; ++i) {
    if (i == 0 || doc[i] != doc[i - 1]) run = (int)i;
    int v = run;
    if (doc[i] == (I)-1) v = (int)i;
    else if (window > 0 && i - window + 1 > v) v = (int)(i - window + 1);
    lo[i] = v;
  }
}

// start of the run of equal document ids that contains position i
template <typename I>
__global__ __launch_bounds__(1024) void doc_run_start_kernel(const I* __restrict__ doc, int64_t T,
                                                             int32_t* __restrict__ start) {
  const int t = threadIdx.x;
  const int64_t len = (T + 1023) / 1024;
  const int64_t b = t * len, e = (b + len < T) ? b + len : T;
  int run = -1;
  for (int64_t i = b; i < e; ++i)
    if (i == 0 || doc[i] != doc[i - 1]) run = (int)i;
  run = lower_max(run);
  for (int64_t i = b; i < e; ++i) {
    if (i == 0 || doc[i] != doc[i - 1]) run = (int)i;
    start[i] = run;
  }
}

template <typename I, typename J>
__global__ __launch_bounds__(256) void dflash_ranges_kernel(
    const I* __restrict__ doc, const int32_t* __restrict__ run_start, const J* __restrict__ anchors,
    int64_t n_anchors, int block_size, int64_t window, int causal_block, int64_t T,
    int32_t* __restrict__ a1, int32_t* __restrict__ b1, int32_t* __restrict__ a2,
    int32_t* __restrict__ b2) {
  const int64_t r = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (r >= n_anchors * block_size) return;
  const int64_t j = r / block_size;
  int64_t a = (int64_t)anchors[j];
  a = a < 0 ? 0 : (a >= T ? T - 1 : a);
  int lo = 0, hi = 0;
  if (doc[a] != (I)-1) {
    lo = run_start[a];
    if (window > 0 && a - window > lo) lo = (int)(a - window);
    hi = (int)a;
    if (hi < lo) hi = lo;
  }
  a1[r] = lo;
  b1[r] = hi;
  a2[r] = (int)(j * block_size);
  b2[r] = causal_block ? (int)(r + 1) : (int)((j + 1) * block_size);
}

// Eight bf16 values times a scalar, rounded back to bf16 (round to nearest even).  The queries
// enter every score product as bf16(q * scale * log2 e): the forward, the dQ kernel (both scale
// their register fragments with this function) and the dK/dV and diagonal-key kernels (which
// read the copy the dQ kernel writes with it) must see the SAME rounded values, or the
// probabilities the backward recomputes would not match the forward's log-sum-exp.
__device__ __forceinline__ u32x4 scale_bf16x8(u32x4 raw, float c) {
  u32x4 w;
  w.x = pack_bf16x2(bf16_lo(raw.x) * c, bf16_hi(raw.x) * c);
  w.y = pack_bf16x2(bf16_lo(raw.y) * c, bf16_hi(raw.y) * c);
  w.z = pack_bf16x2(bf16_lo(raw.z) * c, bf16_hi(raw.z) * c);
  w.w = pack_bf16x2(bf16_lo(raw.w) * c, bf16_hi(raw.w) * c);
  return w;
}

// ---------------------------------------------------------------- transpose
// dst[h][c][perm(r)] = src[h][r][c] for r < rows, c < cols, up to a multiple of 64 of r (zeros past the end): columns ld_dst
// apart, their groups of 32 r ld_32 apart (32: one run per column; 32 * cols and ld_dst = 32: blocks of 32 r, all columns of
// a block together, which a kernel that takes 32 r at a time reads in whole lines).  perm swaps bits
// 2 and 3 of r: inside every group of 16 the order is 0-3, 8-11, 4-7, 12-15, which puts
// the 8 rows a lane half needs as MFMA k-slots (4 g + 0..3 and 8 + 4 g + 0..3) side by
// side, so that operand is ONE 16-byte LDS read.
// One wave per 64 x 64 tile, no LDS: a lane loads an 8 (r) x 8 (c) block with eight 16-byte row loads
// (eight lanes read a whole 128-byte line), transposes it in registers (v_perm_b32) and writes, for each
// of its 8 columns, the two 4-row halves of the block to their permuted places (8 bytes each; the eight
// lanes that share a column fill its 128-byte line in two store instructions).  cols a multiple of 8.
__global__ __launch_bounds__(64) void transpose_bf16_kernel(
    const uint16_t* __restrict__ src, int64_t src_hs, int64_t src_ld, int rows, int cols,
    uint16_t* __restrict__ dst, int64_t dst_hs, int64_t ld_dst, int64_t ld_32) {
  const int h = blockIdx.z;
  const int lane = threadIdx.x;
  const int rb = lane >> 3, cb = lane & 7;
  const int r0 = blockIdx.x * 64 + rb * 8, c0 = blockIdx.y * 64 + cb * 8;
  if (c0 >= cols) return;
  const uint16_t* s = src + (int64_t)h * src_hs + c0;
  u32x4 in[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const u32x4 z = {0, 0, 0, 0};
    in[j] = (r0 + j < rows) ? *reinterpret_cast<const u32x4*>(s + (int64_t)(r0 + j) * src_ld) : z;
  }
  // where the block's two halves go: r0 % 16 == 0 -> r0 and r0 + 8, r0 % 16 == 8 -> r0 - 4 and r0 + 4
  const int p_lo = ((r0 & 8) ? r0 - 4 : r0) & 31, p_hi = ((r0 & 8) ? r0 + 4 : r0 + 8) & 31;
  uint16_t* d = dst + (int64_t)h * dst_hs + (int64_t)c0 * ld_dst + (r0 >> 5) * ld_32;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    // column c0 + i of the block: element e = in[e] element i
    const uint32_t sel = (i & 1) ? 0x07060302u : 0x05040100u;
    const int w = i >> 1;
    u32x2 lo, hi;
    lo.x = __builtin_amdgcn_perm(in[1][w], in[0][w], sel);
    lo.y = __builtin_amdgcn_perm(in[3][w], in[2][w], sel);
    hi.x = __builtin_amdgcn_perm(in[5][w], in[4][w], sel);
    hi.y = __builtin_amdgcn_perm(in[7][w], in[6][w], sel);
    *reinterpret_cast<u32x2*>(d + (int64_t)i * ld_dst + p_lo) = lo;
    *reinterpret_cast<u32x2*>(d + (int64_t)i * ld_dst + p_hi) = hi;
  }
}

// per-lane intervals of the NSB query rows a lane owns, and their wave / block extents
template <int NSB>
struct RowBounds {
  int a1[NSB], b1[NSB], a2[NSB], b2[NSB];
  int w_a1min, w_a1max, w_b1min, w_b1max;
  int w_a2min, w_a2max, w_b2min, w_b2max;
  int blk_a1, blk_b1, blk_a2, blk_b2;
};

// value of the partner lane (lane ^ 32) combined with the own one, through v_permlane32_swap
// (a VALU move) instead of an LDS permute: swapping (x, x) leaves the lower half of the wave's
// values in every lane of the first result and the upper half in the second
__device__ __forceinline__ float half_swap_max(float x) {
  const uint32_t u = __float_as_uint(x);
  const auto s = __builtin_amdgcn_permlane32_swap(u, u, false, false);
  return fmaxf(__uint_as_float(s[0]), __uint_as_float(s[1]));
}
__device__ __forceinline__ float half_swap_sum(float x) {
  const uint32_t u = __float_as_uint(x);
  const auto s = __builtin_amdgcn_permlane32_swap(u, u, false, false);
  return __uint_as_float(s[0]) + __uint_as_float(s[1]);
}

__device__ __forceinline__ int wave_min_i(int v) {
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) v = min(v, __shfl_xor(v, m, 64));
  return v;
}
__device__ __forceinline__ int wave_max_i(int v) {
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) v = max(v, __shfl_xor(v, m, 64));
  return v;
}

template <int NSB, int NW>
__device__ __forceinline__ void load_bounds(const AttnParams& p, const int (&ic)[NSB], int wave,
                                            int lane, int* red /* [4 * NW] LDS */, RowBounds<NSB>& rb) {
  int a1mn = 0x7fffffff, a1mx = 0, b1mn = 0x7fffffff, b1mx = 0;
  int a2mn = 0x7fffffff, a2mx = 0, b2mn = 0x7fffffff, b2mx = 0;
#pragma unroll
  for (int sb = 0; sb < NSB; ++sb) {
    rb.a1[sb] = p.a1[ic[sb]];
    rb.b1[sb] = p.b1 ? p.b1[ic[sb]] : ic[sb] + 1;
    if (p.a2) {
      rb.a2[sb] = p.T + p.a2[ic[sb]];
      rb.b2[sb] = p.T + p.b2[ic[sb]];
    } else {
      rb.a2[sb] = 0; rb.b2[sb] = 0;
    }
    a1mn = min(a1mn, rb.a1[sb]); a1mx = max(a1mx, rb.a1[sb]);
    b1mn = min(b1mn, rb.b1[sb]); b1mx = max(b1mx, rb.b1[sb]);
    a2mn = min(a2mn, rb.a2[sb]); a2mx = max(a2mx, rb.a2[sb]);
    b2mn = min(b2mn, rb.b2[sb]); b2mx = max(b2mx, rb.b2[sb]);
  }
  // wave-uniform values are moved to scalar registers: the tests on them then compile to
  // scalar branches (a masked and an unmasked tile path) instead of per-lane selects
  auto uni = [](int v) { return __builtin_amdgcn_readfirstlane(v); };
  rb.w_a1min = uni(wave_min_i(a1mn)); rb.w_a1max = uni(wave_max_i(a1mx));
  rb.w_b1min = uni(wave_min_i(b1mn)); rb.w_b1max = uni(wave_max_i(b1mx));
  rb.w_a2min = uni(wave_min_i(a2mn)); rb.w_a2max = uni(wave_max_i(a2mx));
  rb.w_b2min = uni(wave_min_i(b2mn)); rb.w_b2max = uni(wave_max_i(b2mx));
  if (lane == 0) {
    red[wave * 4 + 0] = rb.w_a1min; red[wave * 4 + 1] = rb.w_b1max;
    red[wave * 4 + 2] = rb.w_a2min; red[wave * 4 + 3] = rb.w_b2max;
  }
  __syncthreads();
  rb.blk_a1 = red[0]; rb.blk_b1 = red[1]; rb.blk_a2 = red[2]; rb.blk_b2 = red[3];
#pragma unroll
  for (int w = 1; w < NW; ++w) {
    rb.blk_a1 = min(rb.blk_a1, red[w * 4 + 0]); rb.blk_b1 = max(rb.blk_b1, red[w * 4 + 1]);
    rb.blk_a2 = min(rb.blk_a2, red[w * 4 + 2]); rb.blk_b2 = max(rb.blk_b2, red[w * 4 + 3]);
  }
  rb.blk_a1 = uni(rb.blk_a1); rb.blk_b1 = uni(rb.blk_b1);
  rb.blk_a2 = uni(rb.blk_a2); rb.blk_b2 = uni(rb.blk_b2);
}

// Four 16-bit values per lane from LDS, transposed inside every group of 16 lanes: lane 4u + w of
// a group receives, as element j, element w of the 8 bytes that lane 4j + u of the group points at.
typedef short i16x4 __attribute__((ext_vector_type(4)));
typedef short i16x8 __attribute__((ext_vector_type(8)));
__device__ __forceinline__ i16x4 lds_tr16(uint32_t addr) {
  return __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) i16x4*)(uintptr_t)addr);
}
__device__ __forceinline__ i16x4 lds_read_tr16(const uint8_t* p) {
  return lds_tr16((uint32_t)(uintptr_t)(__attribute__((address_space(3))) const uint8_t*)p);
}

// Passes a score block through an empty volatile asm statement.  Placed inside the branch that
// masks a tile it keeps the compiler from turning that branch into selects which every tile, masked
// or not, would then execute (96 vector instructions per tile): volatile asm is never speculated.
__device__ __forceinline__ void pin_block(f32x16& a) {
  asm volatile("" : "+v"(a[0]), "+v"(a[1]), "+v"(a[2]), "+v"(a[3]), "+v"(a[4]), "+v"(a[5]), "+v"(a[6]), "+v"(a[7]));
  asm volatile("" : "+v"(a[8]), "+v"(a[9]), "+v"(a[10]), "+v"(a[11]), "+v"(a[12]), "+v"(a[13]), "+v"(a[14]), "+v"(a[15]));
}

// f(integral_constant<int, B>) .. f(integral_constant<int, E - 1>): a loop that is unrolled whatever its size
template <int B, int E, typename F>
__device__ __forceinline__ void static_for(F&& f) {
  if constexpr (B < E) {
    f(std::integral_constant<int, B>{});
    static_for<B + 1, E>(f);
  }
}

// The 32 x 32 x 16 product of a kernel of one wave per SIMD (512 registers, half of them accumulation registers, which only
// matrix instructions and loads can use).  The builtin's results lie in accumulation registers there, and every score costs a
// move in and a move out.  Here the results lie in ordinary registers and the operands that no vector instruction
// touches (A: just read from LDS; B of the score products: the queries) in the others.  The compiler does not see that an asm
// statement is a matrix instruction: whoever reads a result keeps twelve issue slots clear of the last product on
// it (three products behind it do: each takes the pipe for eight).  Nor does it keep a vector instruction that writes an
// operand two issue slots away from the product (mfma32_operand).
#if SPX_MFMA_BUILTIN
__device__ __forceinline__ void mfma32_from(f32x16& d, bf16x8 a, bf16x8 b, const f32x16& c) { d = mfma32(a, b, c); }
__device__ __forceinline__ void mfma32_onto(f32x16& d, bf16x8 a, bf16x8 b) { d = mfma32(a, b, d); }
__device__ __forceinline__ void mfma32_onto_v(f32x16& d, bf16x8 a, bf16x8 b) { d = mfma32(a, b, d); }
#else
__device__ __forceinline__ void mfma32_from(f32x16& d, bf16x8 a, bf16x8 b, const f32x16& c) {
  asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, %3" : "=&v"(d) : "a"(a), "a"(b), "v"(c));
}
__device__ __forceinline__ void mfma32_onto(f32x16& d, bf16x8 a, bf16x8 b) {
  asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, %0" : "+v"(d) : "a"(a), "a"(b));
}
__device__ __forceinline__ void mfma32_onto_v(f32x16& d, bf16x8 a, bf16x8 b) {  // B in ordinary registers
  asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, %0" : "+v"(d) : "a"(a), "v"(b));
}
#endif
// a product's operand is complete: not to be formed any later, and two issue slots from here to the product
__device__ __forceinline__ void mfma32_operand(u32x4& x) { asm volatile("s_nop 1" : "+v"(x)); }
__device__ __forceinline__ void mfma32_operand(f32x16& x) { asm volatile("s_nop 1" : "+v"(x)); }
// every product under way has arrived
template <int N>
__device__ __forceinline__ void mfma32_drain(f32x16 (&d)[N]) {
  asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");
#pragma unroll
  for (int i = 0; i < N; ++i) asm volatile("" : "+v"(d[i]));
}

// ---------------------------------------------------------------- forward
// One workgroup = 4 waves = 4 * 32 * NSB query rows of one head (NSB = 2: a wave owns two 32-row
// sub-blocks and every K / V^T fragment read from LDS feeds two MFMAs; the kernels run NSB = 1).
// Wave priorities (s_setprio) per phase, (matrix phase, vector phase) per kernel; equal values = no changes.
// Forward: the wave that is in its soft-max gets the higher priority.  Its vector instructions are short and
// slot in between the MFMAs of the other wave, which needs one issue slot per 32 cycles; the other way
// round (matrix phase first) the vector wave waits behind MFMAs that are themselves waiting for the pipe
// (measured at the Llama-3.1-8B shape: 825 TFLOP/s with the matrix phase first, 826 without priorities, 880
// with the vector phase first).  The dQ and dK/dV kernels measure best with the matrix phase first.
#define SPX_FWD_PRIO 0, 3
#define SPX_DQ_PRIO 3, 0
#define SPX_DKV_PRIO 3, 0
constexpr int prio_first(int a, int) { return a; }
constexpr int prio_second(int, int b) { return b; }
template <int M, int V>
struct PrioPair {
  static __device__ __forceinline__ void matrix() { if constexpr (M != V) __builtin_amdgcn_s_setprio(M); }
  static __device__ __forceinline__ void vector() { if constexpr (M != V) __builtin_amdgcn_s_setprio(V); }
};
#define SPX_FWD_PRIO_MFMA() PrioPair<prio_first(SPX_FWD_PRIO), prio_second(SPX_FWD_PRIO)>::matrix()
#define SPX_FWD_PRIO_VALU() PrioPair<prio_first(SPX_FWD_PRIO), prio_second(SPX_FWD_PRIO)>::vector()
#define SPX_DQ_PRIO_MFMA() PrioPair<prio_first(SPX_DQ_PRIO), prio_second(SPX_DQ_PRIO)>::matrix()
#define SPX_DQ_PRIO_VALU() PrioPair<prio_first(SPX_DQ_PRIO), prio_second(SPX_DQ_PRIO)>::vector()
#define SPX_DKV_PRIO_MFMA() PrioPair<prio_first(SPX_DKV_PRIO), prio_second(SPX_DKV_PRIO)>::matrix()
#define SPX_DKV_PRIO_VALU() PrioPair<prio_first(SPX_DKV_PRIO), prio_second(SPX_DKV_PRIO)>::vector()
#define SPX_FWD_MINB 2
#define SPX_DQ_MINB 2
// A key tile is 64 rows of K and of V as they lie in memory, brought global -> LDS directly into the other of two tile
// buffers: a 16-byte LDS write from registers holds the LDS pipe twice as long as a 16-byte read, and these kernels keep
// that pipe busy all the time.  The transposed operand of the second product comes out of the row-major tile through
// transposing LDS reads (dQ: K^T; forward, TR: V^T), or, in larger forward calls, out of a copy V^T made once per call: two
// 8-byte reads for one of 16 cost the forward 5 - 6 %, the copy is a launch of 4 us (fwd_tr).
template <int D, int NW>
struct FwdSmem {
  static constexpr int kTile = kBN * D * 2;  // unpadded, swizzled
  static constexpr int kBuf = 2 * kTile;     // K, V
  static constexpr int kTiles = 2 * kBuf;
  static constexpr int kBytes = kTiles + 4 * NW * (int)sizeof(int);
};

// operand fragments in flight per product (registers: 4 per fragment): the LDS pipe delivers
// well over 150 B/clk per CU, what a wave waits for is the latency of its own reads
#define SPX_FWD_RING 8
template <int D, int NSB, int NW, bool TR>
__global__ __launch_bounds__(64 * NW, D > 128 ? 1 : SPX_FWD_MINB) void attn_fwd_kernel(AttnParams p,
                                                                const uint16_t* __restrict__ Vt,
                                                                uint16_t* __restrict__ O,
                                                                float* __restrict__ LSE) {
  using SM = FwdSmem<D, NW>;
  constexpr int NKK = D / 16;
  constexpr int NDB = D / 32;
  constexpr int BMW = 32 * NSB;
  constexpr int BM = NW * BMW;

  extern __shared__ __attribute__((aligned(16))) uint8_t fwd_smem[];
  int* const red = reinterpret_cast<int*>(fwd_smem + SM::kTiles);

  const int group = p.Hq / p.Hkv;
  const int L = blockIdx.x;
  const int kvh = L % p.Hkv;
  const int rest = L / p.Hkv;
  const int h = kvh * group + rest % group;
  const int n_qb = (p.NQ + BM - 1) / BM;
  const int qb = n_qb - 1 - rest / group;  // late (heavy, under a causal mask) blocks first
  const int m0 = qb * BM;

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // in a scalar register: what derives from it is scalar too
  const int g = lane >> 5, col = lane & 31;
  int i[NSB], ic[NSB];
#pragma unroll
  for (int sb = 0; sb < NSB; ++sb) {
    i[sb] = m0 + wave * BMW + sb * 32 + col;
    ic[sb] = i[sb] < p.NQ ? i[sb] : p.NQ - 1;
  }
  RowBounds<NSB> rb;
  load_bounds<NSB, NW>(p, ic, wave, lane, red, rb);

  // The query fragments carry the soft-max scale and log2(e): the scores then come out of the
  // MFMA in the base-2 exponent domain and need no multiply of their own.
  bf16x8 qf[NSB][NKK];
#pragma unroll
  for (int sb = 0; sb < NSB; ++sb) {
    const uint16_t* qrow = p.Q + (int64_t)h * p.q_hs + (int64_t)ic[sb] * D + g * 8;
#pragma unroll
    for (int kk = 0; kk < NKK; ++kk)
      qf[sb][kk] = as_bf16x8(scale_bf16x8(*reinterpret_cast<const u32x4*>(qrow + kk * 16), p.scale_log2e));
  }
  // Soft-max bookkeeping per query (a lane owns one query; its partner lane ^ 32 the same one):
  //   m_ref  the value subtracted from the scores before the exp2.  It is NOT the running maximum:
  //          it only moves when a tile's largest score exceeds it by more than kRefSlack (or when
  //          the row sees its first key), so most tiles skip the rescaling pass altogether.  A
  //          common factor 2^k on a row's probabilities is exact in binary floating point and
  //          cancels in O / l; the slack only has to keep 2^(s - m_ref) far from overflow.
  //   nref   -m_ref in all sixteen accumulator slots: the C operand of the first score MFMA, so
  //          the subtraction costs no instruction.
  //   l_run  this LANE's part of the row sum (its 32 of a tile's 64 keys); the halves are added
  //          once, after the last tile.
  constexpr float kRefSlack = 12.f;
  f32x16 acc[NSB][NDB], nref[NSB];
  float m_ref[NSB], l_run[NSB];
#pragma unroll
  for (int sb = 0; sb < NSB; ++sb) {
    m_ref[sb] = -INFINITY; l_run[sb] = 0.f;  // -inf: the row has not seen a key yet
#pragma unroll
    for (int r = 0; r < 16; ++r) nref[sb][r] = 0.f;
#pragma unroll
    for (int db = 0; db < NDB; ++db)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[sb][db][r] = 0.f;
  }

  const uint16_t* Kh = p.K + (int64_t)kvh * p.k_hs;
  const uint16_t* Vh = p.V + (int64_t)kvh * p.v_hs;
  const int last_row = p.NKV - 1;

  // ---- tiles as 1 KB wave loads global -> LDS: rows of D * 2 bytes (V^T: 128 bytes), the 16-byte chunk c of row r in
  // slot c ^ swz(r).  K and V^T (32 lanes = 32 rows, one chunk) and V (transposing reads: 4 + 4 rows x 64 bytes, see the dQ
  // kernel) are read differently and swizzled for their own kind of read: conflict free without padding.
  constexpr int RBK = D * 2, CKK = RBK / 16;             // bytes and chunks per row
  constexpr int LPK = (kBN * RBK / 1024) / NW;           // wave loads per wave and tile
  auto swz_k = [](int r) { return CKK == 8 ? (r >> 1) & 7 : r & 15; };
  auto swz_v = [](int r) { return CKK == 8 ? ((r & 4) | ((r >> 2) & 2) | ((r >> 1) & 1)) : ((r & 3) << 2) | ((r >> 2) & 3); };
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)fwd_smem;
  const u32x4 kres = make_rsrc(Kh, (uint32_t)((int64_t)p.NKV * RBK));
  const uint16_t* const Vth = Vt + (int64_t)kvh * D * p.NKVp;
  const u32x4 vres = TR ? make_rsrc(Vh, (uint32_t)((int64_t)p.NKV * RBK))
                        : make_rsrc(Vth, (uint32_t)((int64_t)D * p.NKVp * 2));
  constexpr int LPV = (D * 128 / 1024) / NW;             // V^T tile
  auto swz_vt = [](int r) { return (r >> 1) & 7; };
  constexpr bool kWide = D > 128;  // one wave per SIMD: see wide_pass
  int k_row[TR || kWide ? 1 : LPK], k_col[TR || kWide ? 1 : LPK], v_off[TR || kWide ? 1 : LPV];
  if constexpr (!TR && !kWide) {
#pragma unroll
    for (int j = 0; j < LPK; ++j) {
      const int r = (wave * LPK + j) * (1024 / RBK) + lane / CKK;
      k_row[j] = r;
      k_col[j] = ((lane % CKK) ^ swz_k(r)) * 16;
    }
#pragma unroll
    for (int j = 0; j < LPV; ++j) {
      const int r = (wave * LPV + j) * 8 + lane / 8;
      v_off[j] = r * p.NKVp * 2 + ((lane & 7) ^ swz_vt(r)) * 16;
    }
  }
  auto issue = [&](int n0, int buf) __attribute__((always_inline)) {
    if constexpr (!TR) {
      const uint32_t kb = lds0 + buf * SM::kBuf + wave * LPK * 1024;
      if (n0 + kBN <= p.NKV) {
        // every row of the tile exists: the lane's offset inside a tile is loop invariant, the tile's
        // first row goes into the scalar offset (no vector arithmetic per load)
#pragma unroll
        for (int j = 0; j < LPK; ++j) load_to_lds16<0>(kres, kb + j * 1024, k_row[j] * RBK + k_col[j], n0 * RBK);
      } else {
#pragma unroll
        for (int j = 0; j < LPK; ++j)
          load_to_lds16<0>(kres, kb + j * 1024, min(n0 + k_row[j], last_row) * RBK + k_col[j], 0);
      }
      const uint32_t vb = lds0 + buf * SM::kBuf + SM::kTile + wave * LPV * 1024;
#pragma unroll
      for (int j = 0; j < LPV; ++j) load_to_lds16<0>(vres, vb + j * 1024, v_off[j], n0 * 2);
      return;
    }
    // (offsets recomputed per tile: four vector instructions per load against 2 LPK registers)
    int lane_v = lane;
    if (D > 64) asm volatile("" : "+v"(lane_v));
    const uint32_t kb = lds0 + buf * SM::kBuf + wave * LPK * 1024, vb = kb + SM::kTile;
    const bool whole = n0 + kBN <= p.NKV;
#pragma unroll
    for (int j = 0; j < LPK; ++j) {
      const int r = (wave * LPK + j) * (1024 / RBK) + lane_v / CKK;
      const int ck = ((lane_v % CKK) ^ swz_k(r)) * 16, cv = ((lane_v % CKK) ^ swz_v(r)) * 16;
      if (whole) {
        // every row of the tile exists: its first row goes into the scalar offset
        load_to_lds16<0>(kres, kb + j * 1024, r * RBK + ck, n0 * RBK);
        load_to_lds16<0>(vres, vb + j * 1024, r * RBK + cv, n0 * RBK);
      } else {
        // the last, ragged tile: rows past the end repeat the last one (they are masked out)
        const int rr = min(n0 + r, last_row) * RBK;
        load_to_lds16<0>(kres, kb + j * 1024, rr + ck, 0);
        load_to_lds16<0>(vres, vb + j * 1024, rr + cv, 0);
      }
    }
  };
  // fragment reads: byte offsets of this lane's row and chunk (step 0) inside a K tile
  const int rdk = col * RBK + ((g ^ swz_k(col)) * 16);
  // ... and of the rows 4 (G >> 1) + (s >> 2) (+ 8) of a 16-key step inside a V tile (lane s of 16-lane group G)
  const int tG = lane >> 4, ts = lane & 15;
  const int trow = 4 * (tG >> 1) + (ts >> 2);
  const int tcl = 2 * (tG & 1) + ((ts & 3) >> 1);
  const int rt0 = trow * RBK + ((tcl ^ swz_v(trow)) * 16) + (ts & 1) * 8;
  const int rt1 = (trow + 8) * RBK + ((tcl ^ swz_v(trow + 8)) * 16) + (ts & 1) * 8;
  // The fragment reads as LDS addresses, one register per swizzle term, kept opaque to the
  // compiler: what is added to them per read (buffer, key half, 16-key step) is a constant and goes
  // into the offset field.  Formed on the symbol of the dynamic array instead, every read costs a
  // vector add of that link-time constant.  (Both tile buffers lie inside the 64 KB an offset field reaches.)
  const int rdv = col * 128 + ((g ^ swz_vt(col)) * 16);
  uint32_t krd[NKK], vrd0[TR ? NDB : 1], vrd1[TR ? NDB : 1], vrd[TR ? 1 : 4];
  if constexpr (!kWide) {
#pragma unroll
    for (int j = 0; j < NKK; ++j) {
      krd[j] = lds0 + (uint32_t)(rdk ^ (j * 32));
      asm volatile("" : "+v"(krd[j]));
    }
    if constexpr (!TR) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        vrd[j] = lds0 + (uint32_t)(SM::kTile + (rdv ^ (j * 32)));
        asm volatile("" : "+v"(vrd[j]));
      }
    }
#pragma unroll
    for (int j = 0; j < (TR ? NDB : 0); ++j) {
      vrd0[j] = lds0 + (uint32_t)(SM::kTile + (rt0 ^ (j * 64)));
      vrd1[j] = lds0 + (uint32_t)(SM::kTile + (rt1 ^ (j * 64)));
      asm volatile("" : "+v"(vrd0[j]), "+v"(vrd1[j]));
    }
  }

  // one pass over the key tiles of one interval class.  The tile loop is unrolled over the two tile
  // buffers: the buffer is then a compile-time constant and the fragment reads address it through
  // the immediate offset of ds_read (no vector add per read).
  auto run_pass = [&](const int (&aa)[NSB], const int (&bb)[NSB], int w_amin, int w_amax,
                      int w_bmin, int w_bmax, int blk_a, int blk_b) {
    if (blk_b <= blk_a) return;
    const int n_begin = (blk_a / kBN) * kBN;
    __syncthreads();  // a previous pass may still be reading either buffer
    issue(n_begin, 0);
    auto tile = [&](int n0, auto buf_c) __attribute__((always_inline)) {
      constexpr int buf = decltype(buf_c)::value;
      // this wave's loads of tile n0 have landed; after the barrier everybody's have, and nobody
      // reads the other buffer any more: the next tile goes there
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();
      if (n0 + kBN < blk_b) issue(n0 + kBN, buf ^ 1);
      if (n0 >= w_bmax || n0 + kBN <= w_amin) return;  // nothing visible for this wave

      f32x16 st[NSB][2];
      SPX_FWD_PRIO_MFMA();
      // K fragments go through a ring of four registers: the read of fragment f + 4 is
      // issued right after the MFMA of fragment f, so no MFMA waits for LDS; the two
      // 32-key halves alternate so that consecutive MFMAs use different accumulators
      {
        constexpr int NF = 2 * NKK;
        constexpr int RG = SPX_FWD_RING;
        bf16x8 kfr[RG];
        auto kread = [&](int f) {
          kfr[f % RG] = as_bf16x8(lds_read128(krd[f >> 1] + buf * SM::kBuf + (f & 1) * 32 * RBK));
        };
#pragma unroll
        for (int f = 0; f < RG; ++f) kread(f);
#pragma unroll
        for (int f = 0; f < NF; ++f) {
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int sb = 0; sb < NSB; ++sb)
            st[sb][f & 1] = mfma32(kfr[f % RG], qf[sb][f >> 1], f < 2 ? nref[sb] : st[sb][f & 1]);
          __builtin_amdgcn_sched_barrier(0);
          if (f + RG < NF) kread(f + RG);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      SPX_FWD_PRIO_VALU();
      const bool need_mask = (n0 < w_amax) || (n0 + kBN > w_bmin);
      int m_lo[NSB], m_hi[NSB];
#pragma unroll
      for (int sb = 0; sb < NSB; ++sb) { m_lo[sb] = aa[sb] - n0 - 4 * g; m_hi[sb] = bb[sb] - n0 - 4 * g; }
#pragma unroll
      for (int sb = 0; sb < NSB; ++sb) {
        // running max on the raw scores; the soft-max scale is folded into the exp2 argument
        if (need_mask) {
          // a real (scalar) branch: the asm statement keeps the compiler from turning the
          // masking into selects that every tile would pay for
#pragma unroll
          for (int kb = 0; kb < 2; ++kb) {
            pin_block(st[sb][kb]);
#pragma unroll
            for (int r = 0; r < 16; ++r) {
              // key index = n0 + 4 g + (compile-time part): compare the constant part
              const int cr = kb * 32 + 8 * (r >> 2) + (r & 3);
              if (cr < m_lo[sb] || cr >= m_hi[sb]) st[sb][kb][r] = -INFINITY;
            }
            pin_block(st[sb][kb]);
          }
        }
        // st holds s - m_ref.  Largest of the 32 scores of this lane (three-operand maxima)
        float mx = fmaxf(st[sb][0][0], st[sb][1][0]);
#pragma unroll
        for (int r = 1; r < 16; r += 2) {
          mx = fmaxf(fmaxf(mx, st[sb][0][r]), st[sb][0][r + 1 < 16 ? r + 1 : r]);
          mx = fmaxf(fmaxf(mx, st[sb][1][r]), st[sb][1][r + 1 < 16 ? r + 1 : r]);
        }
        mx = half_swap_max(mx);
        const bool unset = m_ref[sb] == -INFINITY;
        const bool move = mx > -INFINITY && (unset || mx > kRefSlack);
        if (__any(move)) {
          // some row's reference moves: shift its scores, rescale its sum and its accumulator
          asm volatile("; reference moves");
          const float delta = move ? mx : 0.f;
          const float alpha = (move && !unset) ? fast_exp2(-delta) : 1.f;  // unset rows hold zeros
          m_ref[sb] = move ? (unset ? mx : m_ref[sb] + mx) : m_ref[sb];
          const float nr = unset && !move ? 0.f : -m_ref[sb];
#pragma unroll
          for (int r = 0; r < 16; ++r) nref[sb][r] = nr;
#pragma unroll
          for (int kb = 0; kb < 2; ++kb)
#pragma unroll
            for (int r = 0; r < 16; ++r) st[sb][kb][r] -= delta;
          l_run[sb] *= alpha;
#pragma unroll
          for (int db = 0; db < NDB; ++db)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[sb][db][r] *= alpha;
        }
        float rs0 = 0.f, rs1 = 0.f;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const float p0 = fast_exp2(st[sb][0][r]), p1 = fast_exp2(st[sb][1][r]);
          st[sb][0][r] = p0; st[sb][1][r] = p1;
          rs0 += p0; rs1 += p1;
        }
        l_run[sb] += rs0 + rs1;
      }
      SPX_FWD_PRIO_MFMA();
      {
        // V^T fragments through the same kind of ring; fragment f = (16-key step s, D block db)
        constexpr int NF = 4 * NDB;
        constexpr int RG = SPX_FWD_RING;
        bf16x8 vfr[RG];
        auto vread = [&](int f) {
          if constexpr (!TR) {
            vfr[f % RG] = as_bf16x8(lds_read128(vrd[f / NDB] + buf * SM::kBuf + (f % NDB) * 32 * 128));
            return;
          }
          const i16x4 lo = lds_tr16(vrd0[f % NDB] + buf * SM::kBuf + (f / NDB) * 16 * RBK);
          const i16x4 hi = lds_tr16(vrd1[f % NDB] + buf * SM::kBuf + (f / NDB) * 16 * RBK);
          vfr[f % RG] = __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
        };
#pragma unroll
        for (int f = 0; f < RG; ++f) vread(f);
        bf16x8 pb[NSB];
#pragma unroll
        for (int f = 0; f < NF; ++f) {
          const int s = f / NDB, db = f % NDB;
          if (db == 0) {
#pragma unroll
            for (int sb = 0; sb < NSB; ++sb) pb[sb] = pack8(st[sb][s >> 1], (s & 1) * 8);
          }
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int sb = 0; sb < NSB; ++sb) acc[sb][db] = mfma32(vfr[f % RG], pb[sb], acc[sb][db]);
          __builtin_amdgcn_sched_barrier(0);
          if (f + RG < NF) vread(f + RG);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      SPX_FWD_PRIO_VALU();
    };
    for (int n0 = n_begin; n0 < blk_b; n0 += 2 * kBN) {
      tile(n0, std::integral_constant<int, 0>{});
      if (n0 + kBN < blk_b) tile(n0 + kBN, std::integral_constant<int, 1>{});
    }
  };

  // head_dim 256: the accumulators leave one wave per SIMD, so whatever this wave waits for its matrix pipe waits for too, and
  // every other instruction has to be issued while a product runs (32 cycles each).  A tile is one unbroken row of 64 products
  // in four quarters, each with a share of the rest beside it:
  //   S0  scores of keys 0 - 31               second half of the soft-max of the last tile's keys 32 - 63; loads of K
  //   O1  O += V^T P, LAST tile's keys 32 - 63   first half of the soft-max of keys 0 - 31; loads of V
  //   S1  scores of keys 32 - 63              second half of the soft-max of keys 0 - 31
  //   O0  O += V^T P, keys 0 - 31             first half of the soft-max of keys 32 - 63; the one barrier of the tile, four
  //                                           products from the end, and the next tile's first reads behind it
  // Operand fragments run sixteen products ahead through one ring.  V lies in LDS in halves of 32 keys, a ring of four: the second
  // half of a tile is used, and so loaded, one tile late.  Soft-max reference and masking as in run_pass, per half.
  // 16384 causal rows, 16 heads of 256, two K/V heads: 2375 us in the form of the other head sizes (all scores, the whole
  // soft-max, all of O: matrix pipe busy 38 % of the cycles at 2.0 GHz, 176 moves between the register files per tile), 1800
  // like this (62 % at 1.7 GHz: at the power limit); 600 rows 32.0 and 23.0.  The soft-max inside its own tile (two quarters
  // without it, two with all of it) 1946; a ring of eight operands instead of sixteen 1 % more; V^T out of rows of the whole
  // length, 64 bytes per load and row, in the place of blocks of 32 keys 12 % more.
  // (auto: head sizes that do not call it get no body of it, whose fragments their arrays have no room for)
  auto wide_pass = [&](auto a_i, int b_i, int w_amin, int w_amax, int w_bmin, int w_bmax, int blk_a, int blk_b) {
    static_assert(NSB == 1, "one 32-row block per wave");
    if (blk_b <= blk_a) return;
    constexpr int RG = 16;
    constexpr uint32_t kVoff = 2 * SM::kTile, kHalf = SM::kTile / 2;
    int n0 = (blk_a / kBN) * kBN;
    uint32_t par = 0;  // K buffer and pair of V halves of tile n0: 0 or kTile
    // The lane's places in the first load of K and V; a later load of the tile is an XOR and an immediate away.  Rows past the
    // end come in as zeros (they are masked out).  Formed for every tile: kept over the loop they would not leave room for the
    // operands.
    struct Places { int k, v; };
    auto places = [&]() __attribute__((always_inline)) {
      int at = lane;
      asm volatile("" : "+v"(at));
      const int b5 = at >> 5;
      Places pl;
      pl.k = (wave * 16 + b5) * RBK + ((at & 31) ^ b5) * 16;
      pl.v = TR ? (wave * 8 + b5) * RBK + ((at & 31) ^ (b5 << 2) ^ ((wave & 1) << 1)) * 16
                : wave * 4096 + (at >> 2) * 64 + ((at & 3) ^ ((at >> 4) & 3)) * 16;
      return pl;
    };
    // load j (0 .. 7) of a wave's share of K tile n, load j (0 .. 3) of half h of V tile n
    auto issue_k = [&](const Places& pl, int n, uint32_t to, auto jc) __attribute__((always_inline)) {
      constexpr int j = decltype(jc)::value;
      const u32x4 res = make_rsrc(Kh + (int64_t)n * D, (uint32_t)(p.NKV - n) * RBK);
      load_to_lds16<(j & 3) * 1024>(res, lds0 + to + wave * 8192 + (j >> 2) * 4096, pl.k ^ (32 * j | (j >> 2) << 12), 0);
    };
    auto issue_v = [&](const Places& pl, int n, int h2, uint32_t to, auto jc) __attribute__((always_inline)) {
      constexpr int j = decltype(jc)::value;
      const uint32_t dst = lds0 + kVoff + to + h2 * kHalf + wave * 4096;
      if constexpr (TR) {
        const int row = min(n + 32 * h2, p.NKV);
        const u32x4 res = make_rsrc(Vh + (int64_t)row * D, (uint32_t)(p.NKV - row) * RBK);
        load_to_lds16<j * 1024>(res, dst, pl.v ^ (((j & 1) << 7) | ((j >> 1) << 4)), 0);
      } else {
        load_to_lds16<j * 1024>(vres, dst, pl.v, (n + 32 * h2) * (D * 2));  // (blocks of 32 keys: transpose_bf16_kernel)
      }
    };
    // the sixteen loads of a tile: K and the first half of V of tile n1, the second half of tile n0
    auto issue = [&](const Places& pl, int n1, auto jc) __attribute__((always_inline)) {
      constexpr int j = decltype(jc)::value;
      if constexpr (j < 8) issue_k(pl, n1, SM::kTile - par, jc);
      else if constexpr (j < 12) issue_v(pl, n1, 0, SM::kTile - par, std::integral_constant<int, j - 8>{});
      else issue_v(pl, n0, 1, par, std::integral_constant<int, j - 12>{});
    };

    // fragment addresses, one register per swizzle term; the rest is in the offset field.  kr: K buffer of tile n0; vr0, vr1: V
    // halves of the last tile until S1, then of this one
    uint32_t kr[8], vr0[TR ? 4 : 2], vr1[TR ? 4 : 1];
#pragma unroll
    for (int j = 0; j < 8; ++j) kr[j] = lds0 + (uint32_t)(rdk ^ (j * 32));
    if constexpr (TR) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        vr0[j] = lds0 + kVoff + SM::kTile + (uint32_t)(rt0 ^ (j * 64));
        vr1[j] = lds0 + kVoff + SM::kTile + (uint32_t)(rt1 ^ (j * 64));
      }
    } else {
#pragma unroll
      for (int j = 0; j < 2; ++j)
        vr0[j] = lds0 + kVoff + SM::kTile + (uint32_t)(col * 64 + (((g + 2 * j) ^ ((col >> 2) & 3)) * 16));
    }
    bf16x8 fr[RG];
    auto fread = [&](auto fc) __attribute__((always_inline)) {
      constexpr int f = decltype(fc)::value;
      if constexpr ((f & 16) == 0) {
        constexpr int kk = f & 15;
        fr[f % RG] = as_bf16x8(lds_read128(kr[kk & 7] + (f >> 5) * 32 * RBK + (kk >> 3) * 256));
      } else {
        constexpr int h2 = f < 32, s = (f >> 3) & 1, db = f & 7;
        if constexpr (!TR) {
          fr[f % RG] = as_bf16x8(lds_read128(vr0[s] + h2 * kHalf + db * 32 * 64));
        } else {
          const i16x4 lo = lds_tr16(vr0[db & 3] + h2 * kHalf + s * 16 * RBK + (db >> 2) * 256);
          const i16x4 hi = lds_tr16(vr1[db & 3] + h2 * kHalf + s * 16 * RBK + (db >> 2) * 256);
          fr[f % RG] = __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
        }
      }
    };

    f32x16 st[2];
    u32x4 pb[2][2];
    bf16x8 qa[NKK];
#pragma unroll
    for (int kk = 0; kk < NKK; ++kk) {
      qa[kk] = qf[0][kk];
      asm volatile("" : "+a"(qa[kk]));  // (else a copy of them lives in ordinary registers and moves over for every tile)
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) st[1][r] = 0.f;
    float mx = 0.f, rs = 0.f;
    float slack = m_ref[0] == -INFINITY ? -INFINITY : kRefSlack;  // a row without a reference takes its first one
    bool need_mask = false;
    auto slots = [] { __builtin_amdgcn_sched_barrier(0); };
    // the soft-max of one half in 32 pieces, one beside each product of two quarters; its scores are complete from piece 3 on
    auto soft = [&](auto half_c, auto piece_c) __attribute__((always_inline)) {
      constexpr int h2 = decltype(half_c)::value, pc = decltype(piece_c)::value;
      f32x16& s = st[h2];
      if constexpr (pc == 3) {
        asm volatile("" : "+v"(s));
        if (need_mask) {
          const int m_lo = a_i - n0 - 4 * g, m_hi = b_i - n0 - 4 * g;
          asm volatile("" : "+v"(s));
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            const int cr = h2 * 32 + 8 * (r >> 2) + (r & 3);
            if (cr < m_lo || cr >= m_hi) s[r] = -INFINITY;
          }
          asm volatile("" : "+v"(s));
        }
        mx = fmaxf(s[0], s[1]);
#pragma unroll
        for (int r = 2; r < 8; r += 2) mx = fmaxf(fmaxf(mx, s[r]), s[r + 1]);
      } else if constexpr (pc == 4) {
#pragma unroll
        for (int r = 8; r < 16; r += 2) mx = fmaxf(fmaxf(mx, s[r]), s[r + 1]);
      } else if constexpr (pc == 5) {
        mx = half_swap_max(mx);
      } else if constexpr (pc == 6) {
        const bool move = mx > slack;
        if (__builtin_amdgcn_ballot_w64(move) != 0) {
          // some row's reference moves: its sum, what O has taken so far, and the probabilities of the half whose products
          // are under way
          mfma32_drain(st);
          mfma32_drain(acc[0]);
          const bool unset = m_ref[0] == -INFINITY;
          const float delta = move ? mx : 0.f;
          const float alpha = (move && !unset) ? fast_exp2(-delta) : 1.f;  // unset rows hold zeros
          m_ref[0] = move ? (unset ? mx : m_ref[0] + mx) : m_ref[0];
          slack = move ? kRefSlack : slack;
          const float nr = unset && !move ? 0.f : -m_ref[0];
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            nref[0][r] = nr;
            s[r] -= delta;
            st[1 - h2][r] *= alpha;
          }
          pb[1 - h2][0] = __builtin_bit_cast(u32x4, pack8(st[1 - h2], 0));
          pb[1 - h2][1] = __builtin_bit_cast(u32x4, pack8(st[1 - h2], 8));
          mfma32_operand(pb[1 - h2][0]);
          mfma32_operand(pb[1 - h2][1]);
          l_run[0] *= alpha;
#pragma unroll
          for (int db = 0; db < NDB; ++db)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[0][db][r] *= alpha;
          // (a wait that does not name the registers leaves the compiler free to scale the last of them behind it)
          mfma32_operand(nref[0]);
#pragma unroll
          for (int db = 0; db < NDB; ++db) mfma32_operand(acc[0][db]);
        }
        rs = 0.f;
      } else if constexpr (pc >= 7 && pc < 23) {
        s[pc - 7] = fast_exp2(s[pc - 7]);
        rs += s[pc - 7];
      } else if constexpr (pc >= 23 && pc < 31) {
        constexpr int w = pc - 23;
        pb[h2][w >> 2][w & 3] = pack_bf16x2(s[2 * w], s[2 * w + 1]);
        if constexpr ((w & 3) == 3) mfma32_operand(pb[h2][w >> 2]);
      } else if constexpr (pc == 31) {
        l_run[0] += rs;
      }
    };

    // everybody's reads of this tile are done and the next one has landed: over to its buffers
    auto next_tile = [&]() __attribute__((always_inline)) {
      asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
      __syncthreads();
      const uint32_t d = SM::kTile - 2 * par;
#pragma unroll
      for (int j = 0; j < 8; ++j) kr[j] += d;
      par = SM::kTile - par;
      n0 = __builtin_amdgcn_readfirstlane(n0 + kBN);
    };
    // the V addresses from tile n0 - 64 to tile n0 (first: whatever they are at, to n0)
    auto next_v = [&]() __attribute__((always_inline)) {
      const uint32_t d = 2 * par - SM::kTile;
#pragma unroll
      for (int j = 0; j < (TR ? 4 : 2); ++j) {
        vr0[j] += d;
        if constexpr (TR) vr1[j] += d;
      }
    };
    // (past the last tile: this one's loads again, nobody reads them)
    auto ahead = [&]() __attribute__((always_inline)) { return n0 + kBN < blk_b ? n0 + kBN : n0; };
    // tiles that this wave sees nothing of (a run at either end): its share of the loads
    auto skip_to = [&](int stop) __attribute__((always_inline)) {
#pragma unroll 1
      while (n0 < stop) {
        const int n1 = ahead();
        const Places pl = places();
        static_for<0, 16>([&](auto j) __attribute__((always_inline)) { issue(pl, n1, j); });
        next_tile();
      }
    };
    auto tile = [&](auto first_c) __attribute__((always_inline)) {
      constexpr bool first = decltype(first_c)::value;
      const int n1 = ahead();
      const Places pl = places();
      static_for<0, 16>([&](auto fc) __attribute__((always_inline)) {
        constexpr int f = decltype(fc)::value;
        slots();
        if constexpr (f == 0) mfma32_from(st[0], fr[f % RG], qa[f], nref[0]);
        else mfma32_onto(st[0], fr[f % RG], qa[f]);
        slots();
        fread(std::integral_constant<int, f + RG + (first ? 16 : 0)>{});
        if constexpr (!first) soft(std::integral_constant<int, 1>{}, std::integral_constant<int, 16 + f>{});
        if constexpr (f % 2 == 0) issue(pl, n1, std::integral_constant<int, f / 2>{});
      });
      need_mask = (n0 < w_amax) || (n0 + kBN > w_bmin);
      if constexpr (first) mfma32_drain(st);
      static_for<0, 16>([&](auto fc) __attribute__((always_inline)) {
        constexpr int f = decltype(fc)::value;
        if constexpr (!first) {
          slots();
          mfma32_onto_v(acc[0][f & 7], fr[f % RG], as_bf16x8(pb[1][f >> 3]));
          slots();
          fread(std::integral_constant<int, 16 + f + RG>{});
        }
        soft(std::integral_constant<int, 0>{}, fc);
        if constexpr (f % 2 == 0) issue(pl, n1, std::integral_constant<int, 8 + f / 2>{});
      });
      slots();
      next_v();
      static_for<0, 16>([&](auto fc) __attribute__((always_inline)) {
        constexpr int f = decltype(fc)::value;
        slots();
        if constexpr (f == 0) mfma32_from(st[1], fr[f % RG], qa[f], nref[0]);
        else mfma32_onto(st[1], fr[f % RG], qa[f]);
        slots();
        fread(std::integral_constant<int, 32 + f + RG>{});
        soft(std::integral_constant<int, 0>{}, std::integral_constant<int, 16 + f>{});
      });
      static_for<0, 16>([&](auto fc) __attribute__((always_inline)) {
        constexpr int f = decltype(fc)::value;
        slots();
        mfma32_onto_v(acc[0][f & 7], fr[f % RG], as_bf16x8(pb[0][f >> 3]));
        slots();
        soft(std::integral_constant<int, 1>{}, fc);
        if constexpr (f == 8) next_tile();
        if constexpr (f >= 8) {
          fread(std::integral_constant<int, 2 * f - 16>{});
          fread(std::integral_constant<int, 2 * f - 15>{});
        }
      });
      slots();
    };

    __syncthreads();  // a previous pass may still be reading its buffers
    {
      const Places pl = places();
      static_for<0, 8>([&](auto j) __attribute__((always_inline)) { issue_k(pl, n0, 0, j); });
      static_for<0, 4>([&](auto j) __attribute__((always_inline)) { issue_v(pl, n0, 0, 0, j); });
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    skip_to(min(w_amin - kBN + 1, blk_b));
    const int seen = min(w_bmax, blk_b);
    if (n0 < seen) {
#pragma unroll
      for (int j = 0; j < (TR ? 4 : 2); ++j) {  // where the tile before the first one would lie
        vr0[j] -= par;
        if constexpr (TR) vr1[j] -= par;
      }
      static_for<0, RG>([&](auto f) __attribute__((always_inline)) { fread(f); });
      tile(std::true_type{});
#pragma unroll 1
      while (n0 < seen) tile(std::false_type{});
      // the last tile's keys 32 - 63
      mfma32_drain(st);
      static_for<16, 32>([&](auto pc) __attribute__((always_inline)) { soft(std::integral_constant<int, 1>{}, pc); });
      static_for<16, 16 + RG>([&](auto f) __attribute__((always_inline)) { fread(f); });
      static_for<0, 16>([&](auto fc) __attribute__((always_inline)) {
        constexpr int f = decltype(fc)::value;
        slots();
        mfma32_onto_v(acc[0][f & 7], fr[f % RG], as_bf16x8(pb[1][f >> 3]));
        slots();
      });
      mfma32_drain(acc[0]);
    }
    skip_to(blk_b);
  };

  if constexpr (kWide) {
#pragma unroll 1
    for (int c = 0; c < (p.a2 ? 2 : 1); ++c)  // (one copy of the code for both interval classes)
      wide_pass(c ? rb.a2[0] : rb.a1[0], c ? rb.b2[0] : rb.b1[0], c ? rb.w_a2min : rb.w_a1min, c ? rb.w_a2max : rb.w_a1max,
                c ? rb.w_b2min : rb.w_b1min, c ? rb.w_b2max : rb.w_b1max, c ? rb.blk_a2 : rb.blk_a1,
                c ? rb.blk_b2 : rb.blk_b1);
  } else {
    run_pass(rb.a1, rb.b1, rb.w_a1min, rb.w_a1max, rb.w_b1min, rb.w_b1max, rb.blk_a1, rb.blk_b1);
    if (p.a2)
      run_pass(rb.a2, rb.b2, rb.w_a2min, rb.w_a2max, rb.w_b2min, rb.w_b2max, rb.blk_a2, rb.blk_b2);
  }

  // from here on l_run is the whole row's sum in both lanes of a query
#pragma unroll
  for (int sb = 0; sb < NSB; ++sb) l_run[sb] = half_swap_sum(l_run[sb]);
  float (&m_run)[NSB] = m_ref;

  // TTT diagonal keys (j, r), j = 1..n_extra: one dot product each.  The key / value rows of a
  // wave's 32 queries are 32 CONSECUTIVE rows of step j: they come in as whole 1 KB wave loads
  // global -> LDS (a lane reading its own row from global memory touches 32 lines per instruction)
  // into this wave's quarter of the tile buffers, chunk c of row r in slot c ^ (r mod chunks), and
  // each lane then picks its row's pieces from LDS.  The loads of step j + 1 are issued as soon
  // as step j's rows have been read.
  if (p.n_extra > 0) {
    static_assert(NSB == 1, "one 32-row block per wave");
    constexpr int XCK = RBK / 16;                  // 16-byte chunks per row
    constexpr int XRL = 1024 / RBK;                // rows per 1 KB wave load
    constexpr int XNL = 32 / XRL;                  // wave loads per 32 rows
    static_assert(SM::kTiles / NW >= 2 * 32 * RBK, "a wave's share of the tile buffers holds K and V rows");
    __syncthreads();  // every wave is done with the tile buffers
    const uint32_t xk = lds0 + wave * (2 * 32 * RBK), xv = xk + 32 * RBK;
    const int64_t kv_bytes = (int64_t)(p.n_extra + 1) * p.T * RBK;
    const u32x4 xkres = make_rsrc(p.K + (int64_t)kvh * p.k_hs, (uint32_t)kv_bytes);
    const u32x4 xvres = make_rsrc(p.V + (int64_t)kvh * p.v_hs, (uint32_t)kv_bytes);
    int goff[XNL];
#pragma unroll
    for (int n = 0; n < XNL; ++n) {
      const int r = n * XRL + lane / XCK;
      goff[n] = r * RBK + (((lane % XCK) ^ (r & (XCK - 1))) * 16);
    }
    const int row0 = __builtin_amdgcn_readfirstlane(m0 + wave * BMW);
    auto issue_x = [&](const u32x4& res, uint32_t dst, int j) __attribute__((always_inline)) {
      const int soff = __builtin_amdgcn_readfirstlane((j * p.T + row0) * RBK);
#pragma unroll
      for (int n = 0; n < XNL; ++n) load_to_lds16<0>(res, dst + n * 1024, goff[n], soff);
    };
    const uint8_t* const xkp = fwd_smem + wave * (2 * 32 * RBK);
    const uint8_t* const xvp = xkp + 32 * RBK;
    const int xrow = col * RBK, xsw = col & (XCK - 1);
    issue_x(xkres, xk, 1);
    issue_x(xvres, xv, 1);
    for (int j = 1; j <= p.n_extra; ++j) {
      // K rows of step j have landed (the V rows, issued after them, may still be in flight)
      if constexpr (XNL == 8) asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
      else if constexpr (XNL == 4) asm volatile("s_waitcnt vmcnt(4)" ::: "memory");
      else asm volatile("s_waitcnt vmcnt(16)" ::: "memory");
      float dot = 0.f;
#pragma unroll
      for (int kk = 0; kk < NKK; ++kk)
        dot = dot8_bf16(qf[0][kk], *reinterpret_cast<const u32x4*>(xkp + xrow + (((2 * kk + g) ^ xsw) * 16)), dot);
      const float sj = half_swap_sum(dot);  // the query fragments carry the scale
      asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");  // V rows landed, K rows read
      if (j < p.n_extra) issue_x(xkres, xk, j + 1);
      const float m_new = fmaxf(m_run[0], sj);
      const float alpha = fast_exp2(m_run[0] - m_new);  // a row without context keys: exp2(-inf) = 0
      const float pv = fast_exp2(sj - m_new);
      l_run[0] = l_run[0] * alpha + pv;
      m_run[0] = m_new;
#pragma unroll
      for (int db = 0; db < NDB; ++db)
#pragma unroll
        for (int r4 = 0; r4 < 4; ++r4) {
          float vv[4];
          unpack4(*reinterpret_cast<const u32x2*>(xvp + xrow + (((db * 4 + r4) ^ xsw) * 16) + 8 * g), vv);
#pragma unroll
          for (int t = 0; t < 4; ++t)
            acc[0][db][r4 * 4 + t] = fmaf(pv, vv[t], acc[0][db][r4 * 4 + t] * alpha);
        }
      if (j < p.n_extra) {
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // V rows read
        issue_x(xvres, xv, j + 1);
      }
    }
  }

#pragma unroll
  for (int sb = 0; sb < NSB; ++sb) {
    if (i[sb] >= p.NQ) continue;
    const float inv = l_run[sb] > 0.f ? 1.f / l_run[sb] : 0.f;
    uint16_t* orow = O + ((int64_t)i[sb] * p.Hq + h) * D + 4 * g;
#pragma unroll
    for (int db = 0; db < NDB; ++db)
#pragma unroll
      for (int r4 = 0; r4 < 4; ++r4) {
        u32x2 w;
        w.x = pack_bf16x2(acc[sb][db][r4 * 4 + 0] * inv, acc[sb][db][r4 * 4 + 1] * inv);
        w.y = pack_bf16x2(acc[sb][db][r4 * 4 + 2] * inv, acc[sb][db][r4 * 4 + 3] * inv);
        *reinterpret_cast<u32x2*>(orow + db * 32 + 8 * r4) = w;
      }
    // a row that sees no key at all (cannot happen for the two masks built here) gets lse = 0
    if (g == 0) LSE[(int64_t)h * p.NQ + i[sb]] = l_run[sb] > 0.f ? m_run[sb] + fast_log2(l_run[sb]) : 0.f;
  }
}

// ---------------------------------------------------------------- backward
// delta[h, i] = sum_d dO[i, h, d] * O[i, h, d]
// sum over each row of sixteen lanes, left in every lane of the row
__device__ __forceinline__ float row16_sum(float v) {
  // quad_perm [1,0,3,2], quad_perm [2,3,0,1], row_half_mirror, row_mirror: afterwards every lane
  // of a 16-lane row holds the sum over the row
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0xB1, 0xf, 0xf, true));
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x4E, 0xf, 0xf, true));
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x141, 0xf, 0xf, true));
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x140, 0xf, 0xf, true));
  return v;
}

// EPL (4, 8 or 16) consecutive bf16 of one lane in 8- or 16-byte accesses
template <int EPL>
__device__ __forceinline__ void ld_bf16s(const uint16_t* p, float (&v)[EPL]) {
  if constexpr (EPL == 4) {
    const u32x2 u = *reinterpret_cast<const u32x2*>(p);
    v[0] = bf16_lo(u.x); v[1] = bf16_hi(u.x); v[2] = bf16_lo(u.y); v[3] = bf16_hi(u.y);
  } else {
    static_assert(EPL % 8 == 0, "4, 8 or 16 elements per lane");
#pragma unroll
    for (int c = 0; c < EPL / 8; ++c) {
      const u32x4 u = *reinterpret_cast<const u32x4*>(p + 8 * c);
      v[8 * c + 0] = bf16_lo(u.x); v[8 * c + 1] = bf16_hi(u.x);
      v[8 * c + 2] = bf16_lo(u.y); v[8 * c + 3] = bf16_hi(u.y);
      v[8 * c + 4] = bf16_lo(u.z); v[8 * c + 5] = bf16_hi(u.z);
      v[8 * c + 6] = bf16_lo(u.w); v[8 * c + 7] = bf16_hi(u.w);
    }
  }
}
template <int EPL>
__device__ __forceinline__ void st_bf16s(uint16_t* p, const float (&v)[EPL]) {
  if constexpr (EPL == 4) {
    u32x2 u;
    u.x = pack_bf16x2(v[0], v[1]); u.y = pack_bf16x2(v[2], v[3]);
    *reinterpret_cast<u32x2*>(p) = u;
  } else {
#pragma unroll
    for (int c = 0; c < EPL / 8; ++c) {
      u32x4 u;
      u.x = pack_bf16x2(v[8 * c + 0], v[8 * c + 1]); u.y = pack_bf16x2(v[8 * c + 2], v[8 * c + 3]);
      u.z = pack_bf16x2(v[8 * c + 4], v[8 * c + 5]); u.w = pack_bf16x2(v[8 * c + 6], v[8 * c + 7]);
      *reinterpret_cast<u32x4*>(p + 8 * c) = u;
    }
  }
}

// What the dK / dV and diagonal-key kernels read next to the operands: the dQ kernel, which runs first and holds a row's q
// and dO in registers anyway, leaves it behind.  (A prologue of its own read q, O and dO once more: 5 us and a launch at 1024
// rows of 32 heads of 64, 26 us at 4096 of 128, 213 us at 2 x 16384 of 16 heads of 256.)
struct BwdSide {
  int NQp;          // rows rounded up to 128
  uint16_t* qs;     // [Hq][NQ][D]  bf16(q * scale * log2 e)
  float* delta;     // [Hq][NQ]     dO . O of the row
  float* neg;       // -lse and -delta, each [Hq][NQp], zero in the padding: C operands of the dK / dV score products
  int32_t* tb;      // [tile of 64 rows][8]  a1min, a1max, b1min, b1max, a2min, a2max, b2min, b2max
  int32_t* rows;    // [4][NQp]     a1, b1, T + a2, T + b2 as the kernels compare them (empty: class absent, padding)
};
// the last two, by one wave for one tile
__device__ __forceinline__ void interval_ends(const AttnParams& p, const BwdSide& sd, int tile, int lane) {
  const int r = tile * 64 + lane;
  const bool ok = r < p.NQ;
  const int a1 = ok ? p.a1[r] : 0x7fffffff;
  const int b1 = ok ? (p.b1 ? p.b1[r] : r + 1) : 0;
  const int a2 = (ok && p.a2) ? p.T + p.a2[r] : 0x7fffffff;
  const int b2 = (ok && p.a2) ? p.T + p.b2[r] : 0;
  sd.rows[r] = a1; sd.rows[sd.NQp + r] = b1; sd.rows[2 * (int64_t)sd.NQp + r] = a2; sd.rows[3 * (int64_t)sd.NQp + r] = b2;
  const int v[8] = {wave_min_i(a1), wave_max_i(a1), wave_min_i(b1), wave_max_i(b1),
                    wave_min_i(a2), wave_max_i(a2), wave_min_i(b2), wave_max_i(b2)};
  if (lane == 0 && tile * 64 < p.NQ) {
#pragma unroll
    for (int k = 0; k < 8; ++k) sd.tb[tile * 8 + k] = v[k];
  }
}

// dQ: same tiling as the forward (a workgroup covers 128 rows: BwdSide's padding).
//   P^T = exp2(S'^T - lse), dP^T = V dO^T, dS^T = P^T (dP^T - delta), dQ^T += K^T dS^T
template <int D, int NW>
struct DqSmem {
  // the row-major K and V tiles, 64 keys each; the K^T fragments of the dQ product come
  // out of the K tile through transposing LDS reads
  static constexpr int kTileK = kBN * D * 2;
  static constexpr int kBuf = 2 * kTileK;
  static constexpr int kDiag = NW * 2 * 32 * D * 2;  // K and V rows of 32 queries per wave (TTT diagonal keys)
  static constexpr bool kWide = D != 128;  // attn_bwd_dq_kernel's wide_pass
  static constexpr int kStages = D == 64 ? 3 : 2;
  static constexpr int kTiles = kStages * kBuf > kDiag ? kStages * kBuf : kDiag;
  static constexpr int kBytes = kTiles + 4 * NW * (int)sizeof(int);
};

template <int D, int NSB, int NW>
__global__ __launch_bounds__(64 * NW, D > 128 ? 1 : SPX_DQ_MINB) void attn_bwd_dq_kernel(
    AttnParams p, const uint16_t* __restrict__ O, const uint16_t* __restrict__ dO, const float* __restrict__ LSE,
    BwdSide sd, uint16_t* __restrict__ dQ, int64_t dq_hs) {
  using SM = DqSmem<D, NW>;
  constexpr int TB = kBN;
  constexpr int NKK = D / 16;
  constexpr int NDB = D / 32;
  constexpr int BMW = 32 * NSB;
  constexpr int BM = NW * BMW;

  extern __shared__ __attribute__((aligned(16))) uint8_t dq_smem[];
  int* const red = reinterpret_cast<int*>(dq_smem + SM::kTiles);

  const int group = p.Hq / p.Hkv;
  const int L = blockIdx.x;
  const int kvh = L % p.Hkv;
  const int rest = L / p.Hkv;
  const int h = kvh * group + rest % group;
  const int n_qb = (p.NQ + BM - 1) / BM;
  const int qb = n_qb - 1 - rest / group;
  const int m0 = qb * BM;

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 5, col = lane & 31;
  int i[NSB], ic[NSB];
  float lse_i[NSB], delta_i[NSB];
#pragma unroll
  for (int sb = 0; sb < NSB; ++sb) {
    i[sb] = m0 + wave * BMW + sb * 32 + col;
    ic[sb] = i[sb] < p.NQ ? i[sb] : p.NQ - 1;
    lse_i[sb] = LSE[(int64_t)h * p.NQ + ic[sb]];
  }
  if (h == 0)
    for (int t = wave; t < BM / 64; t += NW) interval_ends(p, sd, m0 / 64 + t, lane);
  RowBounds<NSB> rb;
  load_bounds<NSB, NW>(p, ic, wave, lane, red, rb);

  // the query fragments carry scale * log2(e) (see scale_bf16x8); -lse and -delta of the lane's
  // query sit in all sixteen slots of two blocks that the first MFMA of each product takes as its
  // C operand, so s - lse and dP - delta come out of the matrix pipe
  bf16x8 qf[NSB][NKK], dof[NSB][NKK];
  f32x16 nlse[NSB], ndel[NSB];
#pragma unroll
  for (int sb = 0; sb < NSB; ++sb) {
    const uint16_t* qrow = p.Q + (int64_t)h * p.q_hs + (int64_t)ic[sb] * D + g * 8;
    const uint16_t* drow = dO + ((int64_t)ic[sb] * p.Hq + h) * D + g * 8;
#pragma unroll
    for (int kk = 0; kk < NKK; ++kk) {
      qf[sb][kk] = as_bf16x8(scale_bf16x8(*reinterpret_cast<const u32x4*>(qrow + kk * 16), p.scale_log2e));
      dof[sb][kk] = as_bf16x8(*reinterpret_cast<const u32x4*>(drow + kk * 16));
    }
    // delta, and what the kernels behind this one read
    const uint16_t* orow = O + ((int64_t)ic[sb] * p.Hq + h) * D + g * 8;
    float dot = 0.f;
#pragma unroll
    for (int kk = 0; kk < NKK; ++kk) {
      float o8[8], d8[8];
      unpack8(*reinterpret_cast<const u32x4*>(orow + kk * 16), o8);
      unpack8(__builtin_bit_cast(u32x4, dof[sb][kk]), d8);
#pragma unroll
      for (int e = 0; e < 8; ++e) dot = fmaf(o8[e], d8[e], dot);
    }
    delta_i[sb] = half_swap_sum(dot);
    const bool live = i[sb] < p.NQ;
    if (live) {
      uint16_t* qrow_s = sd.qs + ((int64_t)h * p.NQ + i[sb]) * D + g * 8;
#pragma unroll
      for (int kk = 0; kk < NKK; ++kk)
        *reinterpret_cast<u32x4*>(qrow_s + kk * 16) = __builtin_bit_cast(u32x4, qf[sb][kk]);
    }
    if (g == 0) {
      if (live) sd.delta[(int64_t)h * p.NQ + i[sb]] = delta_i[sb];
      sd.neg[(int64_t)h * sd.NQp + i[sb]] = live ? -lse_i[sb] : 0.f;
      sd.neg[((int64_t)p.Hq + h) * sd.NQp + i[sb]] = live ? -delta_i[sb] : 0.f;
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) { nlse[sb][r] = -lse_i[sb]; ndel[sb][r] = -delta_i[sb]; }
  }
  f32x16 acc[NSB][NDB];
#pragma unroll
  for (int sb = 0; sb < NSB; ++sb)
#pragma unroll
    for (int db = 0; db < NDB; ++db)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[sb][db][r] = 0.f;

  const uint16_t* Kh = p.K + (int64_t)kvh * p.k_hs;
  const uint16_t* Vh = p.V + (int64_t)kvh * p.v_hs;
  const int last_row = p.NKV - 1;

  // ---- the two tiles as 1 KB wave loads global -> LDS (chunk c of row r in slot c ^ swz(r))
  constexpr int RBK = D * 2, CKK = RBK / 16;   // bytes / 16-byte chunks per row of K and V
  constexpr int LPK = (TB * RBK / 1024) / NW;
  // (transposing reads touch 4 + 4 rows x 64 bytes: those rows must fall into different 64-byte bank groups)
  auto swz_k = [](int r) { return CKK == 8 ? ((r & 4) | ((r >> 2) & 2) | ((r >> 1) & 1)) : ((r & 3) << 2) | ((r >> 2) & 3); };
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)dq_smem;
  const u32x4 kres = make_rsrc(Kh, (uint32_t)((int64_t)p.NKV * RBK));
  const u32x4 vres = make_rsrc(Vh, (uint32_t)((int64_t)p.NKV * RBK));
  auto issue = [&](int n0, int b) __attribute__((always_inline)) {
    int lane_v = lane;
    asm volatile("" : "+v"(lane_v));  // offsets recomputed per tile, not kept live
    const uint32_t kb0 = lds0 + b * SM::kBuf + wave * LPK * 1024;
#pragma unroll
    for (int j = 0; j < LPK; ++j) {
      const int r = (wave * LPK + j) * (1024 / RBK) + lane_v / CKK;
      const int off = min(n0 + r, last_row) * RBK + ((lane_v % CKK) ^ swz_k(r)) * 16;
      load_to_lds16<0>(kres, kb0 + j * 1024, off, 0);
      load_to_lds16<0>(vres, kb0 + SM::kTileK + j * 1024, off, 0);
    }
  };
  const int rdk = col * RBK + ((g ^ swz_k(col)) * 16);
  // transposing reads: lane s of 16-lane group G points at row 4 (G >> 1) + (s >> 2) (+ 8 for the second read) of a
  // 16-key step, bytes 8 (s & 3) of the 64-byte block 32 db + 16 (G & 1)
  const int tG = lane >> 4, ts = lane & 15;
  const int trow = 4 * (tG >> 1) + (ts >> 2);
  const int tcl = 2 * (tG & 1) + ((ts & 3) >> 1);
  const int rt0 = trow * RBK + ((tcl ^ swz_k(trow)) * 16) + (ts & 1) * 8;
  const int rt1 = (trow + 8) * RBK + ((tcl ^ swz_k(trow + 8)) * 16) + (ts & 1) * 8;

  auto run_pass = [&](const int (&aa)[NSB], const int (&bb)[NSB], int w_amin, int w_amax,
                      int w_bmin, int w_bmax, int blk_a, int blk_b) {
    if (blk_b <= blk_a) return;
    const int n_begin = (blk_a / TB) * TB;
    int buf = 0;
    __syncthreads();  // a previous pass may still be reading either buffer
    issue(n_begin, 0);
    for (int n0 = n_begin; n0 < blk_b; n0 += TB) {
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();
      if (n0 + TB < blk_b) issue(n0 + TB, buf ^ 1);
      const uint8_t* const tile = dq_smem + buf * SM::kBuf;
      buf ^= 1;
      if (n0 >= w_bmax || n0 + TB <= w_amin) continue;

      const bool need_mask = (n0 < w_amax) || (n0 + TB > w_bmin);
#pragma unroll
      for (int sb = 0; sb < NSB; ++sb) {
        // the 32-key halves of the tile one after the other: 32 score registers live
#pragma unroll
        for (int kb = 0; kb < TB / 32; ++kb) {
          f32x16 st, dp;
          // K and V fragments alternate through a ring of four registers (fragment 2 kk is
          // K, 2 kk + 1 is V): the read of fragment f + 4 follows the MFMA of fragment f
          SPX_DQ_PRIO_MFMA();
          {
            constexpr int NF = 2 * NKK;
            bf16x8 fr[4];
            auto fread = [&](int f) {
              fr[f & 3] = as_bf16x8(*reinterpret_cast<const u32x4*>(
                  tile + ((f & 1) ? SM::kTileK : 0) + kb * 32 * RBK + (rdk ^ ((f >> 1) * 32))));
            };
#pragma unroll
            for (int f = 0; f < 4; ++f) fread(f);
#pragma unroll
            for (int f = 0; f < NF; ++f) {
              __builtin_amdgcn_sched_barrier(0);
              if (f & 1) dp = mfma32(fr[f & 3], dof[sb][f >> 1], f == 1 ? ndel[sb] : dp);
              else st = mfma32(fr[f & 3], qf[sb][f >> 1], f == 0 ? nlse[sb] : st);
              __builtin_amdgcn_sched_barrier(0);
              if (f + 4 < NF) fread(f + 4);
            }
            __builtin_amdgcn_sched_barrier(0);
          }
          SPX_DQ_PRIO_VALU();
#pragma unroll
          for (int r = 0; r < 16; ++r) st[r] = fast_exp2(st[r]);
          if (need_mask) {
            // a real (scalar) branch, see the forward kernel
            const int lo = aa[sb] - n0 - 4 * g, hi = bb[sb] - n0 - 4 * g;
            pin_block(st);
#pragma unroll
            for (int r = 0; r < 16; ++r) {
              const int cr = kb * 32 + 8 * (r >> 2) + (r & 3);
              if (cr < lo || cr >= hi) st[r] = 0.f;
            }
            pin_block(st);
          }
#pragma unroll
          for (int r = 0; r < 16; ++r) dp[r] *= st[r];
          SPX_DQ_PRIO_MFMA();
          {
            // K^T fragments through the same kind of ring; fragment f = (16-key step s2, D block db)
            constexpr int NF = 2 * NDB;
            bf16x8 fr[4];
            auto fread = [&](int f) {
              const uint8_t* base = tile + (kb * 32 + (f / NDB) * 16) * RBK;
              const i16x4 lo = lds_read_tr16(base + (rt0 ^ ((f % NDB) * 64)));
              const i16x4 hi = lds_read_tr16(base + (rt1 ^ ((f % NDB) * 64)));
              fr[f & 3] = __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
            };
#pragma unroll
            for (int f = 0; f < 4 && f < NF; ++f) fread(f);
            bf16x8 db8 = pack8(dp, 0);
#pragma unroll
            for (int f = 0; f < NF; ++f) {
              if (f == NDB) db8 = pack8(dp, 8);
              __builtin_amdgcn_sched_barrier(0);
              acc[sb][f % NDB] = mfma32(fr[f & 3], db8, acc[sb][f % NDB]);
              __builtin_amdgcn_sched_barrier(0);
              if (f + 4 < NF) fread(f + 4);
            }
            __builtin_amdgcn_sched_barrier(0);
          }
          SPX_DQ_PRIO_VALU();
        }
      }
    }
  };

  // head_dim 256 with one wave per SIMD (see the forward's wide_pass), 64 with two: the 6 * D / 16 products of a tile in one row,
  // six sixths,
  //   S0, dP0, S1, dP1   scores and dP of keys 0 - 31 and 32 - 63
  //   O0, O1             dQ += K^T dS of the two halves
  // with the tile's loads beside the first two, the exponentials of a half beside its dP, its dS beside the sixth after that,
  // and the barrier and the next tile's first reads beside O1.
  // 16384 causal rows, 16 heads, two K/V heads: 3350 us in the form of the other head sizes (matrix pipe busy 48 % at 1.95 GHz,
  // 64 moves between the register files per half tile), 2520 like this (78 % at 1.6 GHz: at the power limit).  32 heads of 64:
  // 512 rows 15.7 and 14.7, 4096 125 and 114, 8192 under a window of 2048 209 and 196.  At head_dim 128 this needs more
  // registers than two waves of a SIMD have, and with one wave a call of more than one workgroup per compute unit loses:
  // 4096 rows of 32 heads 227 and 233, 8192 of 64 1370 and 1424 (1024 of 32: 32.2 and 27.8).
  // (auto: head sizes that do not call it get no body of it, whose fragments their arrays have no room for)
  auto wide_pass = [&](auto a_i, int b_i, int w_amin, int w_amax, int w_bmin, int w_bmax, int blk_a, int blk_b) {
    static_assert(NSB == 1, "one 32-row block per wave");
    if (blk_b <= blk_a) return;
    constexpr int RG = D > 64 ? 16 : 8, NS = SM::kStages;
    constexpr int kLoads = 2 * LPK;                 // of a wave and tile: rows of K, then of V
    constexpr int XRW = 1024 / RBK;                 // rows per load
    int n0 = (blk_a / TB) * TB;
    uint32_t buf = 0;
    // the lane's place in the first load of a tile, formed for every tile; rows past the end come in as zeros (masked out)
    auto place = [&]() __attribute__((always_inline)) {
      int at = lane;
      asm volatile("" : "+v"(at));
      const int r = wave * (LPK * XRW) + at / CKK;
      return r * RBK + ((at % CKK) ^ swz_k(r)) * 16;
    };
    auto issue = [&](int pl, int n, uint32_t to, auto jc) __attribute__((always_inline)) {
      constexpr int j = decltype(jc)::value % LPK;
      constexpr bool is_v = decltype(jc)::value >= LPK;
      const u32x4 res = make_rsrc((is_v ? Vh : Kh) + (int64_t)n * D, (uint32_t)(p.NKV - n) * RBK);
      // what the row j * XRW adds to the swizzle of the first load's row
      constexpr int dsw = CKK == 8 ? ((j & 1) << 1) : CKK == 16 ? (j & 3) : ((j & 1) << 3) | ((j >> 1) & 3);
      load_to_lds16<(j & 3) * 1024>(res, lds0 + to + (is_v ? SM::kTileK : 0) + wave * (LPK * 1024) + (j >> 2) * 4096,
                                    pl ^ (dsw << 4 | (j >> 2) << 12), 0);
    };
    // fragment addresses, one register per swizzle term: rows (K, V) and transposed (K)
    constexpr int NR = NKK < 8 ? NKK : 8, NT = NDB < 4 ? NDB : 4;
    uint32_t kr[NR], tr0[NT], tr1[NT];
#pragma unroll
    for (int j = 0; j < NR; ++j) kr[j] = lds0 + (uint32_t)(rdk ^ (j * 32));
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      tr0[j] = lds0 + (uint32_t)(rt0 ^ (j * 64));
      tr1[j] = lds0 + (uint32_t)(rt1 ^ (j * 64));
    }
    bf16x8 fr[RG];
    auto fread = [&](auto fc) __attribute__((always_inline)) {
      constexpr int f = decltype(fc)::value, part = f / NKK, i = f % NKK;
      if constexpr (part < 4) {  // K 0, V 0, K 1, V 1
        fr[f % RG] = as_bf16x8(lds_read128(kr[i % NR] + (part & 1) * SM::kTileK + (part >> 1) * 32 * RBK + (i / NR) * 256));
      } else {
        constexpr int db = i % NDB, off = (part - 4) * 32 * RBK + (i / NDB) * 16 * RBK + (db / NT) * 256;
        const i16x4 lo = lds_tr16(tr0[db % NT] + off), hi = lds_tr16(tr1[db % NT] + off);
        fr[f % RG] = __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
      }
    };
    f32x16 st[2], dp[2];
    u32x4 ds[2][2];
#pragma unroll
    for (int kk = 0; kk < NKK; ++kk) asm volatile("" : "+a"(qf[0][kk]), "+a"(dof[0][kk]));
    bool need_mask = false;
    auto slots = [] { __builtin_amdgcn_sched_barrier(0); };
    // p and dS of a half, piece by piece, beside the products from the first of its dP on (slot 0) to the end of the part
    // behind that
    auto soft = [&](auto half_c, auto slot_c) __attribute__((always_inline)) {
      constexpr int h2 = decltype(half_c)::value, sl = decltype(slot_c)::value;
      constexpr int EX = 16 / NKK;                               // exponentials per slot
      constexpr int P0 = NKK > 4 ? NKK + 4 : NKK + 3;            // dS: from this slot on
      constexpr int PN = (8 + 2 * NKK - P0 - 1) / (2 * NKK - P0);  // pairs per slot
      f32x16& s = st[h2];
      if constexpr (sl == 3) asm volatile("" : "+v"(s));  // its last product is three behind
      if constexpr (sl >= 3 && sl < NKK + 3) {
#pragma unroll
        for (int e = EX * (sl - 3); e < EX * (sl - 2); ++e) s[e] = fast_exp2(s[e]);
      }
      if constexpr (sl == NKK + 3) {
        asm volatile("" : "+v"(dp[h2]));
        if (need_mask) {
          const int lo = a_i - n0 - 4 * g, hi = b_i - n0 - 4 * g;
          asm volatile("" : "+v"(s));
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            const int cr = h2 * 32 + 8 * (r >> 2) + (r & 3);
            if (cr < lo || cr >= hi) s[r] = 0.f;
          }
          asm volatile("" : "+v"(s));
        }
      }
      if constexpr (sl >= P0) {
#pragma unroll
        for (int w = PN * (sl - P0); w < PN * (sl - P0 + 1) && w < 8; ++w) {
          ds[h2][w >> 2][w & 3] = pack_bf16x2(dp[h2][2 * w] * s[2 * w], dp[h2][2 * w + 1] * s[2 * w + 1]);
          if ((w & 3) == 3) mfma32_operand(ds[h2][w >> 2]);
        }
      }
    };
    // the next tile has landed (of the loads behind it kStages - 2 tiles are still under way) and everybody's reads of
    // this one are done
    auto next_tile = [&]() __attribute__((always_inline)) {
      asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"((NS - 2) * kLoads) : "memory");
      __syncthreads();
      const uint32_t d = buf + SM::kBuf < NS * SM::kBuf ? SM::kBuf : (uint32_t)-(NS - 1) * SM::kBuf;
#pragma unroll
      for (int j = 0; j < NR; ++j) kr[j] += d;
#pragma unroll
      for (int j = 0; j < NT; ++j) { tr0[j] += d; tr1[j] += d; }
      buf += d;
      n0 = __builtin_amdgcn_readfirstlane(n0 + TB);
    };
    // the tile whose loads go out beside this one's products, and where to: the buffer the last tile left
    // (past the last one: this tile's again, nobody reads them)
    auto ahead = [&]() __attribute__((always_inline)) { return n0 + (NS - 1) * TB < blk_b ? n0 + (NS - 1) * TB : n0; };
    auto behind = [&]() __attribute__((always_inline)) { return buf ? buf - SM::kBuf : (NS - 1) * SM::kBuf; };
    auto skip_to = [&](int stop) __attribute__((always_inline)) {
#pragma unroll 1
      while (n0 < stop) {
        const int n1 = ahead(), pl = place();
        static_for<0, kLoads>([&](auto j) __attribute__((always_inline)) { issue(pl, n1, behind(), j); });
        next_tile();
      }
    };
    __syncthreads();  // a previous pass may still be reading its buffers
    {
      const int pl = place();
      static_for<0, NS - 1>([&](auto tc) __attribute__((always_inline)) {
        constexpr int ti = decltype(tc)::value;
        const int n = n0 + ti * TB < blk_b ? n0 + ti * TB : n0;
        static_for<0, kLoads>([&](auto j) __attribute__((always_inline)) { issue(pl, n, ti * SM::kBuf, j); });
      });
    }
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"((NS - 2) * kLoads) : "memory");
    __syncthreads();
    skip_to(min(w_amin - TB + 1, blk_b));
    const int seen = min(w_bmax, blk_b);
    if (n0 < seen) {
      static_for<0, RG>([&](auto f) __attribute__((always_inline)) { fread(f); });
#pragma unroll 1
      do {
        need_mask = (n0 < w_amax) || (n0 + TB > w_bmin);
        const int n1 = ahead(), pl = place();
        const uint32_t to = behind();
        static_for<0, 6 * NKK>([&](auto fc) __attribute__((always_inline)) {
          constexpr int f = decltype(fc)::value, i = f % NKK, part = f / NKK, kEnd = 6 * NKK, kSync = kEnd - RG / 2;
          using I = std::integral_constant<int, i>;
          using I2 = std::integral_constant<int, i + NKK>;
          using H0 = std::integral_constant<int, 0>;
          using H1 = std::integral_constant<int, 1>;
          slots();
          if constexpr (part == 0 || part == 2) {
            if constexpr (i == 0) mfma32_from(st[part >> 1], fr[f % RG], qf[0][i], nlse[0]);
            else mfma32_onto(st[part >> 1], fr[f % RG], qf[0][i]);
          } else if constexpr (part == 1 || part == 3) {
            if constexpr (i == 0) mfma32_from(dp[part >> 1], fr[f % RG], dof[0][i], ndel[0]);
            else mfma32_onto(dp[part >> 1], fr[f % RG], dof[0][i]);
          } else {
            mfma32_onto_v(acc[0][i % NDB], fr[f % RG], as_bf16x8(ds[part - 4][i / NDB]));
          }
          slots();
          if constexpr (f + RG < kEnd) fread(std::integral_constant<int, f + RG>{});
          if constexpr (part == 1) soft(H0{}, I{});
          if constexpr (part == 2) soft(H0{}, I2{});
          if constexpr (part == 3) soft(H1{}, I{});
          if constexpr (part == 4) soft(H1{}, I2{});
          if constexpr (f < 2 * kLoads && f % 2 == 0) issue(pl, n1, to, std::integral_constant<int, f / 2>{});
          if constexpr (f == kSync) next_tile();
          if constexpr (f >= kSync) {
            fread(std::integral_constant<int, 2 * (f - kSync)>{});
            fread(std::integral_constant<int, 2 * (f - kSync) + 1>{});
          }
        });
        slots();
      } while (n0 < seen);
      mfma32_drain(acc[0]);
    }
    skip_to(blk_b);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // (nothing may land in memory that is used for something else next)
  };

  if constexpr (SM::kWide) {
#pragma unroll 1
    for (int c = 0; c < (p.a2 ? 2 : 1); ++c)  // (one copy of the code for both interval classes)
      wide_pass(c ? rb.a2[0] : rb.a1[0], c ? rb.b2[0] : rb.b1[0], c ? rb.w_a2min : rb.w_a1min, c ? rb.w_a2max : rb.w_a1max,
                c ? rb.w_b2min : rb.w_b1min, c ? rb.w_b2max : rb.w_b1max, c ? rb.blk_a2 : rb.blk_a1,
                c ? rb.blk_b2 : rb.blk_b1);
  } else {
    run_pass(rb.a1, rb.b1, rb.w_a1min, rb.w_a1max, rb.w_b1min, rb.w_b1max, rb.blk_a1, rb.blk_b1);
    if (p.a2)
      run_pass(rb.a2, rb.b2, rb.w_a2min, rb.w_a2max, rb.w_b2min, rb.w_b2max, rb.blk_a2, rb.blk_b2);
  }

  // TTT diagonal keys: the key / value rows of a wave's 32 queries come in as coalesced 1 KB wave
  // loads global -> LDS into the wave's share of the tile buffers (see the forward kernel)
  if (p.n_extra > 0) {
    static_assert(NSB == 1, "one 32-row block per wave");
    constexpr int XCK = RBK / 16, XRL = 1024 / RBK, XNL = 32 / XRL;
    __syncthreads();  // every wave is done with the tile buffers
    const uint32_t xk = lds0 + wave * (2 * 32 * RBK), xv = xk + 32 * RBK;
    const int64_t kv_bytes = (int64_t)(p.n_extra + 1) * p.T * RBK;
    const u32x4 xkres = make_rsrc(Kh, (uint32_t)kv_bytes);
    const u32x4 xvres = make_rsrc(Vh, (uint32_t)kv_bytes);
    int goff[XNL];
#pragma unroll
    for (int n = 0; n < XNL; ++n) {
      const int r = n * XRL + lane / XCK;
      goff[n] = r * RBK + (((lane % XCK) ^ (r & (XCK - 1))) * 16);
    }
    const int row0 = __builtin_amdgcn_readfirstlane(m0 + wave * BMW);
    auto issue_x = [&](const u32x4& res, uint32_t dst, int j) __attribute__((always_inline)) {
      const int soff = __builtin_amdgcn_readfirstlane((j * p.T + row0) * RBK);
#pragma unroll
      for (int n = 0; n < XNL; ++n) load_to_lds16<0>(res, dst + n * 1024, goff[n], soff);
    };
    const uint8_t* const xkp = dq_smem + wave * (2 * 32 * RBK);
    const uint8_t* const xvp = xkp + 32 * RBK;
    const int xrow = col * RBK, xsw = col & (XCK - 1);
    for (int j = 1; j <= p.n_extra; ++j) {
      issue_x(xkres, xk, j);
      issue_x(xvres, xv, j);
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      float dot = 0.f, dpv = 0.f;
#pragma unroll
      for (int kk = 0; kk < NKK; ++kk) {
        const int o = xrow + (((2 * kk + g) ^ xsw) * 16);
        dot = dot8_bf16(qf[0][kk], *reinterpret_cast<const u32x4*>(xkp + o), dot);
        dpv = dot8_bf16(dof[0][kk], *reinterpret_cast<const u32x4*>(xvp + o), dpv);
      }
      dot = half_swap_sum(dot);
      dpv = half_swap_sum(dpv);
      const float pv = fast_exp2(dot - lse_i[0]);  // the query fragments carry the scale
      const float ds = pv * (dpv - delta_i[0]);
#pragma unroll
      for (int db = 0; db < NDB; ++db)
#pragma unroll
        for (int r4 = 0; r4 < 4; ++r4) {
          float kk4[4];
          unpack4(*reinterpret_cast<const u32x2*>(xkp + xrow + (((db * 4 + r4) ^ xsw) * 16) + 8 * g), kk4);
#pragma unroll
          for (int t = 0; t < 4; ++t) acc[0][db][r4 * 4 + t] = fmaf(ds, kk4[t], acc[0][db][r4 * 4 + t]);
        }
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // rows read before the next step overwrites them
    }
  }

#pragma unroll
  for (int sb = 0; sb < NSB; ++sb) {
    if (i[sb] >= p.NQ) continue;
    uint16_t* orow = dQ + (int64_t)h * dq_hs + (int64_t)i[sb] * D + 4 * g;
#pragma unroll
    for (int db = 0; db < NDB; ++db)
#pragma unroll
      for (int r4 = 0; r4 < 4; ++r4) {
        u32x2 w;
        w.x = pack_bf16x2(acc[sb][db][r4 * 4 + 0] * p.scaling, acc[sb][db][r4 * 4 + 1] * p.scaling);
        w.y = pack_bf16x2(acc[sb][db][r4 * 4 + 2] * p.scaling, acc[sb][db][r4 * 4 + 3] * p.scaling);
        *reinterpret_cast<u32x2*>(orow + db * 32 + 8 * r4) = w;
      }
  }
}

}  // namespace spx
#include "attn_dkv.h"
namespace spx {

// dK[kvh, c, :] = scaling * sum of the partial results of the head units of kvh (n_hu / Hkv of them in each of n_sum
// sets), dV likewise (no scaling); bf16 out.  `accumulate`: what dK / dV hold is added (in fp32, one rounding).
struct DkvSum {
  const float *dKp, *dVp;
  int NKV, n_hu, n_sum, Hkv;
  float scaling;
  uint16_t* dK; int64_t dk_hs;
  uint16_t* dV; int64_t dv_hs;
  int accumulate;
};
template <int D>
__device__ __forceinline__ void dkv_sum(const DkvSum& a, int64_t idx) {
  const int64_t per_head = (int64_t)a.NKV * D / 4;  // float4 items
  if (idx >= per_head * a.Hkv) return;
  const int kvh = (int)(idx / per_head);
  const int64_t off = (idx % per_head) * 4;
  const int units = a.n_hu / a.Hkv;
  f32x4 sk = {0, 0, 0, 0}, sv = {0, 0, 0, 0};
  for (int s = 0; s < a.n_sum; ++s)
    for (int u = 0; u < units; ++u) {
      const int64_t base = ((int64_t)(s * a.n_hu + kvh * units + u) * a.NKV) * D + off;
      sk += *reinterpret_cast<const f32x4*>(a.dKp + base);
      sv += *reinterpret_cast<const f32x4*>(a.dVp + base);
    }
  sk *= a.scaling;
  u32x2 wk, wv;
  u32x2* const kp = reinterpret_cast<u32x2*>(a.dK + (int64_t)kvh * a.dk_hs + off);
  u32x2* const vp = reinterpret_cast<u32x2*>(a.dV + (int64_t)kvh * a.dv_hs + off);
  if (a.accumulate) {
    wk = *kp;
    wv = *vp;
    sk.x += bf16_lo(wk.x); sk.y += bf16_hi(wk.x); sk.z += bf16_lo(wk.y); sk.w += bf16_hi(wk.y);
    sv.x += bf16_lo(wv.x); sv.y += bf16_hi(wv.x); sv.z += bf16_lo(wv.y); sv.w += bf16_hi(wv.y);
  }
  wk.x = pack_bf16x2(sk.x, sk.y); wk.y = pack_bf16x2(sk.z, sk.w);
  wv.x = pack_bf16x2(sv.x, sv.y); wv.y = pack_bf16x2(sv.z, sv.w);
  *kp = wk;
  *vp = wv;
}
template <int D>
__global__ __launch_bounds__(256) void attn_dkv_reduce_kernel(DkvSum a) {
  dkv_sum<D>(a, (int64_t)blockIdx.x * 256 + threadIdx.x);
}

// dK / dV of the TTT diagonal keys (j, i), j >= 1: sixteen lanes per (position, K/V head)
// item, four items per wave; each such key is seen by exactly the `group` query heads at its
// own position.  A lane holds D / 16 consecutive elements (one or two 16-byte accesses); the dot
// products are summed over the sixteen lanes with DPP moves (no LDS traffic).  The sums over the
// heads of a group stay in fp32 registers until the one store (one rounding to bf16).
// MAXG = query heads per K/V head whose rows are kept in registers: a group of at most MAXG heads
// reads its query / output-gradient rows once for all diagonals; a wider group walks its heads in
// passes of MAXG inside every diagonal (rows re-read per diagonal, from L2).
// The first sum_blocks workgroups add up the partial results of the other keys (dkv_sum): both are short (5 us each at
// 1024 rows of the 1B shape, 14 + 18 at 3001 of the 8B shape) and share no result, so one launch takes as long as the longer.
template <int D, int MAXG>
__global__ __launch_bounds__(256) void ttt_attn_bwd_diag_kernel(
    const uint16_t* __restrict__ Q, int64_t q_hs, const uint16_t* __restrict__ K, int64_t k_hs,
    const uint16_t* __restrict__ V, int64_t v_hs, const uint16_t* __restrict__ dO,
    const float* __restrict__ LSE, const float* __restrict__ Delta, int T, int n_extra, int Hq,
    int Hkv, float scale_log2e, float scaling, uint16_t* dK, int64_t dk_hs, uint16_t* dV,
    int64_t dv_hs, int accumulate, DkvSum sum, int sum_blocks) {
  if ((int)blockIdx.x < sum_blocks) {
    dkv_sum<D>(sum, (int64_t)blockIdx.x * 256 + threadIdx.x);
    return;
  }
  constexpr int EPL = D / 16;
  // item = kvh * T + i: neighbouring 16-lane rows take neighbouring positions of one K/V head, so
  // their key / value / gradient rows are contiguous in memory.  The tail clamps (no early
  // return: the DPP sums need whole rows of lanes)
  const int64_t n_items = (int64_t)T * Hkv;
  const int64_t raw = (((int64_t)blockIdx.x - sum_blocks) * 4 + (threadIdx.x >> 6)) * 4 + ((threadIdx.x & 63) >> 4);
  const bool live = raw < n_items;
  const int64_t item = live ? raw : n_items - 1;
  const int kvh = (int)(item / T), i = (int)(item % T);
  const int group = Hq / Hkv;
  const int d0 = (threadIdx.x & 15) * EPL;
  const bool one_pass = group <= MAXG;

  float qv[MAXG][EPL], dv[MAXG][EPL], lse_h[MAXG], delta_h[MAXG];
  auto load_heads = [&](int h0, int ng) {
#pragma unroll
    for (int hh = 0; hh < MAXG; ++hh) {
      const int h = kvh * group + h0 + (hh < ng ? hh : 0);
      ld_bf16s<EPL>(Q + (int64_t)h * q_hs + (int64_t)i * D + d0, qv[hh]);
      ld_bf16s<EPL>(dO + ((int64_t)i * Hq + h) * D + d0, dv[hh]);
      lse_h[hh] = LSE[(int64_t)h * T + i];
      delta_h[hh] = Delta[(int64_t)h * T + i];
    }
  };
  if (one_pass) load_heads(0, group);
  // the key / value rows of diagonal j + 1 are requested before diagonal j is worked on: the
  // loop is a chain of dependent global loads otherwise
  float kn[EPL], vn[EPL];
  {
    const int64_t r1 = ((int64_t)T + i) * D + d0;
    ld_bf16s<EPL>(K + (int64_t)kvh * k_hs + r1, kn);
    ld_bf16s<EPL>(V + (int64_t)kvh * v_hs + r1, vn);
  }
  for (int j = 1; j <= n_extra; ++j) {
    const int64_t gko = (int64_t)kvh * dk_hs + ((int64_t)j * T + i) * D + d0;
    const int64_t gvo = (int64_t)kvh * dv_hs + ((int64_t)j * T + i) * D + d0;
    float kv[EPL], vv[EPL], gk[EPL], gv[EPL];
#pragma unroll
    for (int e = 0; e < EPL; ++e) {
      kv[e] = kn[e];
      vv[e] = vn[e];
      gk[e] = 0.f;
      gv[e] = 0.f;
    }
    if (accumulate) {  // what the gradient rows hold is the starting value
      ld_bf16s<EPL>(dK + gko, gk);
      ld_bf16s<EPL>(dV + gvo, gv);
    }
    if (j < n_extra) {
      const int64_t rn = ((int64_t)(j + 1) * T + i) * D + d0;
      ld_bf16s<EPL>(K + (int64_t)kvh * k_hs + rn, kn);
      ld_bf16s<EPL>(V + (int64_t)kvh * v_hs + rn, vn);
    }
    for (int h0 = 0; h0 < group; h0 += MAXG) {
      const int ng = min(group - h0, MAXG);
      if (!one_pass) load_heads(h0, ng);
#pragma unroll
      for (int hh = 0; hh < MAXG; ++hh) {
        if (hh < ng) {
          float dot = 0.f, dpv = 0.f;
#pragma unroll
          for (int e = 0; e < EPL; ++e) {
            dot = fmaf(qv[hh][e], kv[e], dot);
            dpv = fmaf(dv[hh][e], vv[e], dpv);
          }
          dot = row16_sum(dot);
          dpv = row16_sum(dpv);
          const float pv = fast_exp2(fmaf(dot, scale_log2e, -lse_h[hh]));
          const float ds = pv * (dpv - delta_h[hh]) * scaling;
#pragma unroll
          for (int e = 0; e < EPL; ++e) {
            gv[e] = fmaf(pv, dv[hh][e], gv[e]);
            gk[e] = fmaf(ds, qv[hh][e], gk[e]);
          }
        }
      }
    }
    if (live) {
      st_bf16s<EPL>(dK + gko, gk);
      st_bf16s<EPL>(dV + gvo, gv);
    }
  }
}

// ---------------------------------------------------------------- launchers
static int64_t round_up(int64_t a, int64_t b) { return (a + b - 1) / b * b; }

constexpr int kFwdNSB = 1, kFwdNW = 4, kDqNSB = 1, kDqNW = 4;  // 32-row sub-blocks per wave, waves per workgroup

// The split of the dK / dV work with the least estimated time, in steps of 32 query rows (0.8 us).  A workgroup's key
// block costs its steps (on average half the rows of a causal mask, at most all of them) and 17 steps for its start and
// its results.  Pairs of key blocks are equally long, so they run in rounds of `slots` workgroups; single blocks, the
// long ones first, keep the slots busy up to a tail of 0.65 units, or take as long as the longest.  More heads per
// workgroup: fewer starts, and fewer partial results to write and to sum (3.5 TB/s); but no fewer head units than XCDs, or
// workgroups far apart in the sequence share an L2 (16384 rows, 16 heads of 256: 3900 us with one or two heads, 4570 with
// eight).
// Measured (us, kernel + sum): 8192 rows, 64 heads of 128: 2217 with one head and pairs, 1998 with eight heads; 4096, 32
// heads of 128: 306 -> 281 with two heads; 3001: 222 -> 184 with two heads, single; 1024: 63 -> 50 single; 1024, 16 heads
// of 256: 60 -> 48 single.  A workgroup that has all heads of its K/V head (DkvPlan::whole) leaves no partial results: the case
// above 618 + 32 for the sum -> 608, 8192 rows of 64 heads of 128 1976 + 24 -> 1990.  (Cutting the query rows of a block into parts on top of that never paid: the second set of
// partial results costs more than the idle compute units.)
static DkvPlan dkv_plan(int64_t NQ, int64_t NKV, int Hq, int Hkv, int D) {
  const int KB = D == 64 ? DkvCfg<64>::KB : D == 128 ? DkvCfg<128>::KB : DkvCfg<256>::KB, cap = DkvCfg<128>::kListCap;
  const int slots = 256 * (D == 64 ? 2 : 1), group = Hq / Hkv;
  DkvPlan pl;
  pl.n_kb = (int)((NKV + KB - 1) / KB);
  pl.windows = (int)(((NQ + 63) / 64 + cap - 1) / cap);
  pl.heads = 1;
  pl.paired = 0;
  const double avg = ((double)NQ / 32 + 4) / 2, start = 17;
  double best = 1e30;
  for (int h = 1; h <= group && pl.windows == 1; h *= 2) {
    const int n_hu = Hq / h;
    if (group % h || (h > 1 && n_hu % 8)) continue;
    const double sum = h == group ? 0. : (double)n_hu * (double)NKV * D * 8 / 3.5e6 / 0.8;
    const double unit = h * avg + start;
    const double single = std::max(pl.n_kb * n_hu <= slots ? 0. : pl.n_kb * n_hu * unit / slots + 0.65 * unit,
                                   2 * h * avg + start + 12) + sum;
    const double pairs = (double)(((pl.n_kb + 1) / 2 * n_hu + slots - 1) / slots) * 2 * (1.08 * h * avg + start) + sum;
    if (single < best) { best = single; pl.heads = h; pl.paired = 0; }
    if (pairs < best) { best = pairs; pl.heads = h; pl.paired = 1; }
  }
  pl.n_hu = Hq / pl.heads;
  pl.n_k = pl.paired ? (pl.n_kb + 1) / 2 : pl.n_kb * pl.windows;
  return pl;
}

// Forward calls of little work take V^T from transposing reads, larger ones from a copy: the copy pays above about 60 us of
// products at head_dim <= 128 and 1000 us at 256 (at 800 TFLOP/s of a causal mask).  Measured, copy + kernel against
// transposing reads: 512 rows, 32 heads of 64 16.9 / 13.4 us, 2048 of 128 57.7 / 58.3, 4096 of 128 145 / 147; 600 rows of
// 16 heads of 256 26.4 / 24.1, 2000 60.8 / 58.2, 4096 140.2 / 137.9, 8192 489 / 487, 16384 1835 / 1853 (two documents of 16380
// after a second of work, at a lower clock: 3837 / 3860).
static double fwd_us(int64_t NQ, int64_t NKV, int Hq, int D) { return 2. * Hq * (double)NQ * (double)NKV * D / 8e8; }
static bool fwd_tr(int64_t NQ, int64_t NKV, int Hq, int D) { return fwd_us(NQ, NKV, Hq, D) < (D > 128 ? 1000. : 60.); }
static int64_t fwd_workspace_bytes(int64_t NQ, int64_t NKV, int Hq, int Hkv, int D) {
  return fwd_tr(NQ, NKV, Hq, D) ? 256 : round_up((int64_t)Hkv * D * round_up(NKV, 128) * 2, 256);
}
static int64_t bwd_workspace_bytes(int64_t NQ, int64_t NKV, int Hq, int Hkv, int D) {
  const int64_t NQp = round_up(NQ, 128);
  int64_t b = round_up((int64_t)Hq * NQ * 4, 256);                  // delta
  b += round_up(((NQ + 63) / 64) * 32, 256);                        // tile bounds
  b += 2 * round_up((int64_t)dkv_plan(NQ, NKV, Hq, Hkv, D).parts(Hkv) * NKV * D * 4, 256);  // fp32 partial dK, dV
  b += round_up((int64_t)Hq * NQ * D * 2, 256);                     // Q scaled, row-major
  b += round_up(2 * (int64_t)Hq * NQp * 4, 256);                    // -lse, -delta in padded rows
  b += round_up(4 * NQp * 4, 256);                                  // interval ends of every row
  return b;
}

template <int D, bool TR>
static int fwd_lds(const char* fn) {
  static std::atomic<uint64_t> lds_set;  // per instantiation, one bit per device
  return ensure_dynamic_lds(reinterpret_cast<const void*>(&attn_fwd_kernel<D, kFwdNSB, kFwdNW, TR>),
                            FwdSmem<D, kFwdNW>::kBytes, lds_set, fn);
}

template <int D, bool TR>
static int launch_fwd_as(AttnParams p, const uint16_t* vt, uint16_t* O, float* lse, hipStream_t st, const char* fn) {
  constexpr int BM = 32 * kFwdNSB * kFwdNW;
  const int n_qb = (p.NQ + BM - 1) / BM;
  constexpr int smem = FwdSmem<D, kFwdNW>::kBytes;
  if (int rc = fwd_lds<D, TR>(fn)) return rc;
  hipLaunchKernelGGL((attn_fwd_kernel<D, kFwdNSB, kFwdNW, TR>), dim3((unsigned)(n_qb * p.Hq)), dim3(64 * kFwdNW), smem,
                     st, p, vt, O, lse);
  return check_launch(fn);
}

// workspace: room for V^T (fwd_workspace_bytes), or null: transposing reads whatever the size
template <int D>
static int launch_fwd(AttnParams p, void* workspace, uint16_t* O, float* lse, hipStream_t st, const char* fn) {
  if ((int64_t)p.NKVp * D * 2 >= (1ll << 31)) {
    last_error() = std::string(fn) + ": keys of one head must span less than 2 GiB";
    return SPX_ERR_ARG;
  }
  if (!workspace || fwd_tr(p.NQ, p.NKV, p.Hq, D)) return launch_fwd_as<D, true>(p, nullptr, O, lse, st, fn);
  uint16_t* vt = reinterpret_cast<uint16_t*>(workspace);
  dim3 tgrid((unsigned)(p.NKVp / 64), (unsigned)((D + 63) / 64), (unsigned)p.Hkv);
  hipLaunchKernelGGL(transpose_bf16_kernel, tgrid, dim3(64), 0, st, p.V, p.v_hs, (int64_t)D, p.NKV, D,
                     vt, (int64_t)D * p.NKVp, D > 128 ? (int64_t)32 : (int64_t)p.NKVp,
                     D > 128 ? (int64_t)32 * D : (int64_t)32);
  return launch_fwd_as<D, false>(p, vt, O, lse, st, fn);
}

template <int D, bool WHOLE>
static int launch_dkv(const AttnParams& ps, const uint16_t* dOp, const BwdSide& side, const DkvPlan& pl, void* dk, void* dv, int64_t dk_hs,
                      int64_t dv_hs, int accumulate, hipStream_t st, const char* fn) {
  static std::atomic<uint64_t> lds_set;  // per instantiation, one bit per device
  if (int rc = ensure_dynamic_lds(reinterpret_cast<const void*>(&attn_bwd_dkv_kernel<D, WHOLE>), DkvCfg<D>::kBytes, lds_set, fn))
    return rc;
  hipLaunchKernelGGL((attn_bwd_dkv_kernel<D, WHOLE>), dim3((unsigned)(pl.n_k * pl.n_hu)), dim3(512), DkvCfg<D>::kBytes, st, ps, dOp,
                     side.NQp, side.neg, side.rows, side.tb, pl, reinterpret_cast<float*>(dk), reinterpret_cast<float*>(dv), dk_hs,
                     dv_hs, accumulate);
  return SPX_OK;
}

template <int D>
static int launch_bwd(AttnParams p, const uint16_t* Op, const uint16_t* dOp, const float* lse,
                      uint16_t* dQp, int64_t dq_hs, uint16_t* dKp, int64_t dk_hs, uint16_t* dVp,
                      int64_t dv_hs, void* workspace, hipStream_t st, const char* fn, int accumulate = 0) {
  const int NQp = (int)round_up(p.NQ, 128);
  DkvPlan pl = dkv_plan(p.NQ, p.NKV, p.Hq, p.Hkv, D);
  // Rows that see a context and a block of their own: pairs of key blocks are not equally long then.  Single blocks took 0.91 of the
  // time over 105 calls of 1248 to 8192 rows, in one to six documents and under a window, 1.09 at the most (8192 + 8192 keys, 8192 rows
  // of 32 heads of 128 under a window of 2048 568 -> 543 us, 2048 + 4096 in six documents 174 -> 111).  Where the pairs of few rows fit
  // in one round, the starts of a second one weigh more: 512 to 1248 rows 1.05 over 33 calls (1024 + 1024 keys, 32 heads of 128
  // 55 -> 69 us, 64 heads 86 -> 105), but 1488 and 1776 rows 0.93; at head_dim 256 512 to 1024 rows 1.01, 1248 0.89.
  if (p.a2 && pl.paired && (pl.n_k * pl.n_hu > 256 * (D == 64 ? 2 : 1) || p.NQ > (D > 128 ? 1024 : 1280))) {
    pl.paired = 0;
    pl.n_k = pl.n_kb;
  }
  char* w = reinterpret_cast<char*>(workspace);
  float* delta = reinterpret_cast<float*>(w);
  w += round_up((int64_t)p.Hq * p.NQ * 4, 256);
  int32_t* tb = reinterpret_cast<int32_t*>(w);
  w += round_up(((p.NQ + 63) / 64) * 32, 256);
  float* dkp = reinterpret_cast<float*>(w);
  w += round_up((int64_t)pl.parts(p.Hkv) * p.NKV * D * 4, 256);
  float* dvp = reinterpret_cast<float*>(w);
  w += round_up((int64_t)pl.parts(p.Hkv) * p.NKV * D * 4, 256);
  uint16_t* qs = reinterpret_cast<uint16_t*>(w);  // bf16(q * scale * log2 e), [Hq][NQ][D]
  w += round_up((int64_t)p.Hq * p.NQ * D * 2, 256);
  float* neg = reinterpret_cast<float*>(w);       // -lse [Hq][NQp], -delta [Hq][NQp]
  w += round_up(2 * (int64_t)p.Hq * NQp * 4, 256);
  int32_t* mrows = reinterpret_cast<int32_t*>(w); // [4][NQp]

  // (one list of query tiles in LDS; more rows than that are cut into windows at head_dim 256 only)
  if (D <= 128 && (p.NQ + 63) / 64 > DkvCfg<D>::kListCap) {
    last_error() = std::string(fn) + ": more than " + std::to_string(64 * DkvCfg<D>::kListCap) +
                   " query rows in one call at head_dim <= 128";
    return SPX_ERR_ARG;
  }
  // the dK/dV and diagonal-key kernels read the scaled queries: their scores are q' . k with no
  // factor of their own, and what they accumulate against q' carries scale * log2(e) once too
  // often: dK = ln 2 * sum dS q'
  AttnParams ps = p;
  ps.Q = qs;
  ps.q_hs = (int64_t)p.NQ * D;
  // (byte offsets of dO's rows are 32 bits, without a sign; the rows that fill the last tile count)
  if (D > 128 ? (int64_t)p.NQ * p.Hq * D * 2 >= (1ll << 31) : ((int64_t)p.NQ + 64) * p.Hq * D * 2 >= (1ll << 32)) {
    last_error() = std::string(fn) + ": queries must span less than " + (D > 128 ? "2" : "4") + " GiB";
    return SPX_ERR_ARG;
  }
  const BwdSide side = {NQp, qs, delta, neg, tb, mrows};

  constexpr int BM = 32 * kDqNSB * kDqNW;
  static_assert(BM == 128, "the rows of BwdSide are rounded up to a workgroup's");
  const int n_qb = (p.NQ + BM - 1) / BM;
  {
    constexpr int dq_smem = DqSmem<D, kDqNW>::kBytes;
    if ((int64_t)p.NKVp * D * 2 >= (1ll << 31)) {
      last_error() = std::string(fn) + ": keys of one head must span less than 2 GiB";
      return SPX_ERR_ARG;
    }
    static std::atomic<uint64_t> dq_lds_set;  // per head_dim instantiation, one bit per device
    if (int rc = ensure_dynamic_lds(reinterpret_cast<const void*>(&attn_bwd_dq_kernel<D, kDqNSB, kDqNW>), dq_smem,
                                    dq_lds_set, fn))
      return rc;
    hipLaunchKernelGGL((attn_bwd_dq_kernel<D, kDqNSB, kDqNW>), dim3((unsigned)(n_qb * p.Hq)), dim3(64 * kDqNW), dq_smem,
                       st, p, Op, dOp, lse, side, dQp, dq_hs);
  }

  const bool whole = pl.whole(p.Hkv);
  if (int rc = whole ? launch_dkv<D, true>(ps, dOp, side, pl, dKp, dVp, dk_hs, dv_hs, accumulate, st, fn)
                     : launch_dkv<D, false>(ps, dOp, side, pl, dkp, dvp, 0, 0, 0, st, fn))
    return rc;
  const int sum_blocks = whole ? 0 : (int)(((int64_t)p.NKV * D / 4 * p.Hkv + 255) / 256);
  const DkvSum sum = {dkp, dvp, p.NKV, pl.n_hu, pl.windows, p.Hkv, kLn2, dKp, dk_hs, dVp, dv_hs, accumulate};
  if (p.n_extra == 0) {
    if (!whole) hipLaunchKernelGGL(attn_dkv_reduce_kernel<D>, dim3((unsigned)sum_blocks), dim3(256), 0, st, sum);
  } else {
    const dim3 dgrid((unsigned)(sum_blocks + ((int64_t)p.T * p.Hkv + 15) / 16));
    // eight heads per K/V head in registers where they fit (head_dim <= 128), else four
    if (D <= 128 && p.Hq / p.Hkv > 4)
      hipLaunchKernelGGL((ttt_attn_bwd_diag_kernel<D, (D <= 128 ? 8 : 4)>), dgrid, dim3(256), 0, st, ps.Q,
                         ps.q_hs, p.K, p.k_hs, p.V, p.v_hs, dOp, lse, delta, p.T, p.n_extra, p.Hq, p.Hkv,
                         1.f, kLn2, dKp, dk_hs, dVp, dv_hs, accumulate, sum, sum_blocks);
    else
      hipLaunchKernelGGL((ttt_attn_bwd_diag_kernel<D, 4>), dgrid, dim3(256), 0, st, ps.Q, ps.q_hs, p.K,
                         p.k_hs, p.V, p.v_hs, dOp, lse, delta, p.T, p.n_extra, p.Hq, p.Hkv,
                         1.f, kLn2, dKp, dk_hs, dVp, dv_hs, accumulate, sum, sum_blocks);
  }
  return check_launch(fn);
}

static int shape_checks(const char* fn, int64_t NQ, int64_t NKV, int32_t Hq, int32_t Hkv, int32_t D) {
  if (!(NQ > 0 && NQ < (1ll << 24) && NKV > 0 && NKV < (1ll << 26))) return fail_arg(fn, "sequence length out of range");
  if (!(Hkv > 0 && Hq > 0 && Hq % Hkv == 0)) return fail_arg(fn, "Hq must be a multiple of Hkv");
  if (!(D == 64 || D == 128 || D == 256)) return fail_arg(fn, "head_dim must be 64, 128 or 256");
  return SPX_OK;
}

static bool all_aligned16(std::initializer_list<const void*> ps) {
  for (const void* q : ps)
    if (reinterpret_cast<uintptr_t>(q) & 15) return false;
  return true;
}

}  // namespace spx

using namespace spx;

// ================================================================ TTT entry points
extern "C" int spx_ttt_row_lo(const void* document_ids, int doc_kind, int64_t T,
                              int64_t sliding_window, int32_t* row_lo, void* stream) {
  SPX_REQUIRE(doc_kind == SPX_KIND_I32 || doc_kind == SPX_KIND_I64, "document_ids must be int32 or int64");
  SPX_REQUIRE(T > 0 && T < (1ll << 30), "0 < T < 2^30");
  SPX_REQUIRE(document_ids && row_lo, "null buffer");
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  if (doc_kind == SPX_KIND_I32)
    hipLaunchKernelGGL(ttt_row_lo_kernel<int32_t>, dim3(1), dim3(1024), 0, st,
                       reinterpret_cast<const int32_t*>(document_ids), T, sliding_window, row_lo);
  else
    hipLaunchKernelGGL(ttt_row_lo_kernel<int64_t>, dim3(1), dim3(1024), 0, st,
                       reinterpret_cast<const int64_t*>(document_ids), T, sliding_window, row_lo);
  return check_launch(__func__);
}

extern "C" int64_t spx_ttt_attn_workspace_bytes(int64_t T, int32_t Hq, int32_t Hkv, int32_t D,
                                                int32_t backward) {
  return backward ? bwd_workspace_bytes(T, T, Hq, Hkv, D) : fwd_workspace_bytes(T, T, Hq, Hkv, D);
}

static AttnParams ttt_params(const void* q, int64_t q_hs, const void* k, int64_t k_hs, const void* v,
                             int64_t v_hs, const int32_t* row_lo, int64_t T, int32_t ttt_step,
                             int32_t Hq, int32_t Hkv, float scaling) {
  AttnParams p;
  p.Q = reinterpret_cast<const uint16_t*>(q); p.q_hs = q_hs;
  p.K = reinterpret_cast<const uint16_t*>(k); p.k_hs = k_hs;
  p.V = reinterpret_cast<const uint16_t*>(v); p.v_hs = v_hs;
  p.a1 = row_lo; p.b1 = nullptr; p.a2 = nullptr; p.b2 = nullptr;
  p.NQ = (int)T; p.T = (int)T; p.NKV = (int)T; p.NKVp = (int)round_up(T, 128);
  p.n_extra = ttt_step; p.Hq = Hq; p.Hkv = Hkv;
  p.scaling = scaling; p.scale_log2e = scaling * kLog2e;
  return p;
}

// workspace: room for V^T, or null: transposing reads whatever the size (spx_ttt_attn_fwd_static)
static int ttt_attn_fwd_impl(const char* fname, const void* q, int64_t q_head_stride, const void* k,
                             int64_t k_head_stride, const void* v, int64_t v_head_stride, const int32_t* row_lo,
                             int64_t T, int32_t ttt_step, int32_t Hq, int32_t Hkv, int32_t D, float scaling, void* out,
                             float* lse, void* workspace, void* stream) {
  if (!(ttt_step >= 0 && ttt_step < 64)) return fail_arg(fname, "0 <= ttt_step < 64");
  if (!(q && k && v && row_lo && out && lse)) return fail_arg(fname, "null buffer");
  if (q_head_stride < T * D) return fail_arg(fname, "q head stride smaller than T*D");
  if (k_head_stride < (int64_t)(ttt_step + 1) * T * D || v_head_stride < (int64_t)(ttt_step + 1) * T * D)
    return fail_arg(fname, "k/v head stride smaller than (ttt_step+1)*T*D");
  if (q_head_stride % 8 || k_head_stride % 8 || v_head_stride % 8)
    return fail_arg(fname, "head strides must be multiples of 8 elements");
  if (!all_aligned16({q, k, v, out, workspace})) return fail_arg(fname, "buffers must be 16-byte aligned");
  AttnParams p = ttt_params(q, q_head_stride, k, k_head_stride, v, v_head_stride, row_lo, T, ttt_step,
                            Hq, Hkv, scaling);
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  if (D == 256) return launch_fwd<256>(p, workspace, reinterpret_cast<uint16_t*>(out), lse, st, fname);
  if (D == 128) return launch_fwd<128>(p, workspace, reinterpret_cast<uint16_t*>(out), lse, st, fname);
  return launch_fwd<64>(p, workspace, reinterpret_cast<uint16_t*>(out), lse, st, fname);
}

extern "C" int spx_ttt_attn_fwd(const void* q, int64_t q_head_stride, const void* k,
                                int64_t k_head_stride, const void* v, int64_t v_head_stride,
                                const int32_t* row_lo, int64_t T, int32_t ttt_step, int32_t Hq,
                                int32_t Hkv, int32_t D, float scaling, void* out, float* lse,
                                void* workspace, int64_t workspace_bytes, void* stream) {
  if (int rc = shape_checks(__func__, T, T, Hq, Hkv, D)) return rc;
  SPX_REQUIRE(workspace, "null buffer");
  SPX_REQUIRE(workspace_bytes >= fwd_workspace_bytes(T, T, Hq, Hkv, D), "workspace too small");
  return ttt_attn_fwd_impl(__func__, q, q_head_stride, k, k_head_stride, v, v_head_stride, row_lo, T, ttt_step, Hq,
                           Hkv, D, scaling, out, lse, workspace, stream);
}

#define SPX_REQ_FN(cond, what) do { if (!(cond)) return spx::fail_arg(fname, what); } while (0)
static int ttt_attn_bwd_impl(const char* fname, int accumulate, const void* q, int64_t q_head_stride,
                             const void* k, int64_t k_head_stride, const void* v, int64_t v_head_stride,
                             const void* out, const void* dout, const float* lse, const int32_t* row_lo,
                             int64_t T, int32_t ttt_step, int32_t Hq, int32_t Hkv, int32_t D, float scaling,
                             void* dq, int64_t dq_head_stride, void* dk, int64_t dk_head_stride, void* dv,
                             int64_t dv_head_stride, void* workspace, int64_t workspace_bytes,
                             void* stream) {
  if (int rc = shape_checks(fname, T, T, Hq, Hkv, D)) return rc;
  SPX_REQ_FN(ttt_step >= 0 && ttt_step < 64, "0 <= ttt_step < 64");
  SPX_REQ_FN(q && k && v && out && dout && lse && row_lo && dq && dk && dv && workspace, "null buffer");
  const int64_t kv_rows = (int64_t)(ttt_step + 1) * T * D;
  SPX_REQ_FN(q_head_stride >= T * D && dq_head_stride >= T * D, "q / dq head stride smaller than T*D");
  SPX_REQ_FN(k_head_stride >= kv_rows && v_head_stride >= kv_rows && dk_head_stride >= kv_rows &&
              dv_head_stride >= kv_rows, "k/v/dk/dv head stride smaller than (ttt_step+1)*T*D");
  SPX_REQ_FN((q_head_stride | k_head_stride | v_head_stride | dq_head_stride | dk_head_stride |
               dv_head_stride) % 8 == 0, "head strides must be multiples of 8 elements");
  SPX_REQ_FN(workspace_bytes >= bwd_workspace_bytes(T, T, Hq, Hkv, D), "workspace too small");
  SPX_REQ_FN(all_aligned16({q, k, v, out, dout, dq, dk, dv, workspace}), "buffers must be 16-byte aligned");
  AttnParams p = ttt_params(q, q_head_stride, k, k_head_stride, v, v_head_stride, row_lo, T, ttt_step,
                            Hq, Hkv, scaling);
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  auto Op = reinterpret_cast<const uint16_t*>(out);
  auto dOp = reinterpret_cast<const uint16_t*>(dout);
  auto dQp = reinterpret_cast<uint16_t*>(dq);
  auto dKp = reinterpret_cast<uint16_t*>(dk);
  auto dVp = reinterpret_cast<uint16_t*>(dv);
  if (D == 256)
    return launch_bwd<256>(p, Op, dOp, lse, dQp, dq_head_stride, dKp, dk_head_stride, dVp, dv_head_stride,
                           workspace, st, fname, accumulate);
  if (D == 128)
    return launch_bwd<128>(p, Op, dOp, lse, dQp, dq_head_stride, dKp, dk_head_stride, dVp,
                           dv_head_stride, workspace, st, fname, accumulate);
  return launch_bwd<64>(p, Op, dOp, lse, dQp, dq_head_stride, dKp, dk_head_stride, dVp, dv_head_stride,
                        workspace, st, fname, accumulate);
}

extern "C" int spx_ttt_attn_bwd(const void* q, int64_t q_head_stride, const void* k,
                                int64_t k_head_stride, const void* v, int64_t v_head_stride,
                                const void* out, const void* dout, const float* lse,
                                const int32_t* row_lo, int64_t T, int32_t ttt_step, int32_t Hq,
                                int32_t Hkv, int32_t D, float scaling, void* dq,
                                int64_t dq_head_stride, void* dk, int64_t dk_head_stride, void* dv,
                                int64_t dv_head_stride, void* workspace, int64_t workspace_bytes,
                                void* stream) {
  return ttt_attn_bwd_impl(__func__, 0, q, q_head_stride, k, k_head_stride, v, v_head_stride, out, dout, lse,
                           row_lo, T, ttt_step, Hq, Hkv, D, scaling, dq, dq_head_stride, dk, dk_head_stride,
                           dv, dv_head_stride, workspace, workspace_bytes, stream);
}

extern "C" int spx_ttt_attn_bwd_accumulate(const void* q, int64_t q_head_stride, const void* k,
                                           int64_t k_head_stride, const void* v, int64_t v_head_stride,
                                           const void* out, const void* dout, const float* lse,
                                           const int32_t* row_lo, int64_t T, int32_t ttt_step, int32_t Hq,
                                           int32_t Hkv, int32_t D, float scaling, void* dq,
                                           int64_t dq_head_stride, void* dk, int64_t dk_head_stride,
                                           void* dv, int64_t dv_head_stride, void* workspace,
                                           int64_t workspace_bytes, void* stream) {
  return ttt_attn_bwd_impl(__func__, 1, q, q_head_stride, k, k_head_stride, v, v_head_stride, out, dout, lse,
                           row_lo, T, ttt_step, Hq, Hkv, D, scaling, dq, dq_head_stride, dk, dk_head_stride,
                           dv, dv_head_stride, workspace, workspace_bytes, stream);
}

// ================================================================ span attention
// Per query an interval [row_lo, row_hi) of visible keys out of T (no diagonal keys): the mask of a
// padded batch row, where a query sees the non-padding keys up to itself.
static AttnParams span_params(const void* q, int64_t q_hs, const void* k, int64_t k_hs, const void* v,
                              int64_t v_hs, const int32_t* row_lo, const int32_t* row_hi, int64_t T,
                              int32_t Hq, int32_t Hkv, float scaling) {
  AttnParams p = ttt_params(q, q_hs, k, k_hs, v, v_hs, row_lo, T, 0, Hq, Hkv, scaling);
  p.b1 = row_hi;
  return p;
}

extern "C" int spx_span_attn_fwd(const void* q, int64_t q_head_stride, const void* k,
                                 int64_t k_head_stride, const void* v, int64_t v_head_stride,
                                 const int32_t* row_lo, const int32_t* row_hi, int64_t T, int32_t Hq,
                                 int32_t Hkv, int32_t D, float scaling, void* out, float* lse,
                                 void* workspace, int64_t workspace_bytes, void* stream) {
  if (int rc = shape_checks(__func__, T, T, Hq, Hkv, D)) return rc;
  SPX_REQUIRE(q && k && v && row_lo && row_hi && out && lse && workspace, "null buffer");
  SPX_REQUIRE(q_head_stride >= T * D && k_head_stride >= T * D && v_head_stride >= T * D,
              "head stride smaller than T*D");
  SPX_REQUIRE(q_head_stride % 8 == 0 && k_head_stride % 8 == 0 && v_head_stride % 8 == 0,
              "head strides must be multiples of 8 elements");
  SPX_REQUIRE(workspace_bytes >= fwd_workspace_bytes(T, T, Hq, Hkv, D), "workspace too small");
  SPX_REQUIRE(all_aligned16({q, k, v, out, workspace}), "buffers must be 16-byte aligned");
  AttnParams p = span_params(q, q_head_stride, k, k_head_stride, v, v_head_stride, row_lo, row_hi, T, Hq,
                             Hkv, scaling);
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  if (D == 256) return launch_fwd<256>(p, workspace, reinterpret_cast<uint16_t*>(out), lse, st, __func__);
  if (D == 128) return launch_fwd<128>(p, workspace, reinterpret_cast<uint16_t*>(out), lse, st, __func__);
  return launch_fwd<64>(p, workspace, reinterpret_cast<uint16_t*>(out), lse, st, __func__);
}

extern "C" int spx_span_attn_bwd(const void* q, int64_t q_head_stride, const void* k,
                                 int64_t k_head_stride, const void* v, int64_t v_head_stride,
                                 const void* out, const void* dout, const float* lse,
                                 const int32_t* row_lo, const int32_t* row_hi, int64_t T, int32_t Hq,
                                 int32_t Hkv, int32_t D, float scaling, void* dq,
                                 int64_t dq_head_stride, void* dk, int64_t dk_head_stride, void* dv,
                                 int64_t dv_head_stride, void* workspace, int64_t workspace_bytes,
                                 void* stream) {
  if (int rc = shape_checks(__func__, T, T, Hq, Hkv, D)) return rc;
  SPX_REQUIRE(q && k && v && out && dout && lse && row_lo && row_hi && dq && dk && dv && workspace,
              "null buffer");
  SPX_REQUIRE(q_head_stride >= T * D && dq_head_stride >= T * D && k_head_stride >= T * D &&
              v_head_stride >= T * D && dk_head_stride >= T * D && dv_head_stride >= T * D,
              "head stride smaller than T*D");
  SPX_REQUIRE((q_head_stride | k_head_stride | v_head_stride | dq_head_stride | dk_head_stride |
               dv_head_stride) % 8 == 0, "head strides must be multiples of 8 elements");
  SPX_REQUIRE(workspace_bytes >= bwd_workspace_bytes(T, T, Hq, Hkv, D), "workspace too small");
  SPX_REQUIRE(all_aligned16({q, k, v, out, dout, dq, dk, dv, workspace}), "buffers must be 16-byte aligned");
  AttnParams p = span_params(q, q_head_stride, k, k_head_stride, v, v_head_stride, row_lo, row_hi, T, Hq,
                             Hkv, scaling);
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  auto Op = reinterpret_cast<const uint16_t*>(out);
  auto dOp = reinterpret_cast<const uint16_t*>(dout);
  auto dQp = reinterpret_cast<uint16_t*>(dq);
  auto dKp = reinterpret_cast<uint16_t*>(dk);
  auto dVp = reinterpret_cast<uint16_t*>(dv);
  if (D == 256)
    return launch_bwd<256>(p, Op, dOp, lse, dQp, dq_head_stride, dKp, dk_head_stride, dVp, dv_head_stride,
                           workspace, st, __func__);
  if (D == 128)
    return launch_bwd<128>(p, Op, dOp, lse, dQp, dq_head_stride, dKp, dk_head_stride, dVp,
                           dv_head_stride, workspace, st, __func__);
  return launch_bwd<64>(p, Op, dOp, lse, dQp, dq_head_stride, dKp, dk_head_stride, dVp, dv_head_stride,
                        workspace, st, __func__);
}

// ---------------------------------------------------------------- allocation-free variant
// V^T of a large call lies in a device array of the library.  Transposing reads throughout need no array and take 3 - 5 %
// longer: 8192 rows, 64 / 8 heads of 128 1003 us, from the copy 957.  The array serves one call at a time: a call waits, on
// the device, for the event behind the last one's kernels, whichever stream and host thread that came from.  A call under
// capture takes transposing reads: nothing would order its replays.  The wait and the record cost 3 us, so the copy begins
// later here than in fwd_tr, at 120 us of products (4096 rows, 32 heads of 128: 140.4 us without the array, 140.3 with it).
constexpr int64_t kStaticScratchBytes = 16ll << 20;
constexpr double kStaticCopyUs = 120.;
static __device__ __align__(256) unsigned char static_scratch[kStaticScratchBytes];

constexpr int kMaxDevices = 64;
struct StaticScratch {
  std::mutex mu;
  void* base = nullptr;       // this device's array (its name is no host pointer)
  hipEvent_t idle = nullptr;  // behind the kernels of its last user
};
static StaticScratch g_static[kMaxDevices];

static int hip_failed(const char* fn, const char* what, hipError_t e) {
  last_error() = std::string(fn) + ": " + what + ": " + hipGetErrorString(e);
  return SPX_ERR_HIP;
}

// launch(base of the array, or null: transposing reads) on the stream
template <typename F>
static int with_static_scratch(const char* fn, bool copies, hipStream_t st, F launch) {
  hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
  if (copies && hipStreamIsCapturing(st, &capture) != hipSuccess) {
    (void)hipGetLastError();  // (the legacy stream while another one is captured)
    copies = false;
  }
  if (!copies || capture != hipStreamCaptureStatusNone) return launch(nullptr);
  int dev = -1;
  if (hipError_t e = hipGetDevice(&dev)) return hip_failed(fn, "hipGetDevice", e);
  if (dev < 0 || dev >= kMaxDevices) return launch(nullptr);
  StaticScratch& s = g_static[dev];
  std::lock_guard<std::mutex> lock(s.mu);
  if (!s.base)
    if (hipError_t e = hipGetSymbolAddress(&s.base, HIP_SYMBOL(static_scratch))) return hip_failed(fn, "hipGetSymbolAddress", e);
  if (!s.idle) {
    if (hipError_t e = hipEventCreateWithFlags(&s.idle, hipEventDisableTiming)) return hip_failed(fn, "hipEventCreate", e);
  } else if (hipError_t e = hipStreamWaitEvent(st, s.idle, 0)) {
    return hip_failed(fn, "hipStreamWaitEvent", e);
  }
  const int rc = launch(s.base);
  if (hipError_t e = hipEventRecord(s.idle, st)) return hip_failed(fn, "hipEventRecord", e);
  return rc;
}

extern "C" int64_t spx_ttt_attn_fwd_static_max_bytes(void) { return kStaticScratchBytes; }

extern "C" int spx_ttt_attn_fwd_static(const void* q, int64_t q_head_stride, const void* k,
                                       int64_t k_head_stride, const void* v, int64_t v_head_stride,
                                       const int32_t* row_lo, int64_t T, int32_t ttt_step,
                                       int32_t Hq, int32_t Hkv, int32_t D, float scaling, void* out,
                                       float* lse, void* stream) {
  const char* const fname = __func__;
  if (int rc = shape_checks(fname, T, T, Hq, Hkv, D)) return rc;
  if ((int64_t)Hkv * D * round_up(T, 128) * 2 > kStaticScratchBytes)
    return fail_arg(fname, "Hkv * D * round_up(T, 128) * 2 bytes exceed 16 MiB, the limit of this entry point; "
                           "use spx_ttt_attn_fwd with a caller-owned workspace");
  const bool copies = !fwd_tr(T, T, Hq, D) && fwd_us(T, T, Hq, D) >= kStaticCopyUs;
  return with_static_scratch(fname, copies, reinterpret_cast<hipStream_t>(stream), [&](void* workspace) {
    if (int rc = ttt_attn_fwd_impl(fname, q, q_head_stride, k, k_head_stride, v, v_head_stride, row_lo, T, ttt_step, Hq, Hkv,
                                   D, scaling, out, lse, workspace, stream))
      return rc;
    // the form that captured calls take is set up by the first call too, which is made outside capture
    return D == 256 ? fwd_lds<256, true>(fname) : D == 128 ? fwd_lds<128, true>(fname) : fwd_lds<64, true>(fname);
  });
}

// ================================================================ DFlash entry points
extern "C" int spx_dflash_row_ranges(const void* document_ids, int doc_kind, int64_t T,
                                     const void* anchors, int anchor_kind, int64_t n_anchors,
                                     int32_t block_size, int64_t sliding_window, int32_t causal_block,
                                     int32_t* ctx_lo, int32_t* ctx_hi, int32_t* blk_lo, int32_t* blk_hi,
                                     int32_t* run_start_scratch, void* stream) {
  SPX_REQUIRE(doc_kind == SPX_KIND_I32 || doc_kind == SPX_KIND_I64, "document_ids must be int32 or int64");
  SPX_REQUIRE(anchor_kind == SPX_KIND_I32 || anchor_kind == SPX_KIND_I64, "anchors must be int32 or int64");
  SPX_REQUIRE(T > 0 && T < (1ll << 30) && n_anchors > 0 && block_size > 0, "bad sizes");
  SPX_REQUIRE(n_anchors * block_size < (1ll << 24), "too many block rows");
  SPX_REQUIRE(document_ids && anchors && ctx_lo && ctx_hi && blk_lo && blk_hi && run_start_scratch, "null buffer");
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  const unsigned grid = (unsigned)((n_anchors * block_size + 255) / 256);
#define SPX_RANGES(I, J)                                                                          \
  do {                                                                                            \
    hipLaunchKernelGGL(doc_run_start_kernel<I>, dim3(1), dim3(1024), 0, st,                       \
                       reinterpret_cast<const I*>(document_ids), T, run_start_scratch);           \
    hipLaunchKernelGGL((dflash_ranges_kernel<I, J>), dim3(grid), dim3(256), 0, st,                \
                       reinterpret_cast<const I*>(document_ids), run_start_scratch,               \
                       reinterpret_cast<const J*>(anchors), n_anchors, (int)block_size,           \
                       sliding_window, (int)causal_block, T, ctx_lo, ctx_hi, blk_lo, blk_hi);     \
  } while (0)
  if (doc_kind == SPX_KIND_I32 && anchor_kind == SPX_KIND_I32) SPX_RANGES(int32_t, int32_t);
  else if (doc_kind == SPX_KIND_I32) SPX_RANGES(int32_t, int64_t);
  else if (anchor_kind == SPX_KIND_I32) SPX_RANGES(int64_t, int32_t);
  else SPX_RANGES(int64_t, int64_t);
#undef SPX_RANGES
  return check_launch(__func__);
}

extern "C" int64_t spx_dflash_attn_workspace_bytes(int64_t T, int64_t NQ, int32_t Hq, int32_t Hkv,
                                                   int32_t D, int32_t backward) {
  return backward ? bwd_workspace_bytes(NQ, T + NQ, Hq, Hkv, D) : fwd_workspace_bytes(NQ, T + NQ, Hq, Hkv, D);
}

static AttnParams dflash_params(const void* q, int64_t q_hs, const void* k, int64_t k_hs, const void* v,
                                int64_t v_hs, const int32_t* a1, const int32_t* b1, const int32_t* a2,
                                const int32_t* b2, int64_t T, int64_t NQ, int32_t Hq, int32_t Hkv,
                                float scaling) {
  AttnParams p;
  p.Q = reinterpret_cast<const uint16_t*>(q); p.q_hs = q_hs;
  p.K = reinterpret_cast<const uint16_t*>(k); p.k_hs = k_hs;
  p.V = reinterpret_cast<const uint16_t*>(v); p.v_hs = v_hs;
  p.a1 = a1; p.b1 = b1; p.a2 = a2; p.b2 = b2;
  p.NQ = (int)NQ; p.T = (int)T; p.NKV = (int)(T + NQ); p.NKVp = (int)round_up(T + NQ, 128);
  p.n_extra = 0; p.Hq = Hq; p.Hkv = Hkv;
  p.scaling = scaling; p.scale_log2e = scaling * kLog2e;
  return p;
}

extern "C" int spx_dflash_attn_fwd(const void* q, int64_t q_head_stride, const void* k,
                                   int64_t k_head_stride, const void* v, int64_t v_head_stride,
                                   const int32_t* ctx_lo, const int32_t* ctx_hi, const int32_t* blk_lo,
                                   const int32_t* blk_hi, int64_t T, int64_t NQ, int32_t Hq, int32_t Hkv,
                                   int32_t D, float scaling, void* out, float* lse, void* workspace,
                                   int64_t workspace_bytes, void* stream) {
  if (int rc = shape_checks(__func__, NQ, T + NQ, Hq, Hkv, D)) return rc;
  SPX_REQUIRE(T > 0, "T must be positive");
  SPX_REQUIRE(q && k && v && ctx_lo && ctx_hi && blk_lo && blk_hi && out && lse && workspace, "null buffer");
  SPX_REQUIRE(q_head_stride >= NQ * D, "q head stride smaller than NQ*D");
  SPX_REQUIRE(k_head_stride >= (T + NQ) * D && v_head_stride >= (T + NQ) * D,
              "k/v head stride smaller than (T+NQ)*D");
  SPX_REQUIRE(q_head_stride % 8 == 0 && k_head_stride % 8 == 0 && v_head_stride % 8 == 0,
              "head strides must be multiples of 8 elements");
  SPX_REQUIRE(workspace_bytes >= fwd_workspace_bytes(NQ, T + NQ, Hq, Hkv, D), "workspace too small");
  SPX_REQUIRE(all_aligned16({q, k, v, out, workspace}), "buffers must be 16-byte aligned");
  AttnParams p = dflash_params(q, q_head_stride, k, k_head_stride, v, v_head_stride, ctx_lo, ctx_hi,
                               blk_lo, blk_hi, T, NQ, Hq, Hkv, scaling);
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  if (D == 256) return launch_fwd<256>(p, workspace, reinterpret_cast<uint16_t*>(out), lse, st, __func__);
  if (D == 128) return launch_fwd<128>(p, workspace, reinterpret_cast<uint16_t*>(out), lse, st, __func__);
  return launch_fwd<64>(p, workspace, reinterpret_cast<uint16_t*>(out), lse, st, __func__);
}

extern "C" int spx_dflash_attn_bwd(const void* q, int64_t q_head_stride, const void* k,
                                   int64_t k_head_stride, const void* v, int64_t v_head_stride,
                                   const void* out, const void* dout, const float* lse,
                                   const int32_t* ctx_lo, const int32_t* ctx_hi, const int32_t* blk_lo,
                                   const int32_t* blk_hi, int64_t T, int64_t NQ, int32_t Hq, int32_t Hkv,
                                   int32_t D, float scaling, void* dq, int64_t dq_head_stride, void* dk,
                                   int64_t dk_head_stride, void* dv, int64_t dv_head_stride,
                                   void* workspace, int64_t workspace_bytes, void* stream) {
  if (int rc = shape_checks(__func__, NQ, T + NQ, Hq, Hkv, D)) return rc;
  SPX_REQUIRE(T > 0, "T must be positive");
  SPX_REQUIRE(q && k && v && out && dout && lse && ctx_lo && ctx_hi && blk_lo && blk_hi && dq && dk &&
              dv && workspace, "null buffer");
  SPX_REQUIRE(q_head_stride >= NQ * D && dq_head_stride >= NQ * D, "q / dq head stride smaller than NQ*D");
  const int64_t kv_rows = (T + NQ) * D;
  SPX_REQUIRE(k_head_stride >= kv_rows && v_head_stride >= kv_rows && dk_head_stride >= kv_rows &&
              dv_head_stride >= kv_rows, "k/v/dk/dv head stride smaller than (T+NQ)*D");
  SPX_REQUIRE((q_head_stride | k_head_stride | v_head_stride | dq_head_stride | dk_head_stride |
               dv_head_stride) % 8 == 0, "head strides must be multiples of 8 elements");
  SPX_REQUIRE(workspace_bytes >= bwd_workspace_bytes(NQ, T + NQ, Hq, Hkv, D), "workspace too small");
  SPX_REQUIRE(all_aligned16({q, k, v, out, dout, dq, dk, dv, workspace}), "buffers must be 16-byte aligned");
  AttnParams p = dflash_params(q, q_head_stride, k, k_head_stride, v, v_head_stride, ctx_lo, ctx_hi,
                               blk_lo, blk_hi, T, NQ, Hq, Hkv, scaling);
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  auto Op = reinterpret_cast<const uint16_t*>(out);
  auto dOp = reinterpret_cast<const uint16_t*>(dout);
  auto dQp = reinterpret_cast<uint16_t*>(dq);
  auto dKp = reinterpret_cast<uint16_t*>(dk);
  auto dVp = reinterpret_cast<uint16_t*>(dv);
  if (D == 256)
    return launch_bwd<256>(p, Op, dOp, lse, dQp, dq_head_stride, dKp, dk_head_stride, dVp, dv_head_stride,
                           workspace, st, __func__);
  if (D == 128)
    return launch_bwd<128>(p, Op, dOp, lse, dQp, dq_head_stride, dKp, dk_head_stride, dVp,
                           dv_head_stride, workspace, st, __func__);
  return launch_bwd<64>(p, Op, dOp, lse, dQp, dq_head_stride, dKp, dk_head_stride, dVp, dv_head_stride,
                        workspace, st, __func__);
}
