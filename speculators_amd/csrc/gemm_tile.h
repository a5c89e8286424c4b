// bf16 GEMM kernels for gfx950 on smaller tiles than those of gemm_bf16.hip (NT, NN and TN forms, plain, cut along
// the contraction, grouped).  Instantiated, chosen and launched by gemm_tile.hip.
//
// Direct global -> LDS loads, STAGES slabs of 64 contraction indices deep (ring_b), v_mfma_f32_16x16x32_bf16, operand
// fragments double buffered in registers, the LDS reads of the next K step and the loads of the next free slab issued
// between the products, one barrier per slab.  What bounds them is the way into LDS: with one tile on every compute unit
// and K to 16384 the tiles of 64 x 128, 128 x 128 and 256 x 128 all load at 61 - 79 GB/s per compute unit (16 - 20 TB/s over
// the chip) -- 0.31, 0.49 and 0.78 us a slab, 870, 1100 and 1380 TFLOP/s; 256 x 256, NN: 1.50 us, 1430 TFLOP/s, the
// products bound it -- so a larger tile is faster per multiply-add as long as every compute unit has one.
//
// STAGES = 1: one slab buffer and one register set per operand, so four workgroups of 128 x 128 (two of 128 x 256) share a
// compute unit and one's stores, loads and products run beside another's: what a product needs whose contraction is so
// short that a workgroup is mostly start and end.
//
// Results leave in whole 128-byte lines (`line_pair`), past the caches where they are large (STREAM).
// The weight gradients of 512 experts (2.1 GB from 80 rows each, operands in the memory-side cache, back to back) leave at
// 3.2 TB/s as 64-byte pieces, 3.3 in whole lines, 3.6 past the caches and 4.6 with both.
#pragma once

#include <type_traits>

#include "gemm_tile_api.h"
#include "spx_common.h"

namespace spx {
namespace tile {

constexpr int kTK = 64;  // contraction columns per slab
constexpr int kOob = 0x7ffffff0;

typedef short i16x4 __attribute__((ext_vector_type(4)));
typedef short i16x8 __attribute__((ext_vector_type(8)));

__device__ __forceinline__ i16x4 read_tr16(uint32_t addr) {
  return __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) i16x4*)(uintptr_t)addr);
}

// (a template argument: the compiler merges the two stores of a run-time choice into the cached one)
template <bool STREAM>
__device__ __forceinline__ void store_line(void* p, u32x4 v) {
  if constexpr (STREAM) __builtin_nontemporal_store(v, reinterpret_cast<u32x4*>(p));
  else *reinterpret_cast<u32x4*>(p) = v;
}

// Slab buffers of B where A has `stages`.  With two, B has a third, a free one at any time: its loads run under the first K
// step of a slab, A's under the second, instead of all under the second.  Two of each / so, us: 3001 x 28672 -> 4096, NN 565
// / 521, 8192 x 4096 -> 14336, NN 702 / 684, 1777 rows -> 2048 x 10240, TN 82.5 / 78.4, 64 groups of 1024 rows x 2048 -> 1536 403 /
// 388, x 1536 -> 2048, NN 425 / 400.  (With three or four of each, B's loads half a slab later so that they follow each other
// evenly: 0 - 5 % longer.)
__host__ __device__ constexpr int ring_b(int stages) { return stages == 2 ? 3 : stages; }

template <int N>
using at = std::integral_constant<int, N>;

template <int N>
__device__ __forceinline__ void wait_vmcnt() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// One operand of a tile: kR rows of C (or columns of C) x one slab of 64 contraction indices, staged through LDS.
// SLOW = false: the contraction index is contiguous in memory (a row of the operand holds it); LDS holds kR rows
// of 128 bytes, 16-byte chunk c of row r in slot c ^ f(r), f(r) = (r & 7) ^ ((r >> 3) & 1).
// SLOW = true: the contraction index is the slow one (the operand is stored [contraction, kR columns]); LDS holds
// 64 rows of 2 kR bytes, 32-byte piece p of row t in position p ^ h(t), h(t) = t % 4 + 4 (t / 8 % 2), and the
// fragments are taken with the transposing read.
template <int kR, int kWaves, bool SLOW>
struct Operand {
  static constexpr int kBytes = kR * kTK * 2;         // per slab
  static constexpr int kLoads = kBytes / 1024 / kWaves;  // 1 KB wave-loads per wave and slab
  static_assert(kBytes % (1024 * kWaves) == 0, "whole wave-loads");
  static_assert(!SLOW || (kR & (kR - 1)) == 0, "whole rows per wave-load");
  u32x4 rsrc;
  int off[kLoads];
  int kchunk[SLOW ? 1 : 2];  // first contraction index of this lane's chunk inside the slab (even / odd row groups)
  int row_bytes;

  // base: the operand's first element of this tile (and contraction range); rows: how many of the kR lie inside the
  // matrix; len: contraction length
  __device__ __forceinline__ void init(const uint16_t* base, int64_t ld, int rows, int len, int wave, int lane) {
    row_bytes = (int)(ld * 2);
    if (!SLOW) {
      rsrc = make_rsrc(base, len > 0 && rows > 0 ? (uint32_t)((((int64_t)min(rows, kR) - 1) * ld + len) * 2) : 0u);
      const int lrow = lane >> 3;
      const int c0 = (lane & 7) ^ (lrow & 7);
      kchunk[0] = c0 * 8;
      if constexpr (!SLOW) kchunk[1] = (c0 ^ 1) * 8;
#pragma unroll
      for (int j = 0; j < kLoads; ++j) {
        const int g = wave * kLoads + j;  // 8-row group
        const int r = g * 8 + lrow;
        off[j] = r < rows ? (int)(((int64_t)r * ld + (c0 ^ (g & 1)) * 8) * 2) : kOob;
      }
    } else {
      rsrc = make_rsrc(base, len > 0 && rows > 0 ? (uint32_t)((((int64_t)len - 1) * ld + min(rows, kR)) * 2) : 0u);
      constexpr int kRow = kR * 2, kPerLoad = 1024 / kRow, kLanes = kRow / 16;
      const int lrow = lane / kLanes, lpos = lane % kLanes;
#pragma unroll
      for (int j = 0; j < kLoads; ++j) {
        const int r = kPerLoad * (wave * kLoads + j) + lrow;
        const int hr = ((r & 3) | (((r >> 3) & 1) << 2)) & (kR / 16 - 1);
        const int c8 = ((((lpos >> 1) ^ hr) << 1) | (lpos & 1)) * 8;
        off[j] = c8 < rows ? (int)(((int64_t)r * ld + c8) * 2) : kOob;
      }
    }
  }

  // The same with rows picked out of a larger matrix: row r of the operand is row src[r] of `base` (a number outside of
  // 0 .. src_rows - 1: zeros).  The whole of that matrix lies below 2 GiB.
  // SLOW = false: the operand's rows, looked up once here
  __device__ __forceinline__ void init_picked(const uint16_t* base, int64_t ld, int rows, int len, int wave, int lane,
                                              const int32_t* src, int src_rows) {
    init(base, ld, rows, len, wave, lane);
    rsrc = make_rsrc(base, len > 0 ? (uint32_t)((((int64_t)src_rows - 1) * ld + len) * 2) : 0u);
    const int lrow = lane >> 3;
#pragma unroll
    for (int j = 0; j < kLoads; ++j) {
      const int r = (wave * kLoads + j) * 8 + lrow;
      const int from = r < rows ? src[r] : -1;
      off[j] = (uint32_t)from < (uint32_t)src_rows ? off[j] + (int)((int64_t)(from - r) * ld * 2) : kOob;
    }
  }
  // SLOW = true: the contraction's rows, looked up slab by slab (`pick`, a slab ahead of its loads)
  __device__ __forceinline__ void init_picked_slow(const uint16_t* base, int64_t ld, int cols, int wave, int lane, int src_rows) {
    init(base, ld, cols, 1, wave, lane);
    rsrc = make_rsrc(base, (uint32_t)((((int64_t)src_rows - 1) * ld + min(cols, kR)) * 2));
#pragma unroll
    for (int j = 0; j < kLoads; ++j)
      if (off[j] != kOob) off[j] -= slab_row(j, wave, lane) * row_bytes;  // (the column's part alone)
  }
  __device__ __forceinline__ static int slab_row(int j, int wave, int lane) {
    constexpr int kPerLoad = 1024 / (kR * 2);
    return kPerLoad * (wave * kLoads + j) + lane / (kR * 2 / 16);
  }
  __device__ __forceinline__ void pick(int (&rows)[kLoads], const int32_t* src, int src_rows, int k0, int len, int wave,
                                       int lane) const {
#pragma unroll
    for (int j = 0; j < kLoads; ++j) {
      const int k = k0 + slab_row(j, wave, lane);
      const int from = k < len ? src[k] : -1;
      rows[j] = (uint32_t)from < (uint32_t)src_rows ? from : -1;
    }
  }
  __device__ __forceinline__ void load_picked(int j, uint32_t lds, const int (&rows)[kLoads], int wave) const {
    const bool in = rows[j] >= 0 && off[j] != kOob;
    load_to_lds16<0>(rsrc, lds + (wave * kLoads + j) * 1024, in ? off[j] + rows[j] * row_bytes : kOob, 0);
  }

  // wave-load j of the slab at contraction index k0 into the LDS slab at `lds` (this operand's base)
  __device__ __forceinline__ void load(int j, uint32_t lds, int k0, int len, int wave) const {
    const uint32_t dst = lds + (wave * kLoads + j) * 1024;
    if (!SLOW) {
      // (a chunk past the end of the contraction would read the next row: its lane goes out of range)
      const int g = wave * kLoads + j;
      const int kc = k0 + ((g & 1) ? kchunk[SLOW ? 0 : 1] : kchunk[0]);
      load_to_lds16<0>(rsrc, dst, kc < len ? off[j] : kOob, k0 * 2);
    } else {
      // the whole offset is in the vector register, which is what the range check sees
      load_to_lds16<0>(rsrc, dst, (int)((uint32_t)off[j] + (uint32_t)k0 * (uint32_t)row_bytes), 0);
    }
  }

  // fragment f (16 rows of this wave's stripe, which starts at row w0) of K step kk out of the slab at `lds`
  __device__ __forceinline__ static uint32_t read_base(uint32_t lds0, int w0, int lane) {
    const int q = lane >> 4, r16 = lane & 15;
    if (!SLOW) {
      const int fr = (r16 & 7) ^ (r16 >> 3);
      return lds0 + (w0 + r16) * 128 + ((q ^ fr) * 16);
    }
    const int trow = 8 * q + (r16 >> 2);
    return lds0 + trow * (kR * 2) + 8 * (r16 & 3);
  }
  __device__ __forceinline__ static bf16x8 read(uint32_t base, uint32_t slab, int w0, int f, int kk, int lane) {
    if (!SLOW) {
      union { u32x4 u; bf16x8 b; } c;
      c.u = lds_read128((base ^ (kk * 64)) + slab + f * 16 * 128);
      return c.b;
    }
    const int q = lane >> 4, r16 = lane & 15;
    const int h = ((r16 >> 2) | ((q & 1) << 2)) & (kR / 16 - 1);
    const uint32_t a = base + slab + kk * 32 * (kR * 2) + ((((w0 >> 4) + f) ^ h) * 32);
    const i16x4 lo = read_tr16(a), hi = read_tr16(a + 4 * (kR * 2));
    const i16x8 v = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
    return __builtin_bit_cast(bf16x8, v);
  }
};

// The parts of a product whose rows are counted on the device: those that make it shortest, as the host has it for all M rows
// (choose in gemm_tile.hip), for the tiles that are there.  max_parts = 0: as the host says.  In whole numbers, nanoseconds times
// the workgroups that the chip holds: the product, the pass that adds its parts and the host each work the parts out, and have
// to find the same however they are compiled.
struct LiveCut {
  int max_parts, cap, slabs;  // cap: workgroups the chip holds
  int s0, s1;                 // of the tile's Config, in ns
  __host__ __device__ __forceinline__ int parts(int tiles, int64_t results) const {
    int best = 1;
    int64_t ns = 0;
    for (int n = 1; n <= max_parts && (n == 1 || (int64_t)tiles * n <= cap); ++n) {
      const int wgs = tiles * n < cap ? tiles * n : cap;  // (n == 1: as many tiles as there are)
      const int64_t t = ((int64_t)s0 * cap + (int64_t)s1 * wgs) * ((slabs + n - 1) / n) +
                        (n > 1 ? cap * (4100 + n * results * 103 / 100000) : 0);
      if (n == 1 || t < ns) { ns = t; best = n; }
    }
    return tiles > 0 ? best : 1;
  }
};

struct Params {
  const uint16_t* A;
  const uint16_t* B;
  void* C;
  int64_t lda, ldb, ldc;
  int M, N, K;
  int tiles_m, tiles_n;
  int parts;                    // the contraction is cut into this many parts (> 1: fp32 partials in part_ws)
  float* part_ws;               // [parts][M][N]
  const int32_t* tile_tab;      // grouped NT / NN: (group, first row) per tile row, see group_tiles_kernel
  const int32_t* group_off;     // grouped: group boundaries
  const int32_t* m_live;        // how many leading rows of A count (device; null: all M)
  int64_t group_stride;         // elements between the groups' B (NT / NN) or C (TN)
  const int32_t* src;           // PICK: where each of the operand's rows lies in the matrix it is picked from ...
  int src_rows;                 // ... and that matrix's rows
  RowGrade grade;               // GRADE: what the rows are multiplied by
  LiveCut cut;                  // GRADE: parts by the rows that count, [parts][whole tile rows of them][N] then
};

// OUT: 0 = bf16, 1 = bf16 added to C, 2 = fp32, 3 = fp32 added to C.  STREAM: non-temporal stores (OUT 0 and 2).  GRADE: rows
// multiplied by their factors on the way to their rounding (OUT 0; of a product in parts the pass that adds them does it).
// PICK (grouped): the rows of A (1) or B (2) -- of the contraction, where that is the slow index -- are those of a larger
// matrix that p.src names
template <int TM, int TN, int WM, int WN, int STAGES, int MINB, bool AT, bool BT, int OUT, bool STREAM, bool GRADE, int PICK>
__global__ __launch_bounds__(64 * WM * WN, MINB) void gemm_tile_kernel(Params p) {
  static_assert(PICK == 0 || (AT ? BT && STAGES == 1 : PICK == 1), "picked rows: A of the NT and NN forms, one slab of TN");
  constexpr int kWaves = WM * WN, kMI = TM / WM / 16, kNI = TN / WN / 16;
  using OA = Operand<TM, kWaves, AT>;
  using OB = Operand<TN, kWaves, BT>;
  // slab buffers: A and B in turn, or where B has one more, all of A, then all of B
  constexpr int kRingB = ring_b(STAGES);
  constexpr bool kMoreB = kRingB > STAGES;
  constexpr int kStage = kMoreB ? OA::kBytes : OA::kBytes + OB::kBytes;
  constexpr int kBBase = kMoreB ? STAGES * kStage : OA::kBytes;
  constexpr int kL = OA::kLoads + OB::kLoads;
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)smem;

  int M = p.M, K = p.K;
  const uint16_t *A = p.A, *B = p.B;
  void* C = p.C;
  int tiles_m = p.tiles_m;
  if (!AT && p.m_live) {  // the tile grid shrinks to the rows that count
    M = min(M, max(*p.m_live, 0));
    tiles_m = (M + TM - 1) / TM;
  }
  if (!AT && p.tile_tab) tiles_m = min(p.tile_tab[0], tiles_m);
  const int n_tiles = tiles_m * p.tiles_n;
  int parts = p.parts;
  if (GRADE && p.cut.max_parts) parts = p.cut.parts(n_tiles, (int64_t)M * p.N);
  const int n_wg = n_tiles * parts;
  if ((int)blockIdx.x >= n_wg) return;
  // one contiguous run of workgroups per XCD (they go to the eight XCDs round robin), tiles in it first, then parts:
  // an XCD's tiles share their operand bands in its L2, and with eight parts or more an XCD reads only its part of
  // the contraction (12 % at 512 x 2048 x 8192 in 8 parts against all parts of a tile in one XCD)
  int pid;
  {
    const int xcd = blockIdx.x & 7, local = blockIdx.x >> 3, base = n_wg >> 3, rem = n_wg & 7;
    pid = xcd * base + min(xcd, rem) + local;
  }
  const int part = pid / n_tiles;
  pid -= part * n_tiles;
  int tm, tn;
  if (!AT && p.tile_tab) {  // grouped: the column tiles of one tile row run together (they share the group's rows)
    tm = pid / p.tiles_n;
    tn = pid % p.tiles_n;
  } else {
    // groups of four tile rows, columns first inside a group
    constexpr int kGroup = 4;
    const int g = pid / (kGroup * p.tiles_n), r = pid % (kGroup * p.tiles_n);
    const int gs = min(tiles_m - g * kGroup, kGroup);
    tm = g * kGroup + r % gs;
    tn = r / gs;
  }
  int m0 = tm * TM;
  const int n0 = tn * TN;
  if (!AT && p.tile_tab) {
    const int grp = p.tile_tab[1 + 2 * tm];
    m0 = p.tile_tab[2 + 2 * tm];
    M = min(M, max(p.group_off[grp + 1], 0));
    B += (int64_t)grp * p.group_stride;
  }
  if (AT && p.group_off) {  // grouped TN: blockIdx.y = group, the contraction runs over its rows
    const int e = blockIdx.y;
    const int t0 = min(max(p.group_off[e], 0), p.K), t1 = min(max(p.group_off[e + 1], t0), p.K);
    if (PICK != 1) A += (int64_t)t0 * p.lda;
    if (PICK != 2) B += (int64_t)t0 * p.ldb;
    if (PICK) p.src += t0;
    K = t1 - t0;
    C = reinterpret_cast<uint8_t*>(C) + (int64_t)e * p.group_stride * (OUT >= 2 ? 4 : 2);
    if ((OUT & 1) && K == 0) return;
  }
  if (parts > 1) {
    const int slabs = ((K + kTK - 1) / kTK + parts - 1) / parts;
    const int k_begin = part * slabs * kTK;
    A += AT ? (int64_t)k_begin * p.lda : (int64_t)k_begin;
    B += BT ? (int64_t)k_begin * p.ldb : (int64_t)k_begin;
    K = max(min(K - k_begin, slabs * kTK), 0);
  }

  OA oa;
  OB ob;
  if constexpr (PICK == 1 && AT) oa.init_picked_slow(A + m0, p.lda, M - m0, wave, lane, p.src_rows);
  else if constexpr (PICK == 1) oa.init_picked(A, p.lda, M - m0, K, wave, lane, p.src + m0, p.src_rows);
  else oa.init(AT ? A + m0 : A + (int64_t)m0 * p.lda, p.lda, M - m0, K, wave, lane);
  if constexpr (PICK == 2) ob.init_picked_slow(B + n0, p.ldb, p.N - n0, wave, lane, p.src_rows);
  else ob.init(BT ? B + n0 : B + (int64_t)n0 * p.ldb, p.ldb, p.N - n0, K, wave, lane);
  const int wm = (wave / WN) * (TM / WM), wn = (wave % WN) * (TN / WN);
  const uint32_t a_rd = OA::read_base(lds0, wm, lane), b_rd = OB::read_base(lds0 + kBBase, wn, lane);

  f32x4 acc[kNI][kMI];
#pragma unroll
  for (int j = 0; j < kNI; ++j)
#pragma unroll
    for (int i = 0; i < kMI; ++i) acc[j][i] = f32x4{0.f, 0.f, 0.f, 0.f};

  const int nslab = (K + kTK - 1) / kTK;
  int ld_k = 0;  // contraction index of the slab being loaded
  uint32_t ld_at = lds0, ld_at_b = lds0 + kBBase;
  constexpr int kPick = AT ? PICK : 0;
  int picked[kPick == 1 ? OA::kLoads : OB::kLoads];  // rows of the slab that is loaded next
  auto pick = [&](int k0) __attribute__((always_inline)) {
    if constexpr (kPick == 1) oa.pick(picked, p.src, p.src_rows, k0, K, wave, lane);
    else if constexpr (kPick == 2) ob.pick(picked, p.src, p.src_rows, k0, K, wave, lane);
  };
  auto issue_one = [&](int l) __attribute__((always_inline)) {
    if (l < OA::kLoads) {
      if constexpr (kPick == 1) oa.load_picked(l, ld_at, picked, wave);
      else oa.load(l, ld_at, ld_k, K, wave);
    } else {
      const uint32_t to = kMoreB ? ld_at_b : ld_at + kBBase;
      if constexpr (kPick == 2) ob.load_picked(l - OA::kLoads, to, picked, wave);
      else ob.load(l - OA::kLoads, to, ld_k, K, wave);
    }
  };
  auto next_load = [&]() __attribute__((always_inline)) {
    ld_k += kTK;
    ld_at = ld_at + kStage == lds0 + STAGES * kStage ? lds0 : ld_at + kStage;
    if (kMoreB) ld_at_b = ld_at_b + OB::kBytes == lds0 + kBBase + kRingB * OB::kBytes ? lds0 + kBBase : ld_at_b + OB::kBytes;
  };
  constexpr int kSets = STAGES == 1 ? 1 : 2;
  bf16x8 fa[kSets][kMI], fb[kSets][kNI];
  uint32_t rd = 0, rd_b = 0;  // slab buffer the reads go to, and B's where it has more
  auto read_one = [&](int set, int kk, int f) __attribute__((always_inline)) {
    if (f < kMI) fa[set][f] = OA::read(a_rd, rd, wm, f, kk, lane);
    else fb[set][f - kMI] = OB::read(b_rd, kMoreB ? rd_b : rd, wn, f - kMI, kk, lane);
  };
  // Grouped NT and NN: a wave whose rows are all past its group's loads and waits with the others, but multiplies nothing
  // (nor reads its operands, where there are several slab buffers): a group of 80 rows on average is half a tile.  4096 tokens, top 10 of 512 experts of uneven popularity, gate/up 470
  // -> 448 us, down 256 -> 248, its input gradient 227 -> 226, gate/up's 425 -> 416; 12000 tokens 685 -> 676, 409 -> 402, 342 -> 341, 725 -> 695;
  // 80 rows each: no difference.
  constexpr bool kSkip = !AT && STREAM;
  const bool rows_here = !kSkip || __builtin_amdgcn_readfirstlane(m0 + wm < M);
  // One K step of 32: the products on register set `set`; between them the LDS reads that fill the other set with K
  // step rk and the wave-loads [first, last) of a slab
  auto step = [&](int set, int rk, auto first, auto last) __attribute__((always_inline)) {
    constexpr int kFirst = decltype(first)::value, kCount = decltype(last)::value - kFirst;
    if (kSkip && !rows_here) {
#pragma unroll
      for (int l = 0; l < kCount; ++l) issue_one(kFirst + l);
      return;
    }
    constexpr int kN = kNI * kMI, kF = kMI + kNI;
    int reads = 0;
#pragma unroll
    for (int j = 0; j < kNI; ++j)
#pragma unroll
      for (int i = 0; i < kMI; ++i) {
        acc[j][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fb[set][j], fa[set][i], acc[j][i], 0, 0, 0);
        const int idx = j * kMI + i;
        __builtin_amdgcn_sched_barrier(0);
        // reads in the first three quarters of the step, loads evenly
        while (reads < kF && reads * kN * 3 < (idx + 1) * kF * 4) { read_one(set ^ 1, rk, reads++); }
#pragma unroll
        for (int l = 0; l < kCount; ++l)
          if (l * kN / (kCount > 0 ? kCount : 1) == idx) issue_one(kFirst + l);
        __builtin_amdgcn_sched_barrier(0);
      }
  };

  if constexpr (STAGES == 1) {
    auto products = [&]() __attribute__((always_inline)) {
      if (kSkip && !rows_here) return;
#pragma unroll
      for (int j = 0; j < kNI; ++j)
#pragma unroll
        for (int i = 0; i < kMI; ++i)
          acc[j][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fb[0][j], fa[0][i], acc[j][i], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    };
    pick(0);
#pragma unroll
    for (int l = 0; l < kL; ++l) issue_one(l);
    if (nslab > 1) pick(kTK);
    for (int s = 0; s < nslab; ++s) {
      wait_vmcnt<0>();
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      const bool two = K - s * kTK > 32;  // (a last slab of up to 32 indices is one K step)
      if (two) {
#pragma unroll
        for (int f = 0; f < kMI + kNI; ++f) read_one(0, 0, f);
        products();
      }
      const int kk = two ? 1 : 0;
#pragma unroll
      for (int f = 0; f < kMI + kNI; ++f) read_one(0, kk, f);
      if (s + 1 < nslab) {
        // every wave has read its fragments: the buffer is free
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        ld_k += kTK;
#pragma unroll
        for (int l = 0; l < kL; ++l) issue_one(l);
        if (s + 2 < nslab) pick(ld_k + kTK);
      }
      __builtin_amdgcn_sched_barrier(0);
      products();
    }
  } else {
    // The loads of slab s + STAGES are issued under the second K step of slab s, B's under the first where it has a buffer
    // more.  Past the last slab they bring zeros
#pragma unroll
    for (int s = 0; s < STAGES; ++s) {
#pragma unroll
      for (int l = 0; l < kL; ++l) issue_one(l);
      next_load();
    }
    wait_vmcnt<(STAGES - 1) * kL>();
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
#pragma unroll
    for (int f = 0; f < kMI + kNI; ++f) read_one(0, 0, f);
    for (int s = 0; s < nslab; ++s) {
      __builtin_amdgcn_sched_barrier(0);
      step(0, 1, at<OA::kLoads>{}, at<kMoreB ? kL : OA::kLoads>{});
      // every read of slab s has returned; after the barrier for every wave (its buffers are free) and slab s + 1 has
      // landed for everybody
      asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"((STAGES - 2) * kL + (kMoreB ? OB::kLoads : 0)) : "memory");
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      rd = rd + kStage == STAGES * kStage ? 0 : rd + kStage;
      if (kMoreB) rd_b = rd_b + OB::kBytes == kRingB * OB::kBytes ? 0 : rd_b + OB::kBytes;
      step(1, 0, at<0>{}, at<kMoreB ? OA::kLoads : kL>{});
      next_load();
    }
  }
  wait_vmcnt<0>();

  // a lane holds row m of C and, per accumulator, columns 4 q + {0..3} of a 16-column block
  const int q = lane >> 4, r16 = lane & 15;
  if (parts > 1) {
    float* const P = p.part_ws + (int64_t)part * (GRADE && p.cut.max_parts ? tiles_m * TM : p.M) * p.N;
#pragma unroll
    for (int i = 0; i < kMI; ++i) {
      const int m = m0 + wm + i * 16 + r16;
      if (m >= M) continue;
#pragma unroll
      for (int j = 0; j < kNI; ++j) {
        const int n = n0 + wn + j * 16 + 4 * q;
        if (n < p.N) *reinterpret_cast<f32x4*>(P + (int64_t)m * p.N + n) = acc[j][i];
      }
    }
    return;
  }
  if constexpr (OUT >= 2) {
    float* const Cf = reinterpret_cast<float*>(C);
    const bool fast = (p.ldc % 4 == 0) && ((reinterpret_cast<uintptr_t>(Cf) & 15) == 0);
    if (OUT == 2 && fast) {
      const bool lo = r16 < 8;
#pragma unroll
      for (int i = 0; i < kMI; ++i)
#pragma unroll
        for (int j = 0; j < kNI; j += 2) {
          u32x4 x, y;
          line_pair(lo, __builtin_bit_cast(u32x4, acc[j][i]), __builtin_bit_cast(u32x4, acc[j + 1][i]), x, y);
          const int m = m0 + wm + i * 16 + (r16 & 7), n = n0 + wn + j * 16 + (lo ? 0 : 16) + 4 * q;
          float* cp = Cf + (int64_t)m * p.ldc + n;
          if (n + 4 <= p.N) {
            if (m < M) store_line<STREAM>(cp, x);
            if (m + 8 < M) store_line<STREAM>(cp + 8 * p.ldc, y);
          } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              if (n + e >= p.N) continue;
              if (m < M) cp[e] = __uint_as_float(x[e]);
              if (m + 8 < M) cp[8 * p.ldc + e] = __uint_as_float(y[e]);
            }
          }
        }
      return;
    }
#pragma unroll
    for (int i = 0; i < kMI; ++i) {
      const int m = m0 + wm + i * 16 + r16;
      if (m >= M) continue;
#pragma unroll
      for (int j = 0; j < kNI; ++j) {
        const int n = n0 + wn + j * 16 + 4 * q;
        float* cp = Cf + (int64_t)m * p.ldc + n;
        if (fast && n + 4 <= p.N) {
          f32x4 v = acc[j][i];
          if (OUT == 3) v += *reinterpret_cast<const f32x4*>(cp);
          *reinterpret_cast<f32x4*>(cp) = v;
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (n + e < p.N) cp[e] = (OUT == 3 ? cp[e] : 0.f) + acc[j][i][e];
        }
      }
    }
  } else {
    if constexpr (GRADE) {
#pragma unroll
      for (int i = 0; i < kMI; ++i) {
        const int m = m0 + wm + i * 16 + r16;
        const float by = m < M ? p.grade.at(m) : 0.f;
#pragma unroll
        for (int j = 0; j < kNI; ++j) acc[j][i] *= by;
      }
    }
    uint16_t* const Cb = reinterpret_cast<uint16_t*>(C);
    const bool fast = (p.ldc % 8 == 0) && ((reinterpret_cast<uintptr_t>(Cb) & 15) == 0);
    // odd groups of 16 lanes of block j <-> even groups of block j + 1: 8 consecutive columns per lane
    auto pack8 = [](f32x4 a, f32x4 b) __attribute__((always_inline)) {
      const auto s0 = __builtin_amdgcn_permlane16_swap(pack_bf16x2(a[0], a[1]), pack_bf16x2(b[0], b[1]), false, false);
      const auto s1 = __builtin_amdgcn_permlane16_swap(pack_bf16x2(a[2], a[3]), pack_bf16x2(b[2], b[3]), false, false);
      u32x4 v;
      v.x = s0[0]; v.y = s1[0]; v.z = s0[1]; v.w = s1[1];
      return v;
    };
    if constexpr (OUT == 0 && kNI % 4 == 0) {
      if (fast && p.N % 8 == 0) {
        const bool lo = r16 < 8;
#pragma unroll
        for (int i = 0; i < kMI; ++i)
#pragma unroll
          for (int j = 0; j < kNI; j += 4) {
            u32x4 x, y;
            line_pair(lo, pack8(acc[j][i], acc[j + 1][i]), pack8(acc[j + 2][i], acc[j + 3][i]), x, y);
            const int m = m0 + wm + i * 16 + (r16 & 7);
            const int n = n0 + wn + (j + (lo ? 0 : 2) + (q & 1)) * 16 + 4 * (q & 2);
            if (n >= p.N) continue;
            uint16_t* cp = Cb + (int64_t)m * p.ldc + n;
            if (m < M) store_line<STREAM>(cp, x);
            if (m + 8 < M) store_line<STREAM>(cp + 8 * p.ldc, y);
          }
        return;
      }
    }
#pragma unroll
    for (int i = 0; i < kMI; ++i) {
      const int m = m0 + wm + i * 16 + r16;
#pragma unroll
      for (int j = 0; j < kNI; j += 2) {
        f32x4 a = acc[j][i], b = acc[j + 1][i];
        if (OUT == 1 && m < M) {
          const int na = n0 + wn + j * 16 + 4 * q;
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            if (na + e < p.N) a[e] += bf16_bits_to_f32(Cb[(int64_t)m * p.ldc + na + e]);
            if (na + 16 + e < p.N) b[e] += bf16_bits_to_f32(Cb[(int64_t)m * p.ldc + na + 16 + e]);
          }
        }
        const u32x4 v = pack8(a, b);
        const int n = n0 + wn + (j + (q & 1)) * 16 + 4 * (q & 2);
        if (m >= M) continue;
        if (fast && n + 8 <= p.N) {
          *reinterpret_cast<u32x4*>(&Cb[(int64_t)m * p.ldc + n]) = v;
        } else {
          const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
          for (int e = 0; e < 8; ++e)
            if (n + e < p.N) Cb[(int64_t)m * p.ldc + n + e] = (uint16_t)(w[e >> 1] >> (16 * (e & 1)));
        }
      }
    }
  }
}

}  // namespace tile
}  // namespace spx
