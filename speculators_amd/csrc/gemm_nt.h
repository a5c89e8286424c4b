// What the two NT kernels (gemm_bf16.hip: a workgroup a tile; gemm_bf16_walk.hip: workgroups that walk the tiles) share: the
// shape of a tile, the plans of a cut last round and the order of the tiles.
#pragma once

#include "gemm_tile_api.h"
#include "spx_common.h"

namespace spx {

#define SPX_GEMM_WM 2
#define SPX_GEMM_WN 2
#define SPX_GEMM_MINW 1
#define SPX_GEMM_READ_EVERY 2  // MFMAs per LDS fragment read
#define SPX_GEMM_LOAD_EVERY 8  // MFMAs per global -> LDS load ...
#define SPX_GEMM_LOAD_AT 2     // ... of which the load follows this one (the reads follow the odd ones)
constexpr int kWM = SPX_GEMM_WM, kWN = SPX_GEMM_WN;  // waves along M / N of the tile
constexpr int kNW = kWM * kWN;
constexpr int kGemmThreads = 64 * kNW;
constexpr int kTM = 256, kTN = 256, kTK = 64;
constexpr int kMI = kTM / kWM / 16, kNI = kTN / kWN / 16;  // 16x16 accumulators per wave
constexpr int kKSteps = kTK / 32;                          // MFMA K steps per slab
constexpr int kRowBytes = kTK * 2;                          // 128
constexpr int kABytes = kTM * kRowBytes;                    // one slab of A: 32 KB
constexpr int kBBytes = kTN * kRowBytes;
constexpr int kBBase = 2 * kABytes;
constexpr int kGemmSmem = 2 * kABytes + 3 * kBBytes;  // 160 KB: all there is
constexpr int kLA = kTM / 8 / kNW;                  // wave-loads of A per wave per slab
constexpr int kLB = kTN / 8 / kNW;
constexpr int kL = kLA + kLB;
constexpr int kOob = 0x7ffffff0;
static_assert(kABytes == 32768 && kBBytes == 32768, "the buffer toggle flips bit 15");
static_assert(kLA % 4 == 0 && kLB % 4 == 0, "loads are grouped in fours (immediate offsets)");

__device__ __forceinline__ bf16x8 as_frag(u32x4 v) {
  union { u32x4 u; bf16x8 b; } c;
  c.u = v;
  return c.b;
}


// The tiles of the last, partly filled round of a product (n_tiles % cus of them, when they are at most
// half a round): each is cut along the contraction into as many parts as fill the idle compute units
// (at most max_parts, every part at least 16 slabs), so that the round takes a part's time instead of a
// tile's.  384 tiles on 256 compute units: 256 whole tiles, then 128 tiles x 2 halves -- 1.5 rounds of
// work in 1.5 rounds of time instead of 2.  first = index of the first tile that is cut (n_tiles: none).
__host__ __device__ __forceinline__ void tail_plan(int n_tiles, int cus, int nslab, int max_parts, int& first,
                                                   int& parts) {
  first = n_tiles;
  parts = 1;
  if (n_tiles <= 0 || cus <= 0) return;
  const int rem = n_tiles % cus;
  if (rem == 0 || rem * 2 > cus) return;
  int tp = cus / rem;
  if (tp > max_parts) tp = max_parts;
  while (tp > 1 && nslab / tp < 16) --tp;
  if (tp > 1) { first = n_tiles - rem; parts = tp; }
}

// The same for a product whose rows are counted on the device, and for any last round: as many parts (at most max_parts, each
// at least 16 slabs, tiles x parts at most `room` partial tiles) as make it shortest.  The times are those of the 256 x 256 tile,
// as gemm_tile.hip has them, 16 us for a part's start and its 256 KB of partial results, and the pass behind it
// (reduce_us there); one more part has to promise 3 %.  In whole numbers, nanoseconds times compute units: the product, the pass
// that adds its parts and the host each work the plan out, and have to find the same one however they are compiled.
// 400 tiles: 256 whole ones, then 144 in 5 parts, 3 / 5 of a round in the
// place of one.  x 32000, us, all tiles cut in up to 4 parts (where there are at most 512) / so: -> 4096, 6300 live of 9003 rows
// 1455 / 1300, 4500 of them 1416 / 898, 4200 of 6000 1042 / 867; -> 8192, 2150 of 3072 1020 / 865; -> 2048, 1260 of 1800
// 173 / 154, 900 of them 152 / 116, 1800 of them 202 / 208; worst 1800 of 3600 200 / 209.
__host__ __device__ __forceinline__ void live_tail_plan(int n_tiles, int cus, int nslab, int max_parts, int room, int& first,
                                                        int& parts) {
  first = n_tiles;
  parts = 1;
  const int rem = n_tiles > 0 ? n_tiles % cus : 0;
  if (rem == 0) return;
  auto rounds = [&](int wgs, int slabs) __attribute__((always_inline)) {
    const int last = wgs % cus;
    return (int64_t)slabs * ((int64_t)(wgs / cus) * 1410 * cus + (last ? 1180 * cus + 230 * last : 0));
  };
  int64_t best = rounds(rem, nslab) + 6900 * cus;
  for (int p = 2; p <= max_parts && nslab / p >= 16 && rem * p <= room; ++p) {
    const int64_t t = rounds(rem * p, (nslab + p - 1) / p) +
                      (int64_t)cus * (16000 * ((rem * p + cus - 1) / cus) + 4100 + rem * p * 135 / 2);  // (67.5 ns a partial tile)
    if (t * 100 < best * 97) { best = t; first = n_tiles - rem; parts = p; }
  }
}

// a / b for 0 <= a < 2^22, 0 < b: a reciprocal and a correction in the place of the compiler's long division
__device__ __forceinline__ int small_div(int a, int b) {
  int q = (int)((float)a * __builtin_amdgcn_rcpf((float)b));
  const int r = a - q * b;
  q += r >= b ? 1 : r < 0 ? -1 : 0;
  return __builtin_amdgcn_readfirstlane(q);
}

// workgroup id -> place in the order of the work.  Workgroups go to the eight XCDs round robin, XCD x gets the ids x, x + 8, ...: they
// are renumbered so that in every round of 256 workgroups each XCD has 32 consecutive places, and in what is left after the last whole
// round one contiguous piece (the first n % 8 XCDs one more).
__device__ __forceinline__ int xcd_order(int id, int n_wg) {
  constexpr int kRound = 256, kPer = kRound / 8;
  const int xcd = id & 7, local = id >> 3, full = n_wg / kRound * kRound;
  if (id < full) return (local / kPer) * kRound + xcd * kPer + local % kPer;
  const int nr = n_wg - full;
  return full + xcd * (nr >> 3) + min(xcd, nr & 7) + (local - full / 8);
}

// tile index -> (tile row, tile column).  256 consecutive indices (what the chip runs at a time) are a block of
// 16 x 16 tiles, so that a 256-row band of either operand is used by 16 of the tiles in flight, and the blocks walk
// along the longer side of the tile grid; 32 consecutive indices (what one XCD runs: see the kernel) are 8 tiles
// along the longer side x 4 along the shorter, 12 operand bands through that XCD's L2.  In detail: panels of 16
// along the shorter side; inside a panel groups of 8 along the longer side; inside a group the longer side first.
template <bool kSmall = false>  // fewer than 2^22 tiles
__device__ __forceinline__ void tile_coords(int pid, int tiles_m, int tiles_n, int& tile_m, int& tile_n) {
  auto div = [](int a, int b) __attribute__((always_inline)) { return kSmall ? small_div(a, b) : a / b; };
  constexpr int kPanel = 16, kGroup = 8;
  const bool m_long = tiles_m >= tiles_n;
  const int tl = m_long ? tiles_m : tiles_n, ts = m_long ? tiles_n : tiles_m;
  const int panel = div(pid, tl * kPanel);
  const int ps = min(ts - panel * kPanel, kPanel);
  const int p = pid - panel * tl * kPanel;
  const int g = div(p, kGroup * ps);
  const int gsz = min(tl - g * kGroup, kGroup);
  const int r = p - g * kGroup * ps, across = div(r, gsz);
  const int l = g * kGroup + r - across * gsz, sh = panel * kPanel + across;
  tile_m = m_long ? l : sh;
  tile_n = m_long ? sh : l;
}

}  // namespace spx
