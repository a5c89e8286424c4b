// Weight gradients C_e[M_e, N_e] = A_e[T_e, M_e]^T B_e[T_e, N_e] of a list of products in one launch, by workgroups that walk the
// tiles of all of them, one per compute unit: workgroup w takes the tiles w, w + grid, ... of the list.  Tile, slab buffers, order
// of the loads, reads and products are those of gemm_bf16_tn.hip, the stream of slabs across tiles that of gemm_bf16_walk.hip.
//
// One launch each of the kernels before / this, us: 28672 rows -> 4096 x 14336, fp32 (896 tiles, 128 of them cut in two) 2457 / 2234,
// 32000 -> 6144 x 2048 (192 tiles in four parts) 630 / 605, -> 5120 x 2048 (160 in three) 580 / 506, 9003 -> 28672 x 4096 1423 / 1382;
// the four weights of the 1B shape over 1536 rows, fp32, 219 / 167; of an 8B anchored-block layer over 8192 2717 / 2505; the
// five of the multi-token layer over 32000 3672 / 2853.
//
// What this is for: the gradients of a layer's weights are 64 to 1800 tiles each, and alone each ends in a round of tiles that
// does not fill the chip; with few rows (512 tokens x 3 steps: 24 slabs) a tile is a third start and end.  Together they are
// one run of whole rounds, one last round -- cut along the contraction where that is shorter (tail_of) -- and starts and ends
// that run under the products.
// The products come by falling contraction, so that the tiles of a round take about as long as one another.
// The results leave past the caches where the rows of C begin with lines of 128 bytes (1 - 5 % faster so), through them where they do
// not: the first and last line of a row's 256 or 512 bytes are then shared by two tiles, and a part of a line that goes to memory by
// itself costs as much as two.  Past the caches / through them, us: 192 rows -> 5784 x 29112, fp32, 339 / 194, 697 -> 3520 x 7608,
// fp32, 70 / 46, 192 -> 11776 x 9192 133 / 62, 2339 -> 14448 x 3368 208 / 198.

#include <algorithm>

#include "acc_file.h"
#include "gemm_nt.h"
#include "../../include/spx.h"

namespace spx {
namespace tnw {

constexpr int kMaxItems = 8, kMaxParts = 8;
constexpr int kRow = kTM * 2;  // bytes of a row of a slab
static_assert(kTK * kRow == kABytes && kABytes == kBBytes, "a slab of either operand");

struct Item {
  const uint16_t *a, *b;
  void* c;
  int64_t lda, ldb, ldc;
  int M, N, T, tiles_m, tiles_n;
  int first;  // its first tile in the list (INT32_MAX: no such product)
};
struct List {
  Item item[kMaxItems];
  float* part_ws;
  int n_tiles, tail_first, tail_parts;  // the tiles from tail_first on are cut into so many parts
};
typedef const __attribute__((address_space(4))) List* ListPtr;

__device__ __forceinline__ int item_of(ListPtr list, int tile) {
  int e = 0;
#pragma unroll
  for (int i = 1; i < kMaxItems; ++i) e += tile >= list->item[i].first ? 1 : 0;
  return e;
}

typedef short i16x4 __attribute__((ext_vector_type(4)));
typedef short i16x8 __attribute__((ext_vector_type(8)));

// every T at least 129 (three slabs, and so every part), every leading dimension of a and b at least 256, M and N multiples of 8,
// C 16-byte aligned with a leading dimension that is a multiple of 8.  (The list is read where it lies, among the kernel's
// arguments: an index into an argument array would copy it to the lanes' own memory first.)
template <bool F32>
__global__ __launch_bounds__(kGemmThreads, 1) __attribute__((amdgpu_waves_per_eu(1, 1))) void gemm_bf16_tn_walk_kernel(List) {
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  const ListPtr list = (ListPtr)__builtin_amdgcn_kernarg_segment_ptr();
  const int tail_first = list->tail_first, tail_parts = list->tail_parts, n_tail = list->n_tiles - tail_first;
  const int n_wg = tail_first + n_tail * tail_parts;
  if ((int)blockIdx.x >= n_wg) return;
  constexpr int kSize = F32 ? 4 : 2;

  struct Tile {
    const uint16_t *a, *b;         // the first row of its contraction, its first column
    int a_row, b_row;              // bytes between rows
    int slabs, rows_last;          // rows of the last slab
    int cols_a, cols_b;            // its columns that lie inside a and b: the rows and columns of its results
    uint8_t* c;
    int64_t ldc;
    bool lines;                    // the rows of c begin where lines of 128 bytes do
    int part;                      // of a tile that is cut, its place in part_ws, else -1
  };
  auto tile_at = [&](int id) __attribute__((always_inline)) {
    Tile t{};
    t.part = -1;
    if (id >= n_wg) return t;  // nothing: its loads bring zeros
    int pid = xcd_order(id, n_wg);
    int part = 0, parts = 1;
    if (tail_parts > 1 && pid >= tail_first) {
      const int qq = pid - tail_first;
      parts = tail_parts;
      part = small_div(qq, n_tail);
      t.part = qq;  // (part by part, the tiles in their order)
      pid = tail_first + qq - part * n_tail;
    }
    const auto& p = list->item[item_of(list, pid)];
    int tile_m, tile_n;
    tile_coords<true>(pid - p.first, p.tiles_m, p.tiles_n, tile_m, tile_n);
    const int m0 = tile_m * kTM, n0 = tile_n * kTN;
    const int all = (p.T + kTK - 1) / kTK, per = small_div(all + parts - 1, parts), s0 = part * per;
    t.slabs = min(per, all - s0);
    t.rows_last = min(p.T - (s0 + t.slabs - 1) * kTK, kTK);
    t.a_row = (int)(p.lda * 2);
    t.b_row = (int)(p.ldb * 2);
    t.a = p.a + (int64_t)s0 * kTK * p.lda + m0;
    t.b = p.b + (int64_t)s0 * kTK * p.ldb + n0;
    t.cols_a = min(p.M - m0, kTM);
    t.cols_b = min(p.N - n0, kTN);
    t.ldc = p.ldc;
    t.c = reinterpret_cast<uint8_t*>(p.c) + ((int64_t)m0 * p.ldc + n0) * kSize;
    t.lines = ((reinterpret_cast<uint64_t>(p.c) | (uint64_t)(p.ldc * kSize)) & 127) == 0;
    return t;
  };

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int q = lane >> 4, r16 = lane & 15;
  const int wm = (wave / kWN) * (kTM / kWM), wn = (wave % kWN) * (kTN / kWN);

  // loads: load j of an operand brings the slab's rows t0 + 2 j, the 32-byte piece p of row t in position p ^ h(t); the lanes'
  // offsets less the immediate of their place in a group of four.  (Columns past the matrix are those of its next row, or
  // past its end and zero: they end in results that are not stored.)
  const int t0 = 2 * wave * kLA + (lane >> 5);
  int col[kLA];
#pragma unroll
  for (int j = 0; j < kLA; ++j) {
    const int t = t0 + 2 * j, pos = lane & 31, h = (t & 3) | (((t >> 3) & 1) << 2);
    col[j] = ((((pos >> 1) ^ h) << 1) | (pos & 1)) * 16 - (j & 3) * 1024;
  }
  static_assert(kLA == kLB && kLA == kTK / 2 / kNW, "both operands alike");
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)smem;
  const uint32_t lds_a = lds0 + wave * kLA * 1024, lds_b = lds0 + kBBase + wave * kLB * 1024;

  // the slab that is loaded: where it begins, bytes to the next one, its size (a last slab's ends with its rows)
  uint64_t at_a = 0, at_b = 0;
  uint32_t step_a = 0, step_b = 0, size_a = 0, size_b = 0;
  int aoff[kLA], boff[kLB];
  auto load_tile = [&](const Tile& t) __attribute__((always_inline)) {
    at_a = reinterpret_cast<uint64_t>(t.a);
    at_b = reinterpret_cast<uint64_t>(t.b);
    step_a = (uint32_t)t.a_row * kTK;
    step_b = (uint32_t)t.b_row * kTK;
    size_a = t.slabs ? (uint32_t)t.a_row * (kTK - 1) + t.cols_a * 2 : 0;
    size_b = t.slabs ? (uint32_t)t.b_row * (kTK - 1) + t.cols_b * 2 : 0;
    const int row_a = t0 * t.a_row, row_b = t0 * t.b_row;
#pragma unroll
    for (int j = 0; j < kLA; ++j) {
      aoff[j] = row_a + 2 * j * t.a_row + col[j];
      boff[j] = row_b + 2 * j * t.b_row + col[j];
    }
  };
  auto load_last = [&](const Tile& t) __attribute__((always_inline)) {
    size_a = (uint32_t)t.a_row * (t.rows_last - 1) + t.cols_a * 2;
    size_b = (uint32_t)t.b_row * (t.rows_last - 1) + t.cols_b * 2;
  };
  uint32_t buf_a = 0, buf_b = 0;
  auto rsrc = [](uint64_t at, uint32_t size) __attribute__((always_inline)) {
    u32x4 r;
    r.x = __builtin_amdgcn_readfirstlane((uint32_t)at);
    r.y = __builtin_amdgcn_readfirstlane((uint32_t)(at >> 32) & 0xffffu);
    r.z = __builtin_amdgcn_readfirstlane(size);
    r.w = 0x00020000u;
    return r;
  };
  auto issue_one = [&](int l) __attribute__((always_inline)) {
    const bool isa = l < kLA;
    const int j = isa ? l : l - kLA;
    const u32x4 res = isa ? rsrc(at_a, size_a) : rsrc(at_b, size_b);
    const int voff = isa ? aoff[j] : boff[j];
    const uint32_t grp = (isa ? lds_a + buf_a : lds_b + buf_b) + (j & ~3) * 1024;
    switch (j & 3) {
      case 0: load_to_lds16<0>(res, grp, voff, 0); break;
      case 1: load_to_lds16<1024>(res, grp, voff, 0); break;
      case 2: load_to_lds16<2048>(res, grp, voff, 0); break;
      default: load_to_lds16<3072>(res, grp, voff, 0); break;
    }
  };
  auto next_slab = [&]() __attribute__((always_inline)) {
    buf_a ^= kABytes;
    buf_b = buf_b == 2 * kBBytes ? 0 : buf_b + kBBytes;
    at_a += step_a;
    at_b += step_b;
  };

  // reads: per fragment, the address in the buffer that is read
  const int lane_off = (8 * q + (r16 >> 2)) * kRow + (((r16 >> 2) | ((q & 1) << 2)) * 32) + 8 * (r16 & 3);
  uint32_t a_rd[kMI], b_rd[kNI], rd_b = 0;
#pragma unroll
  for (int f = 0; f < kMI; ++f) {
    a_rd[f] = lds0 + (lane_off ^ ((wm / 16 + f) * 32));
    b_rd[f] = lds0 + kBBase + (lane_off ^ ((wn / 16 + f) * 32));
    asm volatile("" : "+v"(a_rd[f]), "+v"(b_rd[f]));  // (otherwise the base goes into the constant: see gemm_bf16_tn.hip)
  }
  bf16x8 fa[2][kMI], fb[2][kNI];
  auto read_one = [&](int set, int kk, int f) __attribute__((always_inline)) {
    const uint32_t at = (f < kMI ? a_rd[f < kMI ? f : 0] : b_rd[f < kMI ? 0 : f - kMI]) + kk * 32 * kRow;
    auto tr = [](uint32_t a) __attribute__((always_inline)) {
      return __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) i16x4*)(uintptr_t)a);
    };
    const bf16x8 v = __builtin_bit_cast(bf16x8, (i16x8)__builtin_shufflevector(tr(at), tr(at + 4 * kRow), 0, 1, 2, 3, 4, 5, 6, 7));
    if (f < kMI) fa[set][f] = v;
    else fb[set][f - kMI] = v;
  };
  AccFile acc;  // accumulator j kMI + i: lane = row wm + 16 i + lane % 16 of C, four columns wn + 16 j + 4 (lane / 16)
  acc.claim();
  // One K step: the products on register set `set`; between them the reads of K step rk into the other, the loads [l0, l0 + 8)
  // of a slab and, in the second, the turns of the read addresses to the next buffers.  fresh: the accumulators start here
  auto step = [&](auto fresh, int set, int rk, int l0, uint32_t turn_a, uint32_t turn_b) __attribute__((always_inline)) {
    each<kMI * kNI>([&](auto at) __attribute__((always_inline)) {
      constexpr int idx = decltype(at)::value, j = idx / kMI, i = idx % kMI;
      // (in front of a fragment's read; the first of A's are read behind the second product)
      if constexpr (idx % 2 == 0 && idx / 2 < kMI + kNI) {
        constexpr int f = idx / 2;
        if (set == 1) {
          if constexpr (f < kMI) a_rd[f] += turn_a;
          else b_rd[f - kMI] += turn_b;
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      acc.product<idx, decltype(fresh)::value>(fb[set][j], fa[set][i]);
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (idx % 2 == 1 && idx / 2 < kMI + kNI) {
        read_one(set ^ 1, rk, idx / 2);
        __builtin_amdgcn_sched_barrier(0);
      }
      if constexpr (idx % 8 == 0) {
        static_assert(kMI * kNI / 8 == kLA, "the loads of an operand under one step");
        issue_one(l0 + idx / 8);
        __builtin_amdgcn_sched_barrier(0);
      }
    });
  };
  uint32_t rd_a = 0;
  // behind: vector memory operations of this wave that are younger than the loads of the slab that is waited for
  auto slab = [&](auto fresh, int behind) __attribute__((always_inline)) {
    __builtin_amdgcn_sched_barrier(0);
    step(fresh, 0, 1, kLA, 0, 0);  // under it the loads of B of slab s+2 into the third buffer
    static_assert(kLB == 8 && kMI * kNI / 2 == 32, "the loads of B and the stores of a tile that may be on their way");
    if (behind > 40) asm volatile("s_waitcnt vmcnt(63) lgkmcnt(0)" ::: "memory");
    else if (behind > 8) asm volatile("s_waitcnt vmcnt(40) lgkmcnt(0)" ::: "memory");
    else asm volatile("s_waitcnt vmcnt(8) lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();  // slab s+1 has landed for everybody, the buffers of slab s are free
    const uint32_t turn_b = rd_b == 2 * kBBytes ? 0u - 2 * kBBytes : kBBytes, turn_a = rd_a ? 0u - kABytes : kABytes;
    rd_b += turn_b;
    rd_a += turn_a;
    step(std::false_type{}, 1, 0, 0, turn_a, turn_b);  // under it the loads of A of slab s+2
    next_slab();
  };

  // workgroup w's tile of a round is its w-th, of the last round its w-th from behind: the long tiles come first, and who had one
  // shall not have one of the last, too
  const int whole = n_wg / 256 * 256;
  auto id_in = [&](int round) __attribute__((always_inline)) {
    const int first = round * (int)gridDim.x;
    return first + (first >= whole ? (int)gridDim.x - 1 - (int)blockIdx.x : (int)blockIdx.x);
  };
  Tile cur = tile_at(id_in(0));
  load_tile(cur);
#pragma unroll
  for (int l = 0; l < kL; ++l) issue_one(l);
  next_slab();
#pragma unroll
  for (int l = 0; l < kL; ++l) issue_one(l);
  next_slab();
  static_assert(kL == 16, "the loads of slab 1 may be on their way");
  asm volatile("s_waitcnt vmcnt(16)" ::: "memory");
  __builtin_amdgcn_s_barrier();
#pragma unroll
  for (int f = 0; f < kMI + kNI; ++f) read_one(0, 0, f);

  int behind = kLB;
  for (int round = 1;; ++round) {
    const int id = id_in(round);
    const Tile next = tile_at(id);
    if (cur.slabs == 3) load_last(cur);
    slab(std::true_type{}, behind);
    int s = 1;
    // under slab s the loads of slab s + 2: whole ones, the last, the next tile's first two
    for (int end = cur.slabs - 3;; ++end) {
      for (; s < end; ++s) slab(std::false_type{}, kLB);
      if (end == cur.slabs - 3) {
        load_last(cur);
      } else {
        if (end == cur.slabs) break;
        load_tile(next);
        ++end;
      }
    }
    acc.wait();
    if (cur.part >= 0) {
      float* const P = list->part_ws + ((int64_t)cur.part << 16) + (wm + r16) * kTN + wn + 4 * q;
      each<kMI * kNI>([&](auto at) __attribute__((always_inline)) {
        constexpr int j = decltype(at)::value / kMI, i = decltype(at)::value % kMI;
        *reinterpret_cast<f32x4*>(P + i * 16 * kTN + j * 16) = acc.read<j * kMI + i>();
      });
      behind = kLB + kMI * kNI;
    } else {
      // (rows past the matrix lie outside the resource, lanes of columns past it get an offset that does)
      const int row_step = (int)(cur.ldc * (16 * kSize));
      const u32x4 cres = make_rsrc(cur.c, (uint32_t)((((int64_t)cur.cols_a - 1) * cur.ldc + cur.cols_b) * kSize));
      const bool lo = r16 < 8;
      const int n = wn + (F32 ? (lo ? 0 : 16) + 4 * q : (lo ? 0 : 32) + (q & 1) * 16 + 4 * (q & 2));
      const int at0 = (int)(((int64_t)(wm + (r16 & 7)) * cur.ldc + n) * kSize);
      // blocks of 16 columns that make a whole line of 128 bytes
      constexpr int kLine = F32 ? 2 : 4;
      auto store_all = [&](auto stream) __attribute__((always_inline)) {
        each<kMI * kNI / kLine>([&](auto at) __attribute__((always_inline)) {
          constexpr int i = decltype(at)::value / (kNI / kLine), j = decltype(at)::value % (kNI / kLine) * kLine;
          u32x4 v0, v1, x, y;
          if constexpr (F32) {
            v0 = __builtin_bit_cast(u32x4, acc.read<j * kMI + i>());
            v1 = __builtin_bit_cast(u32x4, acc.read<(j + 1) * kMI + i>());
          } else {
            auto pack8 = [&](auto block) __attribute__((always_inline)) {  // columns 4 (q & 2) + 0..7 of block + (q & 1)
              const f32x4 a = acc.read<decltype(block)::value * kMI + i>(), b = acc.read<(decltype(block)::value + 1) * kMI + i>();
              const auto s0 = __builtin_amdgcn_permlane16_swap(pack_bf16x2(a[0], a[1]), pack_bf16x2(b[0], b[1]), false, false);
              const auto s1 = __builtin_amdgcn_permlane16_swap(pack_bf16x2(a[2], a[3]), pack_bf16x2(b[2], b[3]), false, false);
              u32x4 v;
              v.x = s0[0]; v.y = s1[0]; v.z = s0[1]; v.w = s1[1];
              return v;
            };
            v0 = pack8(std::integral_constant<int, j>{});
            v1 = pack8(std::integral_constant<int, j + 2>{});
          }
          line_pair(lo, v0, v1, x, y);
          const bool in = n + j * 16 < cur.cols_b;
          buffer_store16<j * 16 * kSize, decltype(stream)::value>(cres, in ? at0 + i * row_step : kOob, x);
          buffer_store16<j * 16 * kSize, decltype(stream)::value>(cres, in ? at0 + i * row_step + row_step / 2 : kOob, y);
        });
      };
      if (cur.lines) store_all(std::true_type{});
      else store_all(std::false_type{});
      behind = kLB + 2 * kMI * kNI / kLine;
    }
    if (next.slabs == 0) break;
    cur = next;
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // (loads that bring zeros may still be landing in LDS)
}

// The cut tiles of a list: C[tile] = the sum of its parts, in their order, fp32, one rounding.  A workgroup takes 8 rows of a tile.
template <bool F32>
__global__ __launch_bounds__(256) void gemm_tn_walk_reduce_kernel(List) {
  const ListPtr list = (ListPtr)__builtin_amdgcn_kernarg_segment_ptr();
  const int n_tail = list->n_tiles - list->tail_first;
  const int at = blockIdx.x >> 5, pid = list->tail_first + at;
  const auto& p = list->item[item_of(list, pid)];
  int tile_m, tile_n;
  tile_coords<true>(pid - p.first, p.tiles_m, p.tiles_n, tile_m, tile_n);
  const int rr = ((int)blockIdx.x & 31) * 8 + ((int)threadIdx.x >> 5), cc = ((int)threadIdx.x & 31) * 8;
  const int m = tile_m * kTM + rr, n = tile_n * kTN + cc;
  if (m >= p.M || n >= p.N) return;
  f32x4 lo = {0.f, 0.f, 0.f, 0.f}, hi = lo;
  for (int i = 0; i < list->tail_parts; ++i) {
    const float* const src = list->part_ws + ((int64_t)(i * n_tail + at) << 16) + rr * kTN + cc;
    lo += *reinterpret_cast<const f32x4*>(src);
    hi += *reinterpret_cast<const f32x4*>(src + 4);
  }
  if constexpr (F32) {
    f32x4* const cp = reinterpret_cast<f32x4*>(reinterpret_cast<float*>(p.c) + (int64_t)m * p.ldc + n);
    cp[0] = lo;
    cp[1] = hi;
  } else {
    u32x4 v;
    v.x = pack_bf16x2(lo[0], lo[1]); v.y = pack_bf16x2(lo[2], lo[3]);
    v.z = pack_bf16x2(hi[0], hi[1]); v.w = pack_bf16x2(hi[2], hi[3]);
    *reinterpret_cast<u32x4*>(reinterpret_cast<uint16_t*>(p.c) + (int64_t)m * p.ldc + n) = v;
  }
}

constexpr int kCus = 256;

// us that a tile's results take: 128 or 256 KB, and the fp32 ones of a part
static float results_us(bool f32) { return f32 ? 10.2f : 5.5f; }
constexpr float kPartUs = 8.f;

// us that `wgs` workgroups of `slabs` slabs take, one to a compute unit.  With the above fitted to 687 products of 130 to 9000 rows,
// results of 48 to 3000 tiles (4 % rms; 1164 others 4 %, 1 - 3 % too low)
static float rounds_us(int64_t wgs, int64_t slabs, float results) {
  const int64_t full = wgs / kCus, last = wgs % kCus;
  return full * (slabs * 1.37f + results) + (last ? slabs * (0.86f + 0.37f * last / kCus) + results : 0.f);
}

// Into how many parts the tiles of the last round are cut (at most kMaxParts, each at least 16 slabs, at most `room` partial
// tiles): as many as make it shortest, with the pass that adds them (50 ns a partial tile).  293 last rounds in parts: 1.001 of the
// better of parts and whole tiles.
static int tail_of(int rem, int slabs_least, int slabs_most, bool f32, int64_t room, float& us) {
  int best = 1;
  us = rem ? rounds_us(rem, slabs_most, results_us(f32)) : 0.f;
  for (int p = 2; rem && p <= kMaxParts && slabs_least / p >= 16 && (int64_t)rem * p <= room; ++p) {
    const float t = rounds_us((int64_t)rem * p, (slabs_most + p - 1) / p, kPartUs) + 4.1f + 0.05f * rem * p;
    if (t < 0.97f * us) { us = t; best = p; }
  }
  return best;
}

struct Plan {
  int order[kMaxItems];
  int n_tiles, tail_parts;
  float us;
};

static int64_t tiles_of(int64_t M, int64_t N) { return ((M + kTM - 1) / kTM) * ((N + kTN - 1) / kTN); }

// false: the walking kernel does not take the list
static bool plan(const spx_tn_product* p, int n, bool f32, int64_t room, Plan& out) {
  if (n < 1 || n > kMaxItems) return false;
  int64_t tiles = 0;
  for (int i = 0; i < n; ++i) {
    // (the kernel divides slabs and parts by small_div)
    if (p[i].T <= 2 * kTK || (p[i].T + kTK - 1) / kTK + kMaxParts >= 1 << 22 || p[i].lda < kTM || p[i].ldb < kTN || p[i].ldc % 8 || (uintptr_t)p[i].c % 16 ||
        kTM * p[i].ldc * (f32 ? 4 : 2) >= 0x7ffffff0ll || kTK * p[i].lda * 2 >= 0x7ffffff0ll || kTK * p[i].ldb * 2 >= 0x7ffffff0ll)
      return false;
    tiles += tiles_of(p[i].M, p[i].N);
    out.order[i] = i;
  }
  if (tiles >= (1 << 21)) return false;
  std::stable_sort(out.order, out.order + n, [&](int a, int b) { return p[a].T > p[b].T; });
  out.n_tiles = (int)tiles;
  out.us = 3.f;
  // the whole rounds of the workgroup that has the first tiles of all of them, and of the one that has the last, then the last round
  const int64_t rem = tiles % kCus;
  int64_t at = 0, first = 0, last = kCus - 1;
  float us_first = 0.f, us_last = 0.f;
  int most = 0, least = 0;
  for (int k = 0; k < n; ++k) {
    const auto& e = p[out.order[k]];
    const int slabs = (int)((e.T + kTK - 1) / kTK);
    at += tiles_of(e.M, e.N);
    for (; first < std::min(at, tiles - rem); first += kCus) us_first += rounds_us(kCus, slabs, results_us(f32));
    for (; last < std::min(at, tiles - rem); last += kCus) us_last += rounds_us(kCus, slabs, results_us(f32));
    if (at > tiles - rem) {
      if (!most) most = slabs;
      least = slabs;
    }
  }
  float us_rem = 0.f;
  out.tail_parts = tail_of((int)rem, least, most, f32, room, us_rem);
  out.us += out.tail_parts > 1 ? std::max(us_first, us_last) + us_rem : std::max(us_first, us_last + us_rem);
  return true;
}

}  // namespace tnw
}  // namespace spx

using namespace spx;

// (partial tiles of a last round that is cut: see tail_of)
static constexpr int64_t kTnRoom = 1024;

extern "C" int64_t spx_gemm_tn_list_workspace_bytes(const spx_tn_product* products, int n, int out_f32) {
  tnw::Plan plan;
  if (!products || !tnw::plan(products, n, out_f32 != 0, kTnRoom, plan) || plan.tail_parts == 1) return 0;
  return (int64_t)(plan.n_tiles % tnw::kCus) * plan.tail_parts * kTM * kTN * (int64_t)sizeof(float);
}

extern "C" float spx_gemm_tn_list_us(const spx_tn_product* products, int n, int out_f32) {
  tnw::Plan plan;
  if (!products || !tnw::plan(products, n, out_f32 != 0, kTnRoom, plan)) return -1.f;
  return plan.us;
}

extern "C" int spx_gemm_bf16_tn_list(const spx_tn_product* products, int n, int out_f32, void* workspace,
                                     int64_t workspace_bytes, void* stream) {
  const char* fname = __func__;
  if (!products || n < 1 || n > tnw::kMaxItems) return fail_arg(fname, "1 .. 8 products");
  for (int i = 0; i < n; ++i) {
    const auto& p = products[i];
    if (int rc = tile::tn_check(fname, p.a, p.lda, p.b, p.ldb, p.c, p.ldc, p.M, p.N, std::min<int64_t>(p.T, 1))) return rc;
    if (p.T <= 0 || p.T >= (1ll << 31)) return fail_arg(fname, "T must be positive and below 2^31");
  }
  tnw::Plan plan;
  const bool have = workspace && (uintptr_t)workspace % 16 == 0;
  if (!tnw::plan(products, n, out_f32 != 0,
                 have ? std::min<int64_t>(workspace_bytes / (kTM * kTN * (int64_t)sizeof(float)), kTnRoom) : 0, plan))
    return fail_arg(fname, "contractions of 129 rows and more, leading dimensions of 256 and more, of c multiples of 8");
  tnw::List list{};
  int first = 0;
  for (int k = 0; k < tnw::kMaxItems; ++k) {
    auto& e = list.item[k];
    if (k >= n) {
      e.first = INT32_MAX;
      continue;
    }
    const auto& p = products[plan.order[k]];
    e = {reinterpret_cast<const uint16_t*>(p.a), reinterpret_cast<const uint16_t*>(p.b), p.c, p.lda, p.ldb, p.ldc,
         (int)p.M, (int)p.N, (int)p.T, (int)((p.M + kTM - 1) / kTM), (int)((p.N + kTN - 1) / kTN), first};
    first += e.tiles_m * e.tiles_n;
  }
  list.part_ws = reinterpret_cast<float*>(workspace);
  list.n_tiles = plan.n_tiles;
  list.tail_parts = plan.tail_parts;
  list.tail_first = plan.n_tiles - (plan.tail_parts > 1 ? plan.n_tiles % tnw::kCus : 0);
  const int n_tail = list.n_tiles - list.tail_first, n_wg = list.tail_first + n_tail * list.tail_parts;
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  static std::atomic<uint64_t> lds_set[2];
  const void* const fn = out_f32 ? reinterpret_cast<const void*>(&tnw::gemm_bf16_tn_walk_kernel<true>)
                                 : reinterpret_cast<const void*>(&tnw::gemm_bf16_tn_walk_kernel<false>);
  if (int rc = ensure_dynamic_lds(fn, kGemmSmem, lds_set[out_f32 ? 1 : 0], fname)) return rc;
  const dim3 grid((unsigned)std::min(n_wg, tnw::kCus)), block(kGemmThreads);
  if (out_f32) hipLaunchKernelGGL(tnw::gemm_bf16_tn_walk_kernel<true>, grid, block, kGemmSmem, st, list);
  else hipLaunchKernelGGL(tnw::gemm_bf16_tn_walk_kernel<false>, grid, block, kGemmSmem, st, list);
  if (int rc = check_launch(fname)) return rc;
  if (!n_tail) return SPX_OK;
  if (out_f32) hipLaunchKernelGGL(tnw::gemm_tn_walk_reduce_kernel<true>, dim3((unsigned)(n_tail * 32)), dim3(256), 0, st, list);
  else hipLaunchKernelGGL(tnw::gemm_tn_walk_reduce_kernel<false>, dim3((unsigned)(n_tail * 32)), dim3(256), 0, st, list);
  return check_launch(fname);
}
