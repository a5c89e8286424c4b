// C[M, N] = A[M, K] B[N, K]^T, or (SLOW) A[M, K] B[K, N], by workgroups that walk the tiles, one per compute unit.  Tile, slab buffers,
// order of the loads, reads and products are those of gemm_bf16.hip -- and for SLOW, of the right operand, those of
// gemm_bf16_tn.hip: whole rows of a slab into LDS, fragments by the transposing read.
//
// Workgroup w takes the tiles w, w + grid, ... of the order there.  The slabs of its tiles are one stream: the loads of the next
// tile's first two slabs are issued under the last two of this one, and the results leave while the next tile is multiplied.
// What a tile of its own pays for between its last product and the next tile's first (the stores on their way, a workgroup's
// start, the first loads' latency: 12 us) is here the conversion and issue of the stores and what the burst of all compute
// units' stores holds up: with the stores dropped 32760 x 2048 -> 12288 would take another 12 % less, 4096 x 4096 -> 28672 7 %.
// A workgroup a tile / this, us: 32760 x 2048 -> 12288 1246 / 1130, 1999 x 2048 -> 32000 200 / 187, 4096 x 4096 -> 32000 741 / 715,
// 4096 x 4096 -> 28672 660 / 623, 4096 x 14336 -> 4096 (one round) 303 / 300, 512 x 2048 -> 32000 (one round) 53.7 / 51.0; in a
// 1B validation pass 3294 / 3208, an MTP step 171.6 / 169.8 ms.
// The results leave in whole 128-byte lines, past the caches (STREAM) where they are larger than the 256 MB cache behind them (walk).
#pragma once

#include "acc_file.h"
#include "gemm_nt.h"

namespace spx {

constexpr int kSlowRow = kTN * 2;  // SLOW: bytes of a row of a slab of B
static_assert(kTK * kSlowRow == kBBytes && kTK / 2 / kNW == kLB, "a slab is as large either way");

// silu(g) u of eight pairs, the bits of swiglu_fwd_kernel.  1 / (1 + e^-g) by the reciprocal instruction and one step of Newton's, whose
// residue is exact, in the place of a division's ten instructions; of a quarter of the sum (the reciprocal of a sum above 2^126 would
// be flushed to zero), and of an infinite sum it is nothing, with or without the step.
__device__ __forceinline__ u32x4 swiglu8(u32x4 g, u32x4 u) {
  auto silu = [](float gv) __attribute__((always_inline)) {
    const float quarter = gv * 0.25f, e = fast_exp2(quarter * (-4.f * 1.44269504f));
    const float sum = fmaf(e, 0.25f, 0.25f), r = __builtin_amdgcn_rcpf(sum);
    return quarter * fmaf(r, fmaf(-fminf(sum, 0x1p127f), r, 1.f), r);
  };
  u32x4 o;
#pragma unroll
  for (int w = 0; w < 4; ++w) {
    const uint32_t s = pack_bf16x2(silu(bf16_lo(g[w])), silu(bf16_hi(g[w])));
    o[w] = pack_bf16x2(bf16_lo(s) * bf16_lo(u[w]), bf16_hi(s) * bf16_hi(u[w]));
  }
  return o;
}

typedef short i16x4 __attribute__((ext_vector_type(4)));
typedef short i16x8 __attribute__((ext_vector_type(8)));

// K: a multiple of 64, at least 192 (and every part of a cut contraction); N and ldc multiples of 8, C 16-byte aligned; SLOW: N a
// multiple of 256.  m_live, part_ws, max_parts, cus, tail_mode, grade: see gemm_bf16_nt_kernel.  parts > 1: all tiles are cut into
// so many (tail_mode 0), which leave fp32 results in part_ws, [parts][M][N].
// B2 (else null): the second half of B's rows -- its first `half` rows are at B, the others at B2, both ldb apart.  A tile of the
// plain form lies in one of them (half % 256 == 0); SLOW: the loads turn to B2 with the slab that starts there (half % 64 == 0),
// which is never the second or third of a tile or of a part of one.  (Asked for at every slab instead of where it comes, the turn
// cost all products of that form 0.5 - 1.4 %.)
// GATE: a gated MLP's first product.  B is the gate's weight, B2 that of the up projection, `half` rows each (a multiple of 256); a
// tile is 128 columns of each, in every wave 64 and the same 64, so that a lane holds what belongs together: `act` =
// swiglu8(gate, up) from the two results as they are rounded (bf16 [M, half], ld_act apart), which leave too where GATE is 2 (in
// C, the gate's columns and behind them the up projection's).  A cut tile's parts lie as its columns do.  Product and SwiGLU launch / this,
// us (of the launch, bound by its traffic, the activation's arithmetic remains, 3.1 us a round of tiles that nothing runs beside): 1999 x
// 2048 -> 2 x 8192 without the two results 110 / 95, 888 rows with them 60.3 / 54.5, 4096 x 4096 -> 2 x 14336 683 (the product the
// library's) / 636, 8192 rows 1358 / 1265, 3001 rows (64 tiles in four parts) 525 / 501.
// (SPX_WALK_KERNEL: the kernel's name, for each source that has forms of it; one body for all -- as a function that kernels call it
// got other registers and ran 1 % longer)
template <bool SLOW, bool GRADE, bool STREAM, int GATE = 0>
__global__ __launch_bounds__(kGemmThreads, SPX_GEMM_MINW)
__attribute__((amdgpu_waves_per_eu(SPX_GEMM_MINW, SPX_GEMM_MINW))) void SPX_WALK_KERNEL(
    const uint16_t* __restrict__ A, int64_t lda, const uint16_t* __restrict__ B, const uint16_t* __restrict__ B2, int half,
    int64_t ldb, uint16_t* __restrict__ C, int64_t ldc, int M, int N, int K, int tiles_m, int tiles_n,
    const int32_t* __restrict__ m_live, float* __restrict__ part_ws, int max_parts, int cus, int tail_mode,
    int parts, RowGrade grade, uint16_t* __restrict__ act, int64_t ld_act) {
  static_assert(!GATE || (!SLOW && !GRADE), "the plain form");
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  const int M_host = M;
  if (m_live) {
    M = min(M, max(*m_live, 0));
    tiles_m = (M + kTM - 1) / kTM;
  }
  const int n_tiles = tiles_m * tiles_n, all_slabs = K / kTK;
  int tail_first = n_tiles, tail_parts = 1;
  if (GRADE && tail_mode) live_tail_plan(n_tiles, cus, all_slabs, max_parts, tail_mode, tail_first, tail_parts);
  else if (tail_mode) tail_plan(n_tiles, cus, all_slabs, max_parts, tail_first, tail_parts);
  if (parts > 1) {
    tail_first = 0;
    tail_parts = parts;
  }
  const int n_tail = n_tiles - tail_first;
  const int n_wg = n_tiles + n_tail * (tail_parts - 1);
  if ((int)blockIdx.x >= n_wg) return;

  struct Tile {
    int m0, n0, slabs, part;  // part: of a tile that is cut, its place in part_ws, else -1
    u32x4 ares, bres;
    int turn;  // SLOW: slabs until B2
  };
  auto tile_at = [&](int id) __attribute__((always_inline)) {
    Tile t;
    if (id >= n_wg) {  // nothing: its loads bring zeros
      t.m0 = t.n0 = t.slabs = 0;
      t.part = -1;
      t.turn = 0x7fffffff;
      t.ares = make_rsrc(A, 0);
      t.bres = make_rsrc(B, 0);
      return t;
    }
    int pid = xcd_order(id, n_wg);
    int k0 = 0;
    t.slabs = all_slabs;
    t.part = -1;
    if (tail_parts > 1 && pid >= tail_first) {
      const int qq = pid - tail_first, part = small_div(qq, n_tail);
      const int per = (all_slabs + tail_parts - 1) / tail_parts;
      t.part = parts > 1 ? part : qq;  // (part by part, the tiles in their order)
      pid = tail_first + qq - part * n_tail;
      k0 = part * per * kTK;
      t.slabs = min(per, all_slabs - part * per);
    }
    int tile_m, tile_n;
    tile_coords<true>(pid, tiles_m, tiles_n, tile_m, tile_n);
    t.m0 = tile_m * kTM;
    t.n0 = tile_n * kTN;
    // (rows past the matrix lie outside the resource: they are lda, ldb >= K apart)
    t.ares = make_rsrc(A + (int64_t)t.m0 * lda + k0, (uint32_t)((((int64_t)min(M - t.m0, kTM) - 1) * lda + K - k0) * 2));
    if constexpr (GATE) {  // (this wave's 64 rows)
      const int w = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
      t.bres = make_rsrc((w & 1 ? B2 : B) + (int64_t)(t.n0 / 2 + w / 2 * 64) * ldb + k0, (uint32_t)((63 * ldb + K - k0) * 2));
      t.turn = 0x7fffffff;
      return t;
    }
    const int at = SLOW ? k0 : t.n0;  // the first row of B
    const bool second = B2 && at >= half;
    const uint16_t* const rows = second ? B2 + (int64_t)(at - half) * ldb : B + (int64_t)at * ldb;
    t.turn = !SLOW || !B2 || second ? 0x7fffffff : (half - k0) / kTK;
    if (SLOW)
      t.bres = make_rsrc(rows + t.n0, (uint32_t)((((int64_t)(B2 && !second ? half : K) - k0 - 1) * ldb + kTN) * 2));
    else
      t.bres = make_rsrc(rows + k0, (uint32_t)((((int64_t)min(N - t.n0, kTN) - 1) * ldb + K - k0) * 2));
    return t;
  };

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int q = lane >> 4, r16 = lane & 15;
  const int wm = (wave / kWN) * (kTM / kWM), wn = (wave % kWN) * (kTN / kWN);

  // loads: the lanes' offsets, less the immediate of their place in a group of four
  int aoff[kLA], boff[kLB];
  static_assert(kLA == kLB, "both operands alike");
#pragma unroll
  for (int j = 0; j < kLA; ++j) {
    const int imm = (j & 3) * 1024;
    const int r = wave * (8 * kLA) + j * 8 + (lane >> 3), chunk = (lane & 7) ^ ((lane >> 3) & 7) ^ (j & 1);
    aoff[j] = (int)(((int64_t)r * lda + chunk * 8) * 2) - imm;
    if (SLOW) {
      const int t = 2 * (wave * kLB + j) + (lane >> 5), pos = lane & 31, h = (t & 3) | (((t >> 3) & 1) << 2);
      boff[j] = (int)(((int64_t)t * ldb + ((((pos >> 1) ^ h) << 1) | (pos & 1)) * 8) * 2) - imm;
    } else if (GATE) {
      boff[j] = (int)(((int64_t)(j * 8 + (lane >> 3)) * ldb + chunk * 8) * 2) - imm;
    } else {
      boff[j] = (int)(((int64_t)r * ldb + chunk * 8) * 2) - imm;
    }
  }
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)smem;
  const uint32_t lds_a = lds0 + wave * kLA * 1024, lds_b = lds0 + kBBase + wave * kLB * 1024;

  Tile cur = tile_at(blockIdx.x);
  u32x4 ares = cur.ares, bres = cur.bres;  // of the slab being loaded
  uint32_t buf_a = 0, buf_b = 0;
  int at_a = 0, at_b = 0;  // bytes to it from the tile's first
  const int slab_b = SLOW ? (int)(ldb * (2 * kTK)) : 2 * kTK;
  auto issue_one = [&](int l) __attribute__((always_inline)) {
    const bool isa = l < kLA;
    const int j = isa ? l : l - kLA;
    const u32x4 res = isa ? ares : bres;
    const int voff = isa ? aoff[j] : boff[j], soff = isa ? at_a : at_b;
    const uint32_t grp = (isa ? lds_a + buf_a : lds_b + buf_b) + (j & ~3) * 1024;
    switch (j & 3) {
      case 0: load_to_lds16<0>(res, grp, voff, soff); break;
      case 1: load_to_lds16<1024>(res, grp, voff, soff); break;
      case 2: load_to_lds16<2048>(res, grp, voff, soff); break;
      default: load_to_lds16<3072>(res, grp, voff, soff); break;
    }
  };
  auto next_slab = [&]() __attribute__((always_inline)) {
    buf_a ^= kABytes;
    buf_b = buf_b == 2 * kBBytes ? 0 : buf_b + kBBytes;
    at_a += 2 * kTK;
    at_b += slab_b;
  };

  // reads: per K step of A (and of B, if that is not SLOW: then per fragment), the address in the buffer that is read
  const int off0 = r16 * kRowBytes + ((q ^ (r16 & 7) ^ (r16 >> 3)) * 16);
  constexpr int kRb = SLOW ? kNI : kKSteps;
  uint32_t a_rd[kKSteps], b_rd[kRb], rd_b = 0;
#pragma unroll
  for (int kk = 0; kk < kKSteps; ++kk) a_rd[kk] = lds0 + wm * kRowBytes + (off0 ^ (kk * 64));
#pragma unroll
  for (int f = 0; f < kRb; ++f) {
    if (SLOW) {
      const int lane_off = (8 * q + (r16 >> 2)) * kSlowRow + (((r16 >> 2) | ((q & 1) << 2)) * 32) + 8 * (r16 & 3);
      b_rd[f] = lds0 + kBBase + (lane_off ^ ((wn / 16 + f) * 32));
    } else {
      b_rd[f] = lds0 + kBBase + wn * kRowBytes + (off0 ^ (f * 64));
    }
    asm volatile("" : "+v"(b_rd[f]));  // (otherwise the base goes into the constant, which no longer fits the offset field)
  }
  bf16x8 fa[2][kMI], fb[2][kNI];
  // operand fragment f (A's first) of K step kk into register set `set`
  auto read_one = [&](int set, int kk, int f) __attribute__((always_inline)) {
    if (f < kMI) {
      fa[set][f] = as_frag(lds_read128(a_rd[kk] + f * 16 * kRowBytes));
    } else if (SLOW) {
      const uint32_t at = b_rd[f - kMI] + kk * 32 * kSlowRow;
      auto tr = [](uint32_t a) __attribute__((always_inline)) {
        return __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) i16x4*)(uintptr_t)a);
      };
      const i16x8 v = __builtin_shufflevector(tr(at), tr(at + 4 * kSlowRow), 0, 1, 2, 3, 4, 5, 6, 7);
      fb[set][f - kMI] = __builtin_bit_cast(bf16x8, v);
    } else {
      fb[set][f - kMI] = as_frag(lds_read128(b_rd[SLOW ? 0 : kk] + (f - kMI) * 16 * kRowBytes));
    }
  };
  AccFile acc;  // accumulator j kMI + i: lane = row wm + 16 i + lane % 16 of C, four columns wn + 16 j + 4 (lane / 16)
  acc.claim();
  static_assert(kMI * kNI == 64, "the accumulators of an AccFile");
  // One K step: the products on register set `set`; between them the reads of K step rk into the other, the loads [l0, l0 + 8)
  // of a slab and the turn of B's read addresses to the next buffer.  fresh: the accumulators start here
  auto step = [&](auto fresh, int set, int rk, int l0, uint32_t turn) __attribute__((always_inline)) {
    each<kMI * kNI>([&](auto at) __attribute__((always_inline)) {
      constexpr int idx = decltype(at)::value, j = idx / kMI, i = idx % kMI;
      acc.product<idx, decltype(fresh)::value>(fb[set][j], fa[set][i]);
      __builtin_amdgcn_sched_barrier(0);
      constexpr int every = SPX_GEMM_READ_EVERY;
      if constexpr (idx % every == every - 1 && idx / every < kMI + kNI) {
        read_one(set ^ 1, rk, idx / every);
        __builtin_amdgcn_sched_barrier(0);
      }
      if constexpr (idx % SPX_GEMM_LOAD_EVERY == SPX_GEMM_LOAD_AT) {
        static_assert(kMI * kNI / SPX_GEMM_LOAD_EVERY == kLA, "the loads of an operand under one step");
        issue_one(l0 + idx / SPX_GEMM_LOAD_EVERY);
        __builtin_amdgcn_sched_barrier(0);
      }
      // (in front of the first read of B, behind the eighth)
      if constexpr (idx % 2 == 0 && idx / 2 < kRb) {
        if (set == 1) b_rd[idx / 2] += turn;
        __builtin_amdgcn_sched_barrier(0);
      }
    });
  };
  // behind: vector memory operations of this wave that are younger than the loads of the slab that is waited for
  auto slab = [&](auto fresh, int behind) __attribute__((always_inline)) {
    __builtin_amdgcn_sched_barrier(0);
    // K step 0 of slab s, under it the loads of B of slab s+2 into the third buffer
    step(fresh, 0, 1, kLA, 0);
    static_assert(kLB == 8 && kMI * kNI / 2 == 32, "the loads of B and the stores of a tile that may be on their way");
    if constexpr (GATE) {
      if (behind > 56) asm volatile("s_waitcnt vmcnt(63) lgkmcnt(0)" ::: "memory");
      else if (behind > 8) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(kLB + (GATE == 1 ? 16 : 48)) : "memory");
      else asm volatile("s_waitcnt vmcnt(8) lgkmcnt(0)" ::: "memory");
    } else if (behind > 40) asm volatile("s_waitcnt vmcnt(63) lgkmcnt(0)" ::: "memory");
    else if (behind > 8) asm volatile("s_waitcnt vmcnt(40) lgkmcnt(0)" ::: "memory");
    else asm volatile("s_waitcnt vmcnt(8) lgkmcnt(0)" ::: "memory");
    // slab s+1 has landed for everybody, the buffers of slab s are free
    __builtin_amdgcn_s_barrier();
    const uint32_t turn = rd_b == 2 * kBBytes ? 0u - 2 * kBBytes : kBBytes;
    rd_b += turn;
#pragma unroll
    for (int kk = 0; kk < kKSteps; ++kk) a_rd[kk] ^= kABytes;
    // K step 1 of slab s, under it the reads of slab s+1 and the loads of A of slab s+2
    step(std::false_type{}, 1, 0, 0, turn);
    next_slab();
  };

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
  for (int id = blockIdx.x;;) {
    id += gridDim.x;
    const Tile next = tile_at(id);
    slab(std::true_type{}, behind);
    int s = 1;
    for (int end = (SLOW && cur.turn < cur.slabs ? cur.turn : cur.slabs) - 2;;) {  // (the loads are two slabs ahead)
      for (; s < end; ++s) slab(std::false_type{}, kLB);
      if (end == cur.slabs) break;
      if (SLOW && end != cur.slabs - 2) {
        bres = make_rsrc(B2 + cur.n0, (uint32_t)((((int64_t)K - half - 1) * ldb + kTN) * 2));
        at_b = 0;
        end = cur.slabs - 2;
        continue;
      }
      end = cur.slabs;
      ares = next.ares;
      bres = next.bres;
      at_a = at_b = 0;
    }
    acc.wait();
    if (GATE && cur.part < 0) {
      // (rows past the matrix lie outside the resources)
      const int rows = min(M - cur.m0, kTM), c0 = cur.n0 / 2;
      const u32x4 ares_out = make_rsrc(act + (int64_t)cur.m0 * ld_act + c0, (uint32_t)((((int64_t)rows - 1) * ld_act + kTN / 2) * 2));
      const u32x4 cres = make_rsrc(C + (int64_t)cur.m0 * ldc + c0,
                                   GATE == 2 ? (uint32_t)((((int64_t)rows - 1) * ldc + half + kTN / 2) * 2) : 0u);
      const bool lo = r16 < 8;
      const int n = wn / 2 + (lo ? 0 : 32) + (q & 1) * 16 + 4 * (q & 2), row = wm + (r16 & 7);
      const int at_act = (int)(((int64_t)row * ld_act + n) * 2), at_c = (int)(((int64_t)row * ldc + n) * 2);
      const int act_step = (int)(ld_act * 16), c_step = (int)(ldc * 16);  // eight rows
      each<kMI>([&](auto at) __attribute__((always_inline)) {
        constexpr int i = decltype(at)::value;
        auto pack8 = [&](auto block) __attribute__((always_inline)) {
          const f32x4 a = acc.read<decltype(block)::value * kMI + i>(), b = acc.read<(decltype(block)::value + 1) * kMI + i>();
          const auto s0 = __builtin_amdgcn_permlane16_swap(pack_bf16x2(a[0], a[1]), pack_bf16x2(b[0], b[1]), false, false);
          const auto s1 = __builtin_amdgcn_permlane16_swap(pack_bf16x2(a[2], a[3]), pack_bf16x2(b[2], b[3]), false, false);
          u32x4 v;
          v.x = s0[0]; v.y = s1[0]; v.z = s0[1]; v.w = s1[1];
          return v;
        };
        using std::integral_constant;
        u32x4 gx, gy, ux, uy;
        line_pair(lo, pack8(integral_constant<int, 0>{}), pack8(integral_constant<int, 2>{}), gx, gy);
        line_pair(lo, pack8(integral_constant<int, 4>{}), pack8(integral_constant<int, 6>{}), ux, uy);
        if constexpr (GATE == 2) {
          buffer_store16<0, STREAM>(cres, at_c + 2 * i * c_step, gx);
          buffer_store16<0, STREAM>(cres, at_c + (2 * i + 1) * c_step, gy);
          buffer_store16<0, STREAM>(cres, at_c + 2 * i * c_step + half * 2, ux);
          buffer_store16<0, STREAM>(cres, at_c + (2 * i + 1) * c_step + half * 2, uy);
        }
        buffer_store16<0, false>(ares_out, at_act + 2 * i * act_step, swiglu8(gx, ux));
        buffer_store16<0, false>(ares_out, at_act + (2 * i + 1) * act_step, swiglu8(gy, uy));
      });
      behind = kLB + (GATE == 1 ? 16 : 48);
    } else if (cur.part >= 0 && parts > 1) {
      // this part's fp32 results, in whole lines (rows and columns past the matrix as below)
      const int cols = min(N - cur.n0, kTN), row_step = N * 64;
      const u32x4 pres = make_rsrc(part_ws + ((int64_t)cur.part * M_host + cur.m0) * N + cur.n0,
                                   (uint32_t)((((int64_t)min(M - cur.m0, kTM) - 1) * N + cols) * 4));
      const bool lo = r16 < 8;
      const int n = wn + (lo ? 0 : 16) + 4 * q;
      const int at0 = (int)(((int64_t)(wm + (r16 & 7)) * N + n) * 4);
      each<kMI * kNI / 2>([&](auto at) __attribute__((always_inline)) {
        constexpr int i = decltype(at)::value / (kNI / 2), j = decltype(at)::value % (kNI / 2) * 2;
        u32x4 x, y;
        const u32x4 v0 = __builtin_bit_cast(u32x4, acc.read<j * kMI + i>());
        const u32x4 v1 = __builtin_bit_cast(u32x4, acc.read<(j + 1) * kMI + i>());
        line_pair(lo, v0, v1, x, y);
        const bool in = n + j * 16 < cols;
        buffer_store16<j * 64, false>(pres, in ? at0 + i * row_step : kOob, x);
        buffer_store16<j * 64, false>(pres, in ? at0 + i * row_step + row_step / 2 : kOob, y);
      });
      behind = kLB + kMI * kNI;
    } else if (cur.part >= 0) {
      // this part's fp32 partial of a tile of the last round: a 256 x 256 tile of its own
      float* const P = part_ws + ((int64_t)cur.part << 16) + (wm + r16) * kTN + wn + 4 * q;
      each<kMI * kNI>([&](auto at) __attribute__((always_inline)) {
        constexpr int j = decltype(at)::value / kMI, i = decltype(at)::value % kMI;
        *reinterpret_cast<f32x4*>(P + i * 16 * kTN + j * 16) = acc.read<j * kMI + i>();
      });
      behind = kLB + kMI * kNI;
    } else {
      // (rows past the matrix lie outside the resource, lanes of columns past it get an offset that does)
      const int cols = min(N - cur.n0, kTN), row_step = (int)(ldc * 32);
      const u32x4 cres = make_rsrc(C + (int64_t)cur.m0 * ldc + cur.n0,
                                   (uint32_t)((((int64_t)min(M - cur.m0, kTM) - 1) * ldc + cols) * 2));
      const bool lo = r16 < 8;
      const int n = wn + (lo ? 0 : 32) + (q & 1) * 16 + 4 * (q & 2);
      const int at0 = (int)(((int64_t)(wm + (r16 & 7)) * ldc + n) * 2);
      float by[kMI];
      if constexpr (GRADE) {
#pragma unroll
        for (int i = 0; i < kMI; ++i) {
          const int m = cur.m0 + wm + i * 16 + r16;
          by[i] = m < M ? grade.at(m) : 0.f;
        }
      }
      each<kMI * kNI / 4>([&](auto at) __attribute__((always_inline)) {
        constexpr int i = decltype(at)::value / (kNI / 4), j = decltype(at)::value % (kNI / 4) * 4;
        auto pack8 = [&](auto block) __attribute__((always_inline)) {  // columns 4 (q & 2) + 0..7 of block + (q & 1)
          f32x4 a = acc.read<decltype(block)::value * kMI + i>(), b = acc.read<(decltype(block)::value + 1) * kMI + i>();
          if constexpr (GRADE) { a *= by[i]; b *= by[i]; }
          const auto s0 = __builtin_amdgcn_permlane16_swap(pack_bf16x2(a[0], a[1]), pack_bf16x2(b[0], b[1]), false, false);
          const auto s1 = __builtin_amdgcn_permlane16_swap(pack_bf16x2(a[2], a[3]), pack_bf16x2(b[2], b[3]), false, false);
          u32x4 v;
          v.x = s0[0]; v.y = s1[0]; v.z = s0[1]; v.w = s1[1];
          return v;
        };
        u32x4 x, y;
        const u32x4 v0 = pack8(std::integral_constant<int, j>{}), v1 = pack8(std::integral_constant<int, j + 2>{});
        line_pair(lo, v0, v1, x, y);
        const bool in = n + j * 16 < cols;
        buffer_store16<j * 32, STREAM>(cres, in ? at0 + i * row_step : kOob, x);
        buffer_store16<j * 32, STREAM>(cres, in ? at0 + i * row_step + row_step / 2 : kOob, y);
      });
      behind = kLB + kMI * kNI / 2;
    }
    if (id >= n_wg) break;
    cur = next;
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // (loads that bring zeros may still be landing in LDS)
}

}  // namespace spx
