// Host side of the tile GEMM kernels (gemm_tile.h): which tile a product gets, and the grouped forms.
//
// The 256 x 256 kernels of gemm_bf16.hip / gemm_bf16_tn.hip are built for products of many tiles with a long
// contraction.  A group of a grouped product is often neither: 512 experts x 80 rows each are 512 ragged row bands,
// and their weight gradient contracts over 80 rows.  Measured there (4096 tokens, top 10 of 512 experts, gate/up
// 2048 -> 1024; 2.1 GB of weights, 430 us at the rate of a copy):
//   forward          256 x 256, 4 waves 573 us -> 128 x 256, 8 waves, 3 slabs 498 -> whole lines past the caches 460
//   input gradient   595 us + 786 us to transpose the weights -> 446 on the weights as they lie (NN form) -> one slab, two
//                    workgroups a compute unit 435
//   weight gradient  bf16, 4 waves 760 us -> 8 waves 696 (1067 us with the fp32 result it replaces) -> 128 x 128, one slab,
//                    four workgroups a compute unit, whole lines past the caches 605 (467 with its operands in the
//                    memory-side cache: what bounds it is waiting for them; each workgroup fetching its share of the
//                    operands 1024 workgroups ahead made it 716)

#include <algorithm>

#include "gemm_tile.h"
#include "gemm_tile_api.h"
#include "../../include/spx.h"

using namespace spx;

namespace spx {
namespace tile {

// tab[0] = number of tile rows of tm rows, then (group, first row) of every tile row: group e contributes
// ceil(rows_e / tm) of them.  One workgroup; thread t owns a contiguous run of groups.
__global__ __launch_bounds__(256) void group_tiles_kernel(const int32_t* __restrict__ group_off, int groups, int rows,
                                                          int tm, int max_tiles, int32_t* __restrict__ tab) {
  __shared__ int sums[256];
  const int t = threadIdx.x;
  const int per = (groups + 255) / 256;
  const int e0 = min(t * per, groups), e1 = min(e0 + per, groups);
  // (offsets are clamped to [0, rows]: the table is sized for that many rows whatever they hold)
  auto clamped = [&](int e) { return min(max(group_off[e], 0), rows); };
  int mine = 0;
  for (int e = e0; e < e1; ++e) mine += (max(clamped(e + 1) - clamped(e), 0) + tm - 1) / tm;
  sums[t] = mine;
  __syncthreads();
  // inclusive prefix sum over the 256 threads
  for (int d = 1; d < 256; d <<= 1) {
    const int v = t >= d ? sums[t - d] : 0;
    __syncthreads();
    sums[t] += v;
    __syncthreads();
  }
  if (t == 255) tab[0] = min(sums[255], max_tiles);  // (offsets that do not ascend could ask for more than that)
  int at = sums[t] - mine;
  for (int e = e0; e < e1; ++e) {
    const int r0 = clamped(e), r1 = clamped(e + 1);
    for (int r = r0; r < r1; r += tm, ++at) {
      if (at >= max_tiles) break;
      tab[1 + 2 * at] = e;
      tab[2 + 2 * at] = r;
    }
  }
}

constexpr int kCus = 256;
constexpr int kPickRows = 256;  // rows a group on average up to which the grouped products take their rows picked

template <int TM, int TN, int WM, int WN, int STAGES, int MINB, bool AT, bool BT, int OUT, bool STREAM, bool GRADE = false,
          int PICK = 0>
static int launch(const char* fname, Params p, int groups_y, hipStream_t st) {
  constexpr int kSmem = (TM * STAGES + TN * ring_b(STAGES)) * kTK * 2;
  static_assert(kSmem * (4 * MINB / (WM * WN)) <= 160 * 1024, "LDS for the workgroups that a compute unit shall hold");
  static std::atomic<uint64_t> lds_set;
  auto* const kernel = &gemm_tile_kernel<TM, TN, WM, WN, STAGES, MINB, AT, BT, OUT, STREAM, GRADE, PICK>;
  if (int rc = ensure_dynamic_lds(reinterpret_cast<const void*>(kernel), kSmem, lds_set, fname)) return rc;
  hipLaunchKernelGGL((gemm_tile_kernel<TM, TN, WM, WN, STAGES, MINB, AT, BT, OUT, STREAM, GRADE, PICK>),
                     dim3((unsigned)std::max(p.tiles_m * p.tiles_n * p.parts, p.cut.max_parts ? p.cut.cap : 0), (unsigned)groups_y),
                     dim3(64 * WM * WN), kSmem,
                     st, p);
  return check_launch(fname);
}

#define SPX_REQ_FN(cond, what) do { if (!(cond)) return spx::fail_arg(fname, what); } while (0)

static int64_t table_entries(int64_t rows, int64_t groups, int tm) { return (rows + tm - 1) / tm + groups; }

// Grouped product over the rows of A: c[r, :] = a[r, :] b_e^T (BT = false, b_e [N, K]) or a[r, :] b_e (BT = true,
// b_e [K, N]).  src: where the rows of A lie in a matrix of src_rows (null: in order); table_ready: the workspace holds the
// table of tile rows already.
template <bool BT>
static int grouped_rows(const char* fname, const void* a, int64_t lda, const void* b, int64_t ldb,
                        int64_t b_group_stride, void* c, int64_t ldc, int64_t rows, int64_t N, int64_t K,
                        const int32_t* group_off, int64_t groups, void* workspace, hipStream_t st,
                        const int32_t* src = nullptr, int64_t src_rows = 0, bool table_ready = false) {
  // Rows a group on average: above 256 the taller tile reads the group's weights half as often (64 groups of 1024 rows,
  // K 2048 -> N 1536, 768 -> 2048: NT 413 -> 404 us, 254 -> 240; of 4096: 1568 -> 1385, 978 -> 876; of 256, 512 groups:
  // 1054 -> 1084, 634 -> 641; NN 220 -> 220, 457 -> 425; of 256: 550 -> 584, 1095 -> 1095).
  const bool wide_m = rows > kPickRows * groups;
  const int tm = wide_m ? 256 : 128;
  const int64_t max_tiles = table_entries(rows, groups, tm), tiles_n = (N + 255) / 256;
  SPX_REQ_FN(max_tiles * tiles_n < (1ll << 31), "too many tiles");
  int32_t* const tab = reinterpret_cast<int32_t*>(workspace);
  if (!table_ready) {
    hipLaunchKernelGGL(group_tiles_kernel, dim3(1), dim3(256), 0, st, group_off, (int)groups, (int)rows, tm,
                       (int)max_tiles, tab);
    if (int rc = check_launch(fname)) return rc;
  }
  Params p{};
  p.A = reinterpret_cast<const uint16_t*>(a);
  p.B = reinterpret_cast<const uint16_t*>(b);
  p.C = c;
  p.lda = lda; p.ldb = ldb; p.ldc = ldc;
  p.M = (int)rows; p.N = (int)N; p.K = (int)K;
  p.tiles_m = (int)max_tiles; p.tiles_n = (int)tiles_n; p.parts = 1;
  p.tile_tab = tab; p.group_off = group_off; p.group_stride = b_group_stride;
  p.src = src; p.src_rows = (int)src_rows;
  if (wide_m) return launch<256, 256, 2, 4, 2, 2, false, BT, 0, true>(fname, p, 1, st);
  // A short contraction is mostly start and end of a tile: two workgroups with one slab each cover them, three slabs of
  // one workgroup do not -- where there are tiles for two (512 groups of 80 rows: K 512 -> N 2048 NT 247 -> 236 us, K 1024
  // -> 2048 NN 430 -> 409; 64 groups of 88 rows: 34 -> 35, 57 -> 66; K 2048: 432 / 431 NT, 234 -> 245 NN)
  const bool short_k = K <= 1024 && groups * tiles_n >= 4 * kCus;
  if (src)
    return short_k ? launch<128, 256, 2, 4, 1, 4, false, BT, 0, true, false, 1>(fname, p, 1, st)
                   : launch<128, 256, 2, 4, 3, 2, false, BT, 0, true, false, 1>(fname, p, 1, st);
  return short_k ? launch<128, 256, 2, 4, 1, 4, false, BT, 0, true>(fname, p, 1, st)
                 : launch<128, 256, 2, 4, 3, 2, false, BT, 0, true>(fname, p, 1, st);
}

int grouped_nt(const char* fname, const void* a, int64_t lda, const void* b, int64_t ldb, int64_t b_group_stride,
               void* c, int64_t ldc, int64_t rows, int64_t N, int64_t K, const int32_t* group_off, int64_t groups,
               void* workspace, void* stream) {
  SPX_REQ_FN(rows > 0 && N > 0 && K > 0, "rows, N, K must be positive");
  SPX_REQ_FN(rows < (1ll << 31) && N < (1ll << 31) && K < (1ll << 31), "dimension too large");
  SPX_REQ_FN(a && b && c, "null buffer");
  SPX_REQ_FN(K % 8 == 0 && lda % 8 == 0 && ldb % 8 == 0, "K, lda, ldb must be multiples of 8");
  SPX_REQ_FN(lda >= K && ldb >= K && ldc >= N, "leading dimension too small");
  SPX_REQ_FN(((uintptr_t)a | (uintptr_t)b) % 16 == 0, "a and b must be 16-byte aligned");
  SPX_REQ_FN((256 * lda + K) * 2 < 0x7ffffff0ll && (256 * ldb + K) * 2 < 0x7ffffff0ll,
             "256 rows of an operand must span less than 2 GiB (32-bit offsets inside a tile)");
  return grouped_rows<false>(fname, a, lda, b, ldb, b_group_stride, c, ldc, rows, N, K, group_off, groups, workspace,
                             reinterpret_cast<hipStream_t>(stream));
}

template <int TM, int TN, int WM, int WN, int STAGES, int MINB, int PICK = 0>
static int launch_tn_tile(const char* fname, Params p, int64_t groups, int out, hipStream_t st) {
  p.tiles_m = (p.M + TM - 1) / TM;
  p.tiles_n = (p.N + TN - 1) / TN;
  switch (out) {
    case 0: return launch<TM, TN, WM, WN, STAGES, MINB, true, true, 0, true, false, PICK>(fname, p, (int)groups, st);
    case 1: return launch<TM, TN, WM, WN, STAGES, MINB, true, true, 1, false, false, PICK>(fname, p, (int)groups, st);
    case 2: return launch<TM, TN, WM, WN, STAGES, MINB, true, true, 2, true, false, PICK>(fname, p, (int)groups, st);
    default: return launch<TM, TN, WM, WN, STAGES, MINB, true, true, 3, false, false, PICK>(fname, p, (int)groups, st);
  }
}

int grouped_tn(const char* fname, const void* a, int64_t lda, const void* b, int64_t ldb, void* c, int64_t ldc,
               int64_t c_group_stride, int64_t M, int64_t N, int64_t rows, const int32_t* group_off, int64_t groups,
               int out_f32, int accumulate, void* stream, const int32_t* src, int64_t src_rows, int operand) {
  Params p{};
  p.A = reinterpret_cast<const uint16_t*>(a);
  p.B = reinterpret_cast<const uint16_t*>(b);
  p.C = c;
  p.lda = lda; p.ldb = ldb; p.ldc = ldc;
  p.M = (int)M; p.N = (int)N; p.K = (int)rows;
  p.parts = 1;
  p.group_off = group_off; p.group_stride = c_group_stride;
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  const int out = (out_f32 ? 2 : 0) + (accumulate ? 1 : 0);
  // Up to 512 rows a group the store of a tile takes longer than its products: small workgroups that overlap one
  // another.  (1024, 2048 results; 256 x 256 with whole lines / 128 x 128: 512 groups of 10 rows 460 / 350 us, of 80
  // 546 / 467, of 256 (1536 columns) 1428 / 1356; 64 groups of 1024 rows 439 / 440 and, 2048 x 768, 250 / 269; of 2048
  // rows 522 / 752.)
  if (src) {
    p.src = src;
    p.src_rows = (int)src_rows;
    return operand ? launch_tn_tile<128, 128, 2, 2, 1, 4, 2>(fname, p, groups, out, st)
                   : launch_tn_tile<128, 128, 2, 2, 1, 4, 1>(fname, p, groups, out, st);
  }
  return rows <= 512 * groups ? launch_tn_tile<128, 128, 2, 2, 1, 4>(fname, p, groups, out, st)
                              : launch_tn_tile<256, 256, 2, 4, 2, 2>(fname, p, groups, out, st);
}

// ------------------------------------------------------------------------------------------ plain products
// C[m, n .. n + 7] = the sum of the parts of a product whose contraction was cut, in their order, fp32, one rounding.
// OUT as in gemm_tile_kernel; grade (OUT 0): what the rows of the sum are multiplied by; cut: the parts were chosen on the
// device, for tiles of tm x tn (one part: the product has stored its results).
template <int OUT>
__global__ __launch_bounds__(256) void parts_reduce_kernel(const float* __restrict__ ws, void* __restrict__ C,
                                                           int64_t ldc, int M_host, int N, int parts,
                                                           const int32_t* __restrict__ m_live, RowGrade grade,
                                                           LiveCut cut, int tm, int tn) {
  const int M = m_live ? min(M_host, max(*m_live, 0)) : M_host;
  if (OUT == 0 && cut.max_parts) {
    const int tiles_m = (M + tm - 1) / tm;
    parts = cut.parts(tiles_m * ((N + tn - 1) / tn), (int64_t)M * N);
    if (parts == 1) return;
    M_host = tiles_m * tm;
  }
  const int n8 = N / 8;
  const int64_t item = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (item >= (int64_t)M * n8) return;
  const int m = (int)(item / n8), n = (int)(item % n8) * 8;
  f32x4 lo = {0.f, 0.f, 0.f, 0.f}, hi = lo;
  for (int p = 0; p < parts; ++p) {
    const float* src = ws + ((int64_t)p * M_host + m) * N + n;
    lo += *reinterpret_cast<const f32x4*>(src);
    hi += *reinterpret_cast<const f32x4*>(src + 4);
  }
  if (OUT == 0 && grade.row) {
    const float by = grade.at(m);
    lo *= by;
    hi *= by;
  }
  if constexpr (OUT >= 2) {
    f32x4* const cp = reinterpret_cast<f32x4*>(reinterpret_cast<float*>(C) + (int64_t)m * ldc + n);
    if (OUT == 3) { lo += cp[0]; hi += cp[1]; }
    cp[0] = lo;
    cp[1] = hi;
  } else {
    u32x4* const cp = reinterpret_cast<u32x4*>(reinterpret_cast<uint16_t*>(C) + (int64_t)m * ldc + n);
    if (OUT == 1) {
      const u32x4 old = *cp;
      lo += f32x4{bf16_lo(old.x), bf16_hi(old.x), bf16_lo(old.y), bf16_hi(old.y)};
      hi += f32x4{bf16_lo(old.z), bf16_hi(old.z), bf16_lo(old.w), bf16_hi(old.w)};
    }
    u32x4 v;
    v.x = pack_bf16x2(lo[0], lo[1]); v.y = pack_bf16x2(lo[2], lo[3]);
    v.z = pack_bf16x2(hi[0], hi[1]); v.w = pack_bf16x2(hi[2], hi[3]);
    *cp = v;
  }
}

template <int OUT>
static int launch_reduce(const char* fname, const float* ws, void* c, int64_t ldc, int64_t M, int64_t N, int parts,
                         const int32_t* m_live, hipStream_t st, const RowGrade& grade = RowGrade{},
                         const LiveCut& cut = LiveCut{}, int tm = 1, int tn = 1) {
  const int64_t items = M * (N / 8);
  hipLaunchKernelGGL(parts_reduce_kernel<OUT>, dim3((unsigned)((items + 255) / 256)), dim3(256), 0, st, ws, c, ldc, (int)M,
                     (int)N, parts, m_live, grade, cut, tm, tn);
  return check_launch(fname);
}

// The tile a product gets.  Every candidate's time is predicted and the shortest taken:
//   rounds of workgroups x (slabs of a part x (s0 + s1 x filled share of the chip) + b)  [us], plus for a contraction
//   in parts the pass that adds them, 4.1 + 1.03 per million fp32 partials.
// s0, s1, b fitted to 180 products (M 256 .. 4096, the projections and heads of the 1B, 8B and 70B drafts and their
// input gradients, 14 configurations each; 5 - 15 % rms).  On those products the choice is within 1.2 % of the best
// candidate in the geometric mean and 1.33 x the 256 x 256 kernel alone (512 x 6144 -> 2048: 45.4 -> 23 us; 360 live
// rows x 32000 -> 2048: 177 -> 62; 2000 x 4096 -> 4096: 71 -> 57; 4096-row products keep the large tile).
// The tiles of 192 rows are for the row counts whose 256-row tiles fill the chip badly -- 2817 .. 3072 rows to 4096 columns
// are 192 tiles of 256 x 256 and exactly 256 of 192 x 256 -- fitted to 99 products of 512 .. 5000 rows (3.5 - 6 % rms).
// Where they are taken, 101 products of 700 .. 5000 rows run in 0.92 of the choice without them (geometric mean, both forms
// alike; the worst 1.04, 700 x 2048 -> 16384): a b^T 1300 x 8192 -> 6144 184 -> 115 us, 1700 x 5120 -> 5120 115 -> 75,
// 2900 x 4096 -> 3072 87 -> 63, 3001 x 14336 -> 4096 301 -> 283; a b 1300 x 14336 -> 4096 164 -> 144, 2300 x 4096 -> 4096
// 90 -> 80, 3001 x 28672 -> 4096 604 -> 556, 5000 x 8192 -> 2048 170 -> 155.
// The walking kernels (gemm_bf16_walk.hip) and the tiles of three slab buffers of B, fitted again to 136 products of 256 .. 8192 rows
// (3.6 - 7 % rms): within 0.4 % of the best candidate.  a b, tiles cut whole on the walking kernel, the choice before / now: 1400 x
// 16384 -> 2048 89 -> 81 us, 3500 rows 186 -> 169, 888 x 28672 -> 4096 186 -> 164, 1100 238 -> 210.
// (Tiles of 128 x 192 and 256 x 192 are the choice for too few further products, and the slow operand of the second form
// takes whole powers of two only.)
enum Tile { kBig = 0, k128x128, k256x128, k64x128, k192x256, kFifth /* NT: 192 x 192, NN: 256 x 256 */, k192x128 /* NN */ };
struct Config {
  int tm, tn, per_cu;
  float s0, s1, b;
};
constexpr Config kNT[] = {{256, 256, 1, 0.69f, 0.63f, 6.2f},   // kBig: gemm_bf16_walk.hip, its last round cut (tail_plan)
                          {128, 128, 1, 0.35f, 0.14f, 4.1f},
                          {256, 128, 1, 0.52f, 0.25f, 5.3f},
                          {64, 128, 2, 0.18f, 0.42f, 3.0f},
                          {192, 256, 1, 0.72f, 0.35f, 6.2f},
                          {192, 192, 1, 0.53f, 0.28f, 6.0f}};
// (form 2, rows counted on the device: the large tile as live_tail_plan prices it)
constexpr Config kLive = {256, 256, 1, 1.18f, 0.23f, 6.9f};
constexpr Config kNN[] = {{256, 256, 1, 0.f, 0.f, 0.f},        // (kFifth)
                          {128, 128, 1, 0.32f, 0.15f, 3.1f},
                          {256, 128, 1, 0.55f, 0.25f, 4.8f},
                          {64, 128, 2, 0.23f, 0.37f, 2.1f},
                          {192, 256, 1, 0.76f, 0.35f, 5.1f},
                          {256, 256, 1, 0.78f, 0.47f, 7.4f},   // gemm_bf16_walk.hip
                          {192, 128, 1, 0.45f, 0.18f, 4.3f}};
// kFifth of the second form where N is no multiple of 256: those workgroups do not walk (walk_takes), and the 256 x 256 tile by eight
// waves takes 6 % longer than the price above.  5 % rms over 40 products of 512 .. 8192 rows -> 896 .. 5000 columns; chosen
// with it / with the price above, us: 1400 x 8192 -> 4160 92.0 / 96.2, 700 x 11520 -> 2880 54.3 / 57.0, 8192 x 4096 -> 2880 167.0 /
// 172.7, the other 37 alike: 1.009 of the best candidate in place of 1.013 in the geometric mean.  (Contractions that end
// inside a slab do not walk either, but there all candidates of this form take as much longer: 30 products are within 1.01 of the
// best as they are priced.)
constexpr Config kNNAside = {256, 256, 1, 0.96f, 0.30f, 7.6f};
// kBig of the first form where no workgroup walks: contractions that end inside a slab or have fewer than three, columns that are no
// multiple of 8.  A workgroup a tile then pays for the start and the end of each.  316 such products of 200 to 12000 rows, contractions
// of 64 to 16000: the choice takes 0.974 of that by the walking kernel's price, 0.929 of that before there was one (by more than 3 %
// slower than that 4, the worst 1.09), and is within 1.023 of the best candidate in place of 1.050.  8288 x 808 -> 2944 62.7 -> 51.3
// us, 2048 x 1336 -> 17784 113 -> 99.
constexpr Config kNTAside = {256, 256, 1, 0.90f, 0.30f, 15.f};
// Weight gradients (contraction slow in both operands): the candidates beside the 256 x 256 kernel of gemm_bf16_tn.hip,
// which keeps whole rounds of its tiles and is given up only for a predicted tenth.  Fitted the same way to 128 products
// (results of 1 .. 768 large tiles, 256 .. 20000 rows, up to 12 parts; 6 - 13 % rms).  Over them the choice takes 0.52 of that
// kernel alone and is within 2.6 % of the best candidate (geometric means; one at 1.03 of it): 2048 x 2048 over 888 rows 29
// -> 14 us, over 1536 40 -> 21; 3072 x 2048 over 1536 41 -> 27; 2048 x 10240 over 1777 97 -> 84; 1024 x 2048 over 2665, in
// two bands of 256 x 256 tiles and a sum before, 49 -> 19; 512 x 512 over 5000 95 -> 15.
constexpr Config kTN[] = {{256, 256, 1, 0.97f, 0.50f, 13.9f},
                          {128, 128, 1, 0.29f, 0.23f, 4.5f},   // 8 waves, 4 slabs
                          {256, 128, 1, 0.50f, 0.34f, 6.8f},
                          {64, 128, 2, 0.22f, 0.42f, 3.4f},
                          {128, 128, 2, 0.40f, 0.57f, 4.2f}};  // 4 waves, 2 slabs: two workgroups a compute unit
constexpr int kTnParts = 32;
constexpr int kMinSlabs = 6, kMaxParts = 12, kSplitFrom = 32;  // (no cut below 32 slabs)

struct Choice {
  int tile, parts;
  float us;
};

// us of the pass that adds the parts of `partials` fp32 results in all
static float reduce_us(float partials) { return 4.1f + 1.03e-6f * partials; }

static float predict(const Config& c, int64_t tiles, int slabs) {
  const int64_t cap = (int64_t)kCus * c.per_cu, full = tiles / cap, rem = tiles % cap;
  float t = full * ((c.s0 + c.s1) * slabs + c.b);
  if (rem) t += (c.s0 + c.s1 * (float)rem / (float)cap) * slabs + c.b;
  return t;
}

// (form 2: b a^T with the count of rows on the device.  No tiles of 192 rows there: the 256 x 256 kernel cuts its contraction
// by the rows that count, which the host does not know -- 3001 rows x 32000 -> 4096, two thirds of them counting: 516 us
// in parts, 661 on 192 x 256 tiles.)
static Choice choose(int form, int64_t M, int64_t N, int64_t K, int max_parts, bool can_split) {
  const int slabs = (int)((K + kTK - 1) / kTK);
  const bool nn = form == 1;
  const Config* const table = nn ? kNN : kNT;
  Choice best{kBig, 1, 1e30f};
  if (!nn) {
    const Config& c = form == 2 ? kLive : K % kTK || K < 3 * kTK || N % 8 ? kNTAside : table[kBig];
    const int64_t tiles = ((M + 255) / 256) * ((N + 255) / 256), rem = tiles % kCus;
    int64_t cut = 0;
    int tp = 1;
    if (max_parts > 1 && rem && rem * 2 <= kCus) {
      tp = (int)std::min<int64_t>(kCus / rem, max_parts);
      while (tp > 1 && slabs / tp < 16) --tp;
      cut = tp > 1 ? rem : 0;
    }
    best.us = predict(c, tiles - cut, slabs);
    if (cut) best.us += predict(c, cut * tp, (slabs + tp - 1) / tp) + reduce_us((float)(cut * tp * 65536));
  }
  for (int t = 1; t < (nn ? 7 : form == 2 ? (int)k192x256 : 6); ++t) {
    const Config& c = nn && t == kFifth && N % 256 ? kNNAside : table[t];
    const int64_t tiles = ((M + c.tm - 1) / c.tm) * ((N + c.tn - 1) / c.tn);
    const int64_t cap = (int64_t)kCus * c.per_cu;
    for (int parts = 1; parts <= kMaxParts; ++parts) {
      // a cut fills a round that is not full, and only that
      if (parts > 1 && (!can_split || max_parts <= 1 || slabs < kSplitFrom || slabs / parts < kMinSlabs ||
                        tiles * parts > cap))
        break;
      float us = predict(c, tiles * parts, (slabs + parts - 1) / parts);
      if (parts > 1) us += reduce_us((float)(parts * M * N));
      if (us < best.us) best = Choice{t, parts, us};
    }
  }
  return best;
}

// The most that the parts of a product cut on the device (LiveCut) leave behind, in floats; 0: it is not cut there.
static int64_t live_cut_floats(const Config& c, int64_t M, int64_t N, int64_t K, int max_parts) {
  if (max_parts <= 1 || (K + kTK - 1) / kTK < kSplitFrom) return 0;
  const int64_t tiles_n = (N + c.tn - 1) / c.tn, rows = (M + c.tm - 1) / c.tm * c.tm;
  if (tiles_n * 2 > kCus * c.per_cu) return 0;
  return std::min<int64_t>((int64_t)kCus * c.per_cu * c.tm * c.tn, kMaxParts * rows * N);
}

static LiveCut live_cut(const Config& c, int64_t K) {
  const int slabs = (int)((K + kTK - 1) / kTK);
  return {std::min(kMaxParts, slabs / kMinSlabs), kCus * c.per_cu, slabs, (int)(c.s0 * 1000.f + 0.5f), (int)(c.s1 * 1000.f + 0.5f)};
}

static Choice choose_tn(int64_t M, int64_t N, int64_t T, bool can_split) {
  const int slabs = (int)((T + kTK - 1) / kTK);
  const int64_t big = ((M + 255) / 256) * ((N + 255) / 256);
  Choice best{kBig, 1, predict(kTN[kBig], big, slabs) / 1.1f};
  if (big % kCus == 0) return best;
  for (int t = 1; t < 5; ++t) {
    const Config& c = kTN[t];
    const int64_t tiles = ((M + c.tm - 1) / c.tm) * ((N + c.tn - 1) / c.tn);
    for (int parts = 1; parts <= kTnParts; ++parts) {
      if (parts > 1 && (!can_split || slabs / parts < kMinSlabs || tiles * parts > (int64_t)kCus * c.per_cu)) break;
      float us = predict(c, tiles * parts, (slabs + parts - 1) / parts);
      if (parts > 1) us += reduce_us((float)(parts * M * N));
      if (us < best.us) best = Choice{t, parts, us};
    }
  }
  return best;
}

template <int OUT>
static int launch_tn_dense(const char* fname, int tile, const Params& p, hipStream_t st) {
  switch (tile) {
    case 1: return launch<128, 128, 2, 4, 4, 2, true, true, OUT, false>(fname, p, 1, st);
    case 2: return launch<256, 128, 4, 2, 3, 2, true, true, OUT, false>(fname, p, 1, st);
    case 3: return launch<64, 128, 2, 2, 3, 2, true, true, OUT, false>(fname, p, 1, st);
    default: return launch<128, 128, 2, 2, 2, 2, true, true, OUT, false>(fname, p, 1, st);
  }
}

static int dense_check(const char* fname, int form, const void* a, int64_t lda, const void* b, int64_t ldb,
                       const void* c, int64_t ldc, int64_t M, int64_t N, int64_t K) {
  SPX_REQ_FN(form == 0 || form == 1, "form must be 0 (a b^T) or 1 (a b)");
  SPX_REQ_FN(M > 0 && N > 0 && K > 0, "M, N, K must be positive");
  SPX_REQ_FN(M < (1ll << 31) && N < (1ll << 31) && K < (1ll << 31), "dimension too large");
  SPX_REQ_FN(a && b && c, "null buffer");
  SPX_REQ_FN(K % 8 == 0 && lda % 8 == 0 && ldb % 8 == 0, "K, lda, ldb must be multiples of 8");
  SPX_REQ_FN(lda >= K && ldb >= (form ? N : K) && ldc >= N, "leading dimension too small");
  SPX_REQ_FN(((uintptr_t)a | (uintptr_t)b) % 16 == 0, "a and b must be 16-byte aligned");
  SPX_REQ_FN((256 * lda + K) * 2 < 0x7ffffff0ll, "256 rows of a must span less than 2 GiB (32-bit offsets)");
  if (form == 0)
    SPX_REQ_FN((256 * ldb + K) * 2 < 0x7ffffff0ll, "256 rows of b must span less than 2 GiB (32-bit offsets)");
  else
    SPX_REQ_FN(N % 8 == 0 && (K + 4 * kTK) * ldb * 2 < 0x7ffffff0ll,
               "N must be a multiple of 8 and b span less than 2 GiB (32-bit offsets)");
  return SPX_OK;
}

template <bool BT>
static int launch_dense(const char* fname, int tile, const Params& p, hipStream_t st) {
  switch (tile) {
    case k128x128: return launch<128, 128, 2, 4, 4, 2, false, BT, 0, false>(fname, p, 1, st);
    case k256x128: return launch<256, 128, 4, 2, 3, 2, false, BT, 0, false>(fname, p, 1, st);
    case k64x128: return launch<64, 128, 2, 2, 3, 2, false, BT, 0, false>(fname, p, 1, st);
    case k192x256: return launch<192, 256, 2, 4, 2, 2, false, BT, 0, false>(fname, p, 1, st);
    default:
      if constexpr (!BT) return launch<192, 192, 4, 2, 3, 2, false, false, 0, false>(fname, p, 1, st);
      if (tile == k192x128) return launch<192, 128, 2, 4, 4, 2, false, BT, 0, false>(fname, p, 1, st);
      return launch<256, 256, 2, 4, 2, 2, false, BT, 0, false>(fname, p, 1, st);
  }
}

// (the tiles of form 2)
static int launch_graded(const char* fname, int tile, const Params& p, hipStream_t st) {
  switch (tile) {
    case k128x128: return launch<128, 128, 2, 4, 4, 2, false, false, 0, false, true>(fname, p, 1, st);
    case k256x128: return launch<256, 128, 4, 2, 3, 2, false, false, 0, false, true>(fname, p, 1, st);
    default: return launch<64, 128, 2, 2, 3, 2, false, false, 0, false, true>(fname, p, 1, st);
  }
}

}  // namespace tile
}  // namespace spx

extern "C" int64_t spx_gemm_grouped_workspace_bytes(int64_t rows, int64_t groups) {
  if (rows < 0 || groups < 0) return 0;
  return (int64_t)sizeof(int32_t) * (1 + 2 * tile::table_entries(rows, groups, 128));
}

extern "C" int spx_gemm_bf16_nn_grouped(const void* a, int64_t lda, const void* b, int64_t ldb,
                                        int64_t b_group_stride, void* c, int64_t ldc, int64_t rows, int64_t N,
                                        int64_t K, const int32_t* group_offsets, int64_t groups, void* workspace,
                                        int64_t workspace_bytes, void* stream) {
  const char* fname = __func__;
  SPX_REQ_FN(rows > 0 && N > 0 && K > 0, "rows, N, K must be positive");
  SPX_REQ_FN(rows < (1ll << 31) && N < (1ll << 31) && K < (1ll << 31), "dimension too large");
  SPX_REQ_FN(a && b && c, "null buffer");
  SPX_REQ_FN(groups > 0 && groups < (1 << 24), "groups must be positive");
  SPX_REQ_FN(group_offsets && workspace, "null group offsets or workspace");
  SPX_REQ_FN(workspace_bytes >= spx_gemm_grouped_workspace_bytes(rows, groups), "workspace too small");
  SPX_REQ_FN(((uintptr_t)workspace) % 4 == 0 && b_group_stride % 8 == 0 && b_group_stride >= 0,
             "unaligned workspace or group stride");
  SPX_REQ_FN(K % 8 == 0 && N % 8 == 0 && lda % 8 == 0 && ldb % 8 == 0, "K, N, lda, ldb must be multiples of 8");
  SPX_REQ_FN(lda >= K && ldb >= N && ldc >= N, "leading dimension too small");
  SPX_REQ_FN(((uintptr_t)a | (uintptr_t)b) % 16 == 0, "a and b must be 16-byte aligned");
  SPX_REQ_FN((256 * lda + K) * 2 < 0x7ffffff0ll && (K + 4 * tile::kTK) * ldb * 2 < 0x7ffffff0ll,
             "256 rows of a and one group of b must span less than 2 GiB (32-bit offsets)");
  return tile::grouped_rows<true>(fname, a, lda, b, ldb, b_group_stride, c, ldc, rows, N, K, group_offsets, groups,
                                  workspace, reinterpret_cast<hipStream_t>(stream));
}

extern "C" int spx_gemm_bf16_grouped_picked(int form, const void* a, int64_t lda, const int32_t* src_row,
                                            int64_t src_rows, const void* b, int64_t ldb, int64_t b_group_stride, void* c,
                                            int64_t ldc, int64_t rows, int64_t N, int64_t K, const int32_t* group_offsets,
                                            int64_t groups, void* table, int64_t table_bytes, int table_ready,
                                            void* stream) {
  const char* fname = __func__;
  SPX_REQ_FN(form == 0 || form == 1, "form must be 0 (a b^T) or 1 (a b)");
  SPX_REQ_FN(rows > 0 && N > 0 && K > 0, "rows, N, K must be positive");
  SPX_REQ_FN(rows < (1ll << 31) && N < (1ll << 31) && K < (1ll << 31), "dimension too large");
  SPX_REQ_FN(a && b && c, "null buffer");
  SPX_REQ_FN(groups > 0 && groups < (1 << 24) && rows <= tile::kPickRows * groups, "up to 256 rows a group on average");
  SPX_REQ_FN(group_offsets && table, "null group offsets or table");
  SPX_REQ_FN(table_bytes >= spx_gemm_grouped_workspace_bytes(rows, groups), "table too small");
  SPX_REQ_FN(((uintptr_t)table) % 4 == 0 && b_group_stride % 8 == 0 && b_group_stride >= 0,
             "unaligned table or group stride");
  SPX_REQ_FN(K % 8 == 0 && lda % 8 == 0 && ldb % 8 == 0 && (!form || N % 8 == 0),
             "K, lda, ldb (and N of a b) must be multiples of 8");
  SPX_REQ_FN(lda >= K && ldb >= (form ? N : K) && ldc >= N, "leading dimension too small");
  SPX_REQ_FN(((uintptr_t)a | (uintptr_t)b) % 16 == 0, "a and b must be 16-byte aligned");
  SPX_REQ_FN((256 * lda + K) * 2 < 0x7ffffff0ll && (form ? (K + 4 * tile::kTK) * ldb : 256 * ldb + K) * 2 < 0x7ffffff0ll,
             "256 rows of a and of one group of b must span less than 2 GiB (32-bit offsets)");
  SPX_REQ_FN(!src_row || (src_rows > 0 && src_rows * lda * 2 < 0x7ffffff0ll),
             "the matrix that rows are picked from must have rows and span less than 2 GiB (32-bit offsets)");
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  return form ? tile::grouped_rows<true>(fname, a, lda, b, ldb, b_group_stride, c, ldc, rows, N, K, group_offsets, groups, table,
                                         st, src_row, src_rows, table_ready != 0)
              : tile::grouped_rows<false>(fname, a, lda, b, ldb, b_group_stride, c, ldc, rows, N, K, group_offsets, groups, table,
                                          st, src_row, src_rows, table_ready != 0);
}

extern "C" int spx_gemm_bf16_tn_grouped_picked(const void* a, int64_t lda, const void* b, int64_t ldb, const int32_t* src_row,
                                               int64_t src_rows, int operand, void* c, int64_t ldc, int64_t c_group_stride,
                                               int64_t M, int64_t N, int64_t rows, const int32_t* group_offsets,
                                               int64_t groups, int out_f32, int accumulate, void* stream) {
  const char* fname = __func__;
  if (int rc = tile::tn_check(fname, a, lda, b, ldb, c, ldc, M, N, rows)) return rc;
  SPX_REQ_FN(group_offsets && groups > 0 && groups < 65536, "null group offsets or a group count outside 1 .. 65535");
  SPX_REQ_FN(c_group_stride >= (M - 1) * ldc + N, "groups of c overlap");
  SPX_REQ_FN(c_group_stride % (out_f32 ? 4 : 8) == 0, "the groups of c must be 16-byte aligned among each other");
  SPX_REQ_FN(rows <= tile::kPickRows * groups, "up to 256 rows a group on average");
  SPX_REQ_FN(operand == 0 || operand == 1, "operand must be 0 (a) or 1 (b)");
  SPX_REQ_FN(src_row && src_rows > 0 && src_rows * (operand ? ldb : lda) * 2 < 0x7ffffff0ll,
             "the matrix that rows are picked from must have rows and span less than 2 GiB (32-bit offsets)");
  return tile::grouped_tn(fname, a, lda, b, ldb, c, ldc, c_group_stride, M, N, rows, group_offsets, groups, out_f32, accumulate,
                          stream, src_row, src_rows, operand);
}

// whether the contraction of a product may be cut: the partials are stored in groups of four columns
static bool can_split(int64_t N) { return N % 8 == 0; }

extern "C" int64_t spx_gemm_auto_workspace_bytes(int form, int64_t M, int64_t N, int64_t K, int32_t max_parts) {
  if (M <= 0 || N <= 0 || K <= 0 || max_parts < 1) return 0;
  const tile::Choice c = tile::choose(form, M, N, K, max_parts, can_split(N));
  if (c.tile == tile::kBig) return max_parts > 1 ? spx_gemm_tail_workspace_bytes() : 0;
  const int64_t cut = form == 2 && can_split(N) ? tile::live_cut_floats(tile::kNT[c.tile], M, N, K, max_parts) : 0;
  return std::max(c.parts > 1 ? c.parts * M * N : 0, cut) * (int64_t)sizeof(float);
}

extern "C" float spx_gemm_auto_us(int form, int64_t M, int64_t N, int64_t K, int32_t max_parts) {
  if (M <= 0 || N <= 0 || K <= 0 || max_parts < 1) return 0.f;
  return tile::choose(form, M, N, K, max_parts, can_split(N)).us;
}

extern "C" int spx_gemm_auto_tile(int form, int64_t M, int64_t N, int64_t K, int32_t max_parts) {
  if (M <= 0 || N <= 0 || K <= 0 || max_parts < 1) return 0;
  return tile::choose(form, M, N, K, max_parts, can_split(N)).tile;
}

// left: where the number of partial results goes that are left in the workspace (NULL: they are added here)
static int auto_product(const char* fname, int form, const void* a, int64_t lda, const void* b, int64_t ldb, void* c,
                        int64_t ldc, int64_t M, int64_t N, int64_t K, const int32_t* m_live, int32_t max_parts,
                        void* workspace, int64_t workspace_bytes, int32_t* left, void* stream, const void* b2 = nullptr) {
  if (left) *left = 1;
  SPX_REQ_FN(max_parts >= 1 && max_parts <= 8, "max_parts must be 1 .. 8");
  if (int rc = tile::dense_check(fname, form, a, lda, b, ldb, c, ldc, M, N, K)) return rc;
  const bool vec = ldc % 8 == 0 && ((uintptr_t)c) % 16 == 0;  // (what the pass that adds the parts stores)
  const tile::Choice ch = tile::choose(form == 0 && m_live ? 2 : form, M, N, K, max_parts, can_split(N) && vec && workspace);
  if (ch.tile == tile::kBig) {
    if (m_live) return spx_gemm_bf16_nt_rows(a, lda, b, ldb, c, ldc, M, N, K, m_live, stream);
    if (max_parts > 1 && workspace && workspace_bytes >= spx_gemm_tail_workspace_bytes())
      return spx_gemm_bf16_nt_tail(a, lda, b, ldb, c, ldc, M, N, K, max_parts, workspace, workspace_bytes, stream);
    return spx_gemm_bf16_nt(a, lda, b, ldb, c, ldc, M, N, K, stream);
  }
  SPX_REQ_FN(ch.parts == 1 || (workspace_bytes >= (int64_t)ch.parts * M * N * (int64_t)sizeof(float) &&
                               ((uintptr_t)workspace) % 16 == 0),
             "workspace too small or unaligned");
  const tile::Config& cfg = (form ? tile::kNN : tile::kNT)[ch.tile];
  tile::Params p{};
  p.A = reinterpret_cast<const uint16_t*>(a);
  p.B = reinterpret_cast<const uint16_t*>(b);
  p.C = c;
  p.lda = lda; p.ldb = ldb; p.ldc = ldc;
  p.M = (int)M; p.N = (int)N; p.K = (int)K;
  const int64_t tiles_m = (M + cfg.tm - 1) / cfg.tm, tiles_n = (N + cfg.tn - 1) / cfg.tn;
  SPX_REQ_FN(tiles_m * tiles_n * ch.parts < (1ll << 31), "too many tiles");
  p.tiles_m = (int)tiles_m; p.tiles_n = (int)tiles_n; p.parts = ch.parts;
  p.part_ws = reinterpret_cast<float*>(workspace);
  p.m_live = m_live;
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  const int64_t wgs = tiles_m * tiles_n * ch.parts;
  if (form && ch.tile == tile::kFifth && walk_takes(true, c, ldb, ldc, N, K, wgs, ch.parts)) {
    const WalkArgs w = {p.A, lda, p.B, ldb, reinterpret_cast<uint16_t*>(c), ldc, M, N, K, m_live, p.part_ws, 1, 0, tile::kCus,
                        wgs, RowGrade{}, ch.parts, reinterpret_cast<const uint16_t*>(b2)};
    if (int rc = walk(fname, true, w, st)) return rc;
  } else {
    SPX_REQ_FN(!b2, "a second half of b: sizes that workgroups walk");
    if (int rc = form ? tile::launch_dense<true>(fname, ch.tile, p, st) : tile::launch_dense<false>(fname, ch.tile, p, st)) return rc;
  }
  if (ch.parts == 1) return SPX_OK;
  if (left) {
    *left = ch.parts;
    return SPX_OK;
  }
  return tile::launch_reduce<0>(fname, p.part_ws, c, ldc, M, N, ch.parts, m_live, st);
}

extern "C" int spx_gemm_bf16_auto(int form, const void* a, int64_t lda, const void* b, int64_t ldb, void* c,
                                  int64_t ldc, int64_t M, int64_t N, int64_t K, const int32_t* m_live,
                                  int32_t max_parts, void* workspace, int64_t workspace_bytes, void* stream) {
  return auto_product(__func__, form, a, lda, b, ldb, c, ldc, M, N, K, m_live, max_parts, workspace, workspace_bytes, nullptr,
                      stream);
}

extern "C" int spx_gemm_bf16_auto_parts(int form, const void* a, int64_t lda, const void* b, int64_t ldb, void* c,
                                        int64_t ldc, int64_t M, int64_t N, int64_t K, int32_t max_parts, void* workspace,
                                        int64_t workspace_bytes, int32_t* parts, void* stream) {
  const char* fname = __func__;
  SPX_REQ_FN(parts, "null buffer");
  return auto_product(fname, form, a, lda, b, ldb, c, ldc, M, N, K, nullptr, max_parts, workspace, workspace_bytes, parts,
                      stream);
}

extern "C" int spx_gemm_pair_takes(int form, int64_t M, int64_t N, int64_t K, int64_t ldb, int32_t max_parts) {
  if ((form != 0 && form != 1) || M <= 0 || N <= 0 || K <= 0 || ldb < (form ? N : K) || ldb % 8 || max_parts < 1 || max_parts > 8) return 0;
  const int64_t half = (form ? K : N) / 2;
  if (half * 2 != (form ? K : N) || half % (form ? 64 : 256)) return 0;
  const tile::Choice ch = tile::choose(form, M, N, K, max_parts, can_split(N));
  const int64_t tiles = (M + 255) / 256 * ((N + 255) / 256);
  if (ch.tile != (form ? tile::kFifth : tile::kBig)) return 0;
  if (form) {  // (a part's first two slabs lie in the same half: they are requested before its tile is turned to)
    const int64_t slabs = K / 64, per = (slabs + ch.parts - 1) / ch.parts, before = slabs / 2 % per;
    if (before == 1 || before == 2) return 0;
  }
  return walk_takes(form == 1, nullptr, ldb, N, N, K, tiles + (form ? tiles * (ch.parts - 1) : 8 * tile::kCus), form ? ch.parts : 1);
}

extern "C" int spx_gemm_bf16_pair(int form, const void* a, int64_t lda, const void* b, const void* b2, int64_t ldb, void* c, int64_t ldc,
                                  int64_t M, int64_t N, int64_t K, int32_t max_parts, void* workspace, int64_t workspace_bytes,
                                  int32_t* parts, void* stream) {
  const char* fname = __func__;
  if (parts) *parts = 1;
  if (int rc = tile::dense_check(fname, form, a, lda, b, ldb, c, ldc, M, N, K)) return rc;
  SPX_REQ_FN(b2 && ((uintptr_t)b2) % 16 == 0, "null or unaligned second half");
  SPX_REQ_FN(ldc % 8 == 0 && ((uintptr_t)c) % 16 == 0, "ldc must be a multiple of 8 and c 16-byte aligned");
  SPX_REQ_FN(spx_gemm_pair_takes(form, M, N, K, ldb, max_parts) && 256 * ldc * 2 < 0x7ffffff0ll, "sizes that spx_gemm_pair_takes refuses");
  if (form) {
    const int64_t need = spx_gemm_auto_workspace_bytes(1, M, N, K, max_parts);
    SPX_REQ_FN(need == 0 || (workspace && ((uintptr_t)workspace) % 16 == 0 && workspace_bytes >= need),
               "workspace too small, null or unaligned");
    return auto_product(fname, 1, a, lda, b, ldb, c, ldc, M, N, K, nullptr, max_parts, workspace, workspace_bytes, parts, stream, b2);
  }
  const bool cut = max_parts > 1 && workspace && ((uintptr_t)workspace) % 16 == 0 && workspace_bytes >= spx_gemm_tail_workspace_bytes();
  return nt_pair(fname, a, lda, b, b2, ldb, c, ldc, M, N, K, cut ? reinterpret_cast<float*>(workspace) : nullptr, max_parts, stream);
}

// The weights in the product's own epilogue (a load per row and a multiply per result) or in the pass that adds its parts; the
// rows are put back in place by a launch that moves them.  Product and that launch, weights applied by the launch (a second
// rounding) / here, us: 360 live rows of 512 x 32000 -> 2048 65 / 64, 2100 of 3001 -> 4096 524 / 526, 2867 of 4096 -> 4096 652 / 651,
// 5734 of 8192 -> 8192 2280 / 2291.
extern "C" int spx_gemm_bf16_rows_graded(const void* a, int64_t lda, const void* b, int64_t ldb, void* c, int64_t ldc,
                                         int64_t M, int64_t N, int64_t K, const int32_t* m_live, const int32_t* row,
                                         const float* row_weight, const float* scale, float factor, int32_t max_parts,
                                         int32_t split_parts, void* workspace, int64_t workspace_bytes, void* stream) {
  const char* fname = __func__;
  SPX_REQ_FN(max_parts >= 1 && max_parts <= 8 && split_parts >= 1 && split_parts <= 8, "parts must be 1 .. 8");
  SPX_REQ_FN(m_live && row && row_weight && scale, "null row count, rows, weights or scale");
  SPX_REQ_FN(!workspace || ((uintptr_t)workspace) % 16 == 0, "unaligned workspace");
  if (int rc = tile::dense_check(fname, 0, a, lda, b, ldb, c, ldc, M, N, K)) return rc;
  const RowGrade grade = {row, row_weight, scale, factor};
  const bool vec = ldc % 8 == 0 && ((uintptr_t)c) % 16 == 0;  // (what the pass that adds the parts stores)
  const tile::Choice ch = tile::choose(2, M, N, K, max_parts, can_split(N) && vec && workspace);
  const int64_t part = M * N * (int64_t)sizeof(float);
  if (ch.tile == tile::kBig) {
    return nt_rows_graded(fname, a, lda, b, ldb, c, ldc, M, N, K, m_live, grade, reinterpret_cast<float*>(workspace),
                          workspace ? workspace_bytes / (int64_t)sizeof(float) : 0, split_parts, stream);
  }
  SPX_REQ_FN(ch.parts == 1 || workspace_bytes >= ch.parts * part, "workspace too small");
  const tile::Config& cfg = tile::kNT[ch.tile];
  tile::Params p{};
  p.A = reinterpret_cast<const uint16_t*>(a);
  p.B = reinterpret_cast<const uint16_t*>(b);
  p.C = c;
  p.lda = lda; p.ldb = ldb; p.ldc = ldc;
  p.M = (int)M; p.N = (int)N; p.K = (int)K;
  const int64_t tiles_m = (M + cfg.tm - 1) / cfg.tm, tiles_n = (N + cfg.tn - 1) / cfg.tn;
  SPX_REQ_FN(tiles_m * tiles_n * ch.parts < (1ll << 31), "too many tiles");
  p.tiles_m = (int)tiles_m; p.tiles_n = (int)tiles_n; p.parts = ch.parts;
  p.part_ws = reinterpret_cast<float*>(workspace);
  p.m_live = m_live;
  p.grade = grade;
  // The host cuts for all M rows; the parts chosen for the live ones, us: x 32000 -> 2048, 1075 live of 1536 rows 172 -> 141,
  // 768 of them 162 -> 93, 716 of 1024 98 -> 92, 512 of them 92 -> 69, 620 of 888 98 -> 90; -> 4096, 460 of 1536 345 -> 123; all rows
  // live: as before.
  const int64_t floats = tile::live_cut_floats(cfg, M, N, K, max_parts);
  if (can_split(N) && vec && workspace && floats && workspace_bytes >= floats * (int64_t)sizeof(float)) p.cut = tile::live_cut(cfg, K);
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  if (int rc = tile::launch_graded(fname, ch.tile, p, st)) return rc;
  if (ch.parts == 1 && !p.cut.max_parts) return SPX_OK;
  return tile::launch_reduce<0>(fname, p.part_ws, c, ldc, M, N, ch.parts, m_live, st, grade, p.cut, cfg.tm, cfg.tn);
}

extern "C" int64_t spx_gemm_graded_workspace_bytes(int64_t M, int64_t N, int64_t K, int32_t max_parts, int32_t split_parts) {
  if (M <= 0 || N <= 0 || K <= 0 || max_parts < 1 || split_parts < 1) return 0;
  if (tile::choose(2, M, N, K, max_parts, can_split(N)).tile != tile::kBig)
    return spx_gemm_auto_workspace_bytes(2, M, N, K, max_parts);
  return nt_rows_graded_floats(M, N, K, std::min(split_parts, 8)) * (int64_t)sizeof(float);
}

extern "C" int32_t spx_gemm_graded_parts(int64_t M, int64_t N, int64_t K, int32_t max_parts, int32_t split_parts,
                                         int64_t workspace_bytes, int64_t live) {
  if (M <= 0 || N <= 0 || K <= 0 || max_parts < 1 || split_parts < 1) return 1;
  const tile::Choice ch = tile::choose(2, M, N, K, max_parts, can_split(N) && workspace_bytes > 0);
  live = std::min(std::max<int64_t>(live, 0), M);
  if (ch.tile == tile::kBig) return nt_rows_graded_parts(live, N, K, workspace_bytes / (int64_t)sizeof(float), split_parts);
  const tile::Config& cfg = tile::kNT[ch.tile];
  const int64_t floats = tile::live_cut_floats(cfg, M, N, K, max_parts);
  if (!can_split(N) || !floats || workspace_bytes < floats * (int64_t)sizeof(float)) return ch.parts;
  return tile::live_cut(cfg, K).parts((int)((live + cfg.tm - 1) / cfg.tm * ((N + cfg.tn - 1) / cfg.tn)), live * N);
}

// ------------------------------------------------------------------------------------------ weight gradients
extern "C" int32_t spx_gemm_tn_parts(int64_t M, int64_t N, int64_t T) {
  if (M <= 0 || N <= 0 || T <= 0) return 1;
  return tile::choose_tn(M, N, T, true).parts;
}

extern "C" float spx_gemm_tn_us(int64_t M, int64_t N, int64_t T) {
  if (M <= 0 || N <= 0 || T <= 0) return 0.f;
  return tile::choose_tn(M, N, T, true).us;
}

extern "C" int spx_gemm_tn_tile(int64_t M, int64_t N, int64_t T) {
  if (M <= 0 || N <= 0 || T <= 0) return 0;
  return tile::choose_tn(M, N, T, true).tile;
}

extern "C" int64_t spx_gemm_tn_workspace_bytes(int64_t M, int64_t N, int64_t T) {
  const int32_t parts = spx_gemm_tn_parts(M, N, T);
  return parts > 1 ? (int64_t)parts * M * N * (int64_t)sizeof(float) : 0;
}

extern "C" int spx_gemm_bf16_tn_auto(const void* a, int64_t lda, const void* b, int64_t ldb, void* c, int64_t ldc,
                                     int64_t M, int64_t N, int64_t T, int out_f32, int accumulate, void* workspace,
                                     int64_t workspace_bytes, void* stream) {
  const char* fname = __func__;
  if (int rc = tile::tn_check(fname, a, lda, b, ldb, c, ldc, M, N, T)) return rc;
  const bool vec = ldc % 8 == 0 && ((uintptr_t)c) % 16 == 0;  // (what the pass that adds the parts stores)
  const tile::Choice ch = tile::choose_tn(M, N, T, vec && workspace);
  if (ch.tile == tile::kBig || (accumulate && ch.parts == 1))  // (the small tiles write results, they add to none)
    return (out_f32 ? spx_gemm_bf16_tn_f32 : spx_gemm_bf16_tn)(a, lda, b, ldb, c, ldc, M, N, T, accumulate, stream);
  SPX_REQ_FN(ch.parts == 1 || (workspace_bytes >= (int64_t)ch.parts * M * N * (int64_t)sizeof(float) &&
                               ((uintptr_t)workspace) % 16 == 0),
             "workspace too small or unaligned");
  const tile::Config& cfg = tile::kTN[ch.tile];
  tile::Params p{};
  p.A = reinterpret_cast<const uint16_t*>(a);
  p.B = reinterpret_cast<const uint16_t*>(b);
  p.C = c;
  p.lda = lda; p.ldb = ldb; p.ldc = ldc;
  p.M = (int)M; p.N = (int)N; p.K = (int)T;
  const int64_t tiles_m = (M + cfg.tm - 1) / cfg.tm, tiles_n = (N + cfg.tn - 1) / cfg.tn;
  SPX_REQ_FN(tiles_m * tiles_n * ch.parts < (1ll << 31), "too many tiles");
  p.tiles_m = (int)tiles_m; p.tiles_n = (int)tiles_n; p.parts = ch.parts;
  p.part_ws = reinterpret_cast<float*>(workspace);
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  if (int rc = out_f32 ? tile::launch_tn_dense<2>(fname, ch.tile, p, st) : tile::launch_tn_dense<0>(fname, ch.tile, p, st))
    return rc;
  if (ch.parts == 1) return SPX_OK;
  switch ((out_f32 ? 2 : 0) + (accumulate ? 1 : 0)) {
    case 0: return tile::launch_reduce<0>(fname, p.part_ws, c, ldc, M, N, ch.parts, nullptr, st);
    case 1: return tile::launch_reduce<1>(fname, p.part_ws, c, ldc, M, N, ch.parts, nullptr, st);
    case 2: return tile::launch_reduce<2>(fname, p.part_ws, c, ldc, M, N, ch.parts, nullptr, st);
    default: return tile::launch_reduce<3>(fname, p.part_ws, c, ldc, M, N, ch.parts, nullptr, st);
  }
}
#undef SPX_REQ_FN
