// Host side of the tile GEMM kernels (gemm_tile.h): which tile a product gets, and the grouped forms.
//
// The 256 x 256 kernels of gemm_bf16.hip / gemm_bf16_tn.hip are built for products of many tiles with a long
// contraction.  A group of a grouped product is often neither: 512 experts x 80 rows each are 512 ragged row bands,
// and their weight gradient contracts over 80 rows.  Measured there (4096 tokens, top 10 of 512 experts, gate/up
// 2048 -> 1024; 2.1 GB of weights, 430 us at the rate of a copy):
//   forward          256 x 256, 4 waves 573 us -> 128 x 256, 8 waves, 3 slabs 456 us
//   input gradient   595 us + 786 us to transpose the weights -> 459 us on the weights as they lie (NN form)
//   weight gradient  bf16, 4 waves 760 us -> 8 waves 698 us (1067 us with the fp32 result it replaces)

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

template <int TM, int TN, int WM, int WN, int STAGES, int MINB, bool AT, bool BT, int OUT>
static int launch(const char* fname, Params p, int groups_y, hipStream_t st) {
  constexpr int kSmem = (TM + TN) * kTK * 2 * STAGES;
  static std::atomic<uint64_t> lds_set;
  auto* const kernel = &gemm_tile_kernel<TM, TN, WM, WN, STAGES, MINB, AT, BT, OUT>;
  if (int rc = ensure_dynamic_lds(reinterpret_cast<const void*>(kernel), kSmem, lds_set, fname)) return rc;
  hipLaunchKernelGGL((gemm_tile_kernel<TM, TN, WM, WN, STAGES, MINB, AT, BT, OUT>),
                     dim3((unsigned)(p.tiles_m * p.tiles_n * p.parts), (unsigned)groups_y), dim3(64 * WM * WN), kSmem,
                     st, p);
  return check_launch(fname);
}

#define SPX_REQ_FN(cond, what) do { if (!(cond)) return spx::fail_arg(fname, what); } while (0)

static int64_t table_entries(int64_t rows, int64_t groups, int tm) { return (rows + tm - 1) / tm + groups; }

// Grouped product over the rows of A: c[r, :] = a[r, :] b_e^T (BT = false, b_e [N, K]) or a[r, :] b_e (BT = true,
// b_e [K, N]).
template <bool BT>
static int grouped_rows(const char* fname, const void* a, int64_t lda, const void* b, int64_t ldb,
                        int64_t b_group_stride, void* c, int64_t ldc, int64_t rows, int64_t N, int64_t K,
                        const int32_t* group_off, int64_t groups, void* workspace, bool wide_m, hipStream_t st) {
  const int tm = wide_m ? 256 : 128;
  const int64_t max_tiles = table_entries(rows, groups, tm), tiles_n = (N + 255) / 256;
  SPX_REQ_FN(max_tiles * tiles_n < (1ll << 31), "too many tiles");
  int32_t* const tab = reinterpret_cast<int32_t*>(workspace);
  hipLaunchKernelGGL(group_tiles_kernel, dim3(1), dim3(256), 0, st, group_off, (int)groups, (int)rows, tm,
                     (int)max_tiles, tab);
  if (int rc = check_launch(fname)) return rc;
  Params p{};
  p.A = reinterpret_cast<const uint16_t*>(a);
  p.B = reinterpret_cast<const uint16_t*>(b);
  p.C = c;
  p.lda = lda; p.ldb = ldb; p.ldc = ldc;
  p.M = (int)rows; p.N = (int)N; p.K = (int)K;
  p.tiles_m = (int)max_tiles; p.tiles_n = (int)tiles_n; p.parts = 1;
  p.tile_tab = tab; p.group_off = group_off; p.group_stride = b_group_stride;
  return wide_m ? launch<256, 256, 2, 4, 2, 2, false, BT, 0>(fname, p, 1, st)
                : launch<128, 256, 2, 4, 3, 2, false, BT, 0>(fname, p, 1, st);
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
                             false, reinterpret_cast<hipStream_t>(stream));
}

int grouped_tn(const char* fname, const void* a, int64_t lda, const void* b, int64_t ldb, void* c, int64_t ldc,
               int64_t c_group_stride, int64_t M, int64_t N, int64_t rows, const int32_t* group_off, int64_t groups,
               int out_f32, int accumulate, void* stream) {
  Params p{};
  p.A = reinterpret_cast<const uint16_t*>(a);
  p.B = reinterpret_cast<const uint16_t*>(b);
  p.C = c;
  p.lda = lda; p.ldb = ldb; p.ldc = ldc;
  p.M = (int)M; p.N = (int)N; p.K = (int)rows;
  p.tiles_m = (int)((M + 255) / 256); p.tiles_n = (int)((N + 255) / 256); p.parts = 1;
  p.group_off = group_off; p.group_stride = c_group_stride;
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  switch ((out_f32 ? 2 : 0) + (accumulate ? 1 : 0)) {
    case 0: return launch<256, 256, 2, 4, 2, 2, true, true, 0>(fname, p, (int)groups, st);
    case 1: return launch<256, 256, 2, 4, 2, 2, true, true, 1>(fname, p, (int)groups, st);
    case 2: return launch<256, 256, 2, 4, 2, 2, true, true, 2>(fname, p, (int)groups, st);
    default: return launch<256, 256, 2, 4, 2, 2, true, true, 3>(fname, p, (int)groups, st);
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
  // 256 rows a group on average: the taller tile reads the group's weights half as often.  16384 tokens, top 8 of 512
  // experts of width 768 (256 rows): 1176 us with 128 rows a tile, 1183 us with 256; 320 rows 249 / 243 us; 2560
  // rows 833 / 729 us
  return tile::grouped_rows<true>(fname, a, lda, b, ldb, b_group_stride, c, ldc, rows, N, K, group_offsets, groups,
                                  workspace, rows > 256 * groups, reinterpret_cast<hipStream_t>(stream));
}
#undef SPX_REQ_FN
