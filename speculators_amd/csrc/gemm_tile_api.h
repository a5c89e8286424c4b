// Entry points of gemm_tile.hip for the other GEMM sources (arguments as in the C entry points that call them).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace spx {

// What the rows of a packed product are multiplied by before their one rounding: row m of the result is row row[m] of the
// whole, with a weight of its own and a scalar on the device (row == nullptr: nothing).
struct RowGrade {
  const int32_t* row;
  const float* weight;
  const float* scale;
  float factor;
  __device__ __forceinline__ float at(int m) const { return weight[row[m]] * (*scale * factor); }
};

// spx_gemm_bf16_nt_rows with graded rows, its last round cut where part_ws has room (gemm_bf16.hip)
int nt_rows_graded(const char* fname, const void* a, int64_t lda, const void* b, int64_t ldb, void* c, int64_t ldc, int64_t M,
                   int64_t N, int64_t K, const int32_t* m_live, const RowGrade& grade, float* part_ws, int64_t part_floats,
                   int max_parts, void* stream);
// the most floats of part_ws that it uses for any number of rows up to M
int64_t nt_rows_graded_floats(int64_t M, int64_t N, int64_t K, int max_parts);
// the parts of its last round of tiles for `live` rows
int nt_rows_graded_parts(int64_t live, int64_t N, int64_t K, int64_t part_floats, int max_parts);

// A product by workgroups that walk its tiles (gemm_bf16_walk.hip): a b^T or (slow) a b, n_grid = its tiles and the parts of
// those that are cut; m_live, part_ws, max_parts, tail_mode, grade as in the 256 x 256 kernel of gemm_bf16.hip.  slow: no grade.
struct WalkArgs {
  const uint16_t* a;
  int64_t lda;
  const uint16_t* b;
  int64_t ldb;
  uint16_t* c;
  int64_t ldc, M, N, K;
  const int32_t* m_live;
  float* part_ws;
  int max_parts, tail_mode, cus;
  int64_t n_grid;
  RowGrade grade;
  int parts = 1;  // > 1: the contraction is cut whole, fp32 results in part_ws, [parts][M][N]
  const uint16_t* b2 = nullptr;  // the second half of b's rows (half of N, slow: of K), where they are not behind the first
};
bool walk_takes(bool slow, const void* c, int64_t ldb, int64_t ldc, int64_t N, int64_t K, int64_t n_grid, int parts = 1);
int walk(const char* fname, bool slow, const WalkArgs& w, hipStream_t st);

// a b^T of the 256 x 256 kernels, its last round cut where there is part_ws, b's second half of rows at b2 (gemm_bf16.hip); the sizes
// are what walk_takes says
int nt_pair(const char* fname, const void* a, int64_t lda, const void* b, const void* b2, int64_t ldb, void* c, int64_t ldc, int64_t M,
            int64_t N, int64_t K, float* part_ws, int max_parts, void* stream);

namespace tile {

int grouped_nt(const char* fname, const void* a, int64_t lda, const void* b, int64_t ldb, int64_t b_group_stride,
               void* c, int64_t ldc, int64_t rows, int64_t N, int64_t K, const int32_t* group_off, int64_t groups,
               void* workspace, void* stream);
int grouped_tn(const char* fname, const void* a, int64_t lda, const void* b, int64_t ldb, void* c, int64_t ldc,
               int64_t c_group_stride, int64_t M, int64_t N, int64_t rows, const int32_t* group_off, int64_t groups,
               int out_f32, int accumulate, void* stream, const int32_t* src = nullptr, int64_t src_rows = 0,
               int operand = 0);

// the argument rules of every weight-gradient product (gemm_bf16_tn.hip)
int tn_check(const char* fname, const void* a, int64_t lda, const void* b, int64_t ldb, const void* c, int64_t ldc, int64_t M,
             int64_t N, int64_t T);

}  // namespace tile
}  // namespace spx
