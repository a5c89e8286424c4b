// Entry points of gemm_tile.hip for the other GEMM sources (arguments as in the C entry points that call them).
#pragma once

#include <stdint.h>

namespace spx {
namespace tile {

int grouped_nt(const char* fname, const void* a, int64_t lda, const void* b, int64_t ldb, int64_t b_group_stride,
               void* c, int64_t ldc, int64_t rows, int64_t N, int64_t K, const int32_t* group_off, int64_t groups,
               void* workspace, void* stream);
int grouped_tn(const char* fname, const void* a, int64_t lda, const void* b, int64_t ldb, void* c, int64_t ldc,
               int64_t c_group_stride, int64_t M, int64_t N, int64_t rows, const int32_t* group_off, int64_t groups,
               int out_f32, int accumulate, void* stream);

// the argument rules of every weight-gradient product (gemm_bf16_tn.hip)
int tn_check(const char* fname, const void* a, int64_t lda, const void* b, int64_t ldb, const void* c, int64_t ldc, int64_t M,
             int64_t N, int64_t T);

}  // namespace tile
}  // namespace spx
