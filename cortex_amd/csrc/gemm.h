// gemm.h -- the float matrix product of ops_gemm.hip.
#pragma once

#include "common.h"

namespace cthip {

// c = alpha * a b + beta * c: a [m, k], stored so if row_major_a, else [k, m]; b [k, n], stored [n, k] if row_major_b, else
// as it is.
struct GemmProduct {
  const float* a;
  const float* b;
  float* c;
  int64_t lda, ldb, ldc, m, n, k;
  bool row_major_a, row_major_b;
  float alpha, beta;
};
// Whether gemm_split forms this product; what it does not is the library's.
bool gemm_split_takes(const GemmProduct& p);
int gemm_split(hipStream_t s, const GemmProduct& p);

}  // namespace cthip
