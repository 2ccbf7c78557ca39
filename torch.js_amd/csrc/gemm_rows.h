// The product of a few rows with a transposed matrix (gemm_rows.hip).
#pragma once

#include "gemm_args.h"
#include "wave.h"

namespace tjh {

constexpr int64_t kFewRows = 8;

// C = alpha A B^T + beta C (+ bias_mode 0, 1 or 2) with act 0, 1 (aux null)
// or 3, for M <= kFewRows, any K, strides and float-aligned pointers.
int gemm_rows(const GemmArgs& g, int cus);

}  // namespace tjh
