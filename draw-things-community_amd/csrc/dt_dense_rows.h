// Launcher of the few-rows Dense kernel (dt_dense_rows.hip).
#pragma once
#include "dt_dense_kernel.h"

namespace dt {

constexpr int kRowsMax = 64;  // rows of X the kernel takes

// Features per workgroup for a launch of `n_total` features, or 0 where the kernel does not apply.
int dense_rows_features(int64_t M, int64_t K, int qbits, int nib, int64_t n_total);

// One problem (DenseArgs::g[0]) with its weights' tiles numbered in blocks of `features`.
dt_status dense_rows_launch(hipStream_t s, const DenseArgs& a, int qbits, int features);

}  // namespace dt
