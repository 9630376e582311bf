// sort_rows.h -- stable sort of a column's rows by value.
#pragma once

#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

#include "rtscan_hip.h"

namespace rts {

// Device bytes of workspace that sort_rows needs for n rows.
size_t sort_rows_workspace(int64_t n);

// val[i], pos[i] = the i-th smallest value of col and its row, rows of equal value in row
// order (asynchronous on s).  work is 16-byte aligned, the others need not be; none overlap.
// 1 <= n < 2^31.
hipError_t sort_rows(const CODE *col, int64_t n, CODE *val, uint32_t *pos, void *work, hipStream_t s);

}  // namespace rts
