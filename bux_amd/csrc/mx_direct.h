// The MXFP8 rows GEMM for short groups (mx_direct.hip): which calls it takes, and its
// launch. grouped_mx.hip's launch asks first.
#pragma once

#include "common.h"

namespace bux {

// The first row of the kernel's block `i` of a tile that starts at `lo`: 64 bits, since a
// tile of a list's last rows and its blocks past them reach beyond 2^31.
constexpr int DIRECT_BLOCK = 32;  // rows a wave
__host__ __device__ __forceinline__ int64_t direct_row(int32_t lo, uint32_t i) {
  return lo + static_cast<int64_t>(DIRECT_BLOCK) * i;
}

// The blocks of rows a wave of rows_direct_kernel takes of a rows GEMM of `m` rows in
// `groups` groups, `n` columns: 1 or 2, or 0 where the call is grouped_mx.hip's.
int rows_direct(int64_t m, int32_t groups, int64_t n);

// As grouped_mx.hip's launch_rows: `list` a tile list of `slots` records (its starts
// before them), the operands in the tiled layout, `bias` NULL or
// (groups, n) of out_dtype, y (height, n) of it.
int launch_rows_direct(const uint8_t* a_values, const uint8_t* a_scales, const uint8_t* b_values,
                       const uint8_t* b_scales, const void* list, int64_t slots, int32_t groups,
                       int64_t m, int64_t n, int64_t k, int64_t height, int out_dtype,
                       const void* bias, void* y, hipStream_t s);

}  // namespace bux
