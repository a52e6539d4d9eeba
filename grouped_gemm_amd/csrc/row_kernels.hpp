// Launches of the row-wise kernels (row_kernels.hip) the C ABI (gmm_api.hip) is built on.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace gg {

// out = gradients of gate | up (rows, 2 * cols) from grad, the gradient of silu(gate) * up
// (rows, cols); two-byte element types (kBF16, kF16).
hipError_t swiglu_backward(const void* gate_up, const void* grad, void* out, int64_t rows, int64_t cols, int dt,
                           hipStream_t stream);

// dst[d] = sum of the rows r of src with row_index[r] == d, in fp32, rounded once (zeros where there
// are none); `scratch` holds sum_rows_scratch_bytes, 4-byte aligned, any contents.
uint64_t sum_rows_scratch_bytes(int64_t rows, int64_t destinations);
hipError_t sum_rows(const void* src, const int32_t* row_index, void* dst, int64_t rows, int64_t destinations,
                    int64_t cols, int dt, void* scratch, hipStream_t stream);

// dst (batches, dst_rows, dst_cols) = src (batches, src_rows, src_cols) in the upper left corner of
// each batch, zeros elsewhere; elements of 1 or 2 bytes, dst's rows whole 16-byte chunks on 16-byte
// boundaries, src aligned to its elements only.
hipError_t pad_rows(const void* src, void* dst, int64_t batches, int64_t src_rows, int64_t src_cols, int64_t dst_rows,
                    int64_t dst_cols, int elem_bytes, hipStream_t stream);
// dst (batches, dst_rows, dst_cols) = the upper left corner of each batch of src (batches, src_rows,
// src_cols); elements of 2 bytes, both aligned to their elements only.
hipError_t unpad_rows(const void* src, void* dst, int64_t batches, int64_t src_rows, int64_t src_cols, int64_t dst_rows,
                      int64_t dst_cols, hipStream_t stream);

}  // namespace gg
