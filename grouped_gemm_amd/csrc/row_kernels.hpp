// Launches of the row-wise kernels (row_kernels.hip) the C ABI (gmm_api.hip) is built on.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace gg {

// out = gradients of gate | up (rows, 2 * cols) from grad, the gradient of silu(gate) * up
// (rows, cols); two-byte element types (kBF16, kF16).
hipError_t swiglu_backward(const void* gate_up, const void* grad, void* out, int64_t rows, int64_t cols, int dt,
                           hipStream_t stream);

}  // namespace gg
