// Row-wise passes of the operators' backward, bound by memory: everything elementwise between two
// grouped GEMMs goes over its tensors once.
#include "row_kernels.hpp"

#include "gmm_kernel.hpp"

namespace gg {
namespace {

constexpr int kRowThreads = 256;
// Enough workgroups to fill 256 compute units eight waves deep; larger tensors are walked in strides.
constexpr uint32_t kRowBlocks = 2048;

template <int DT>
__device__ __forceinline__ float widen(uint16_t bits) {
  if constexpr (DT == kBF16) {
    return __builtin_bit_cast(float, (uint32_t)bits << 16);
  } else {
    return (float)__builtin_bit_cast(_Float16, bits);
  }
}

template <int DT>
__device__ __forceinline__ uint16_t narrow(float v) {
  if constexpr (DT == kBF16) {
    return __builtin_bit_cast(uint16_t, (__bf16)v);
  } else {
    return __builtin_bit_cast(uint16_t, (_Float16)v);
  }
}

template <int VEC>
struct Halves {
  uint16_t v[VEC];
} __attribute__((aligned(VEC * 2)));

// Derivative of silu(gate) * up for gate | up side by side in a row: reads gate, up and the
// gradient of the product once, writes the gradients of both.  Bound by memory, so one pass and
// accesses of up to 16 bytes (VEC elements); items are numbered along the rows, so consecutive lanes
// touch consecutive memory.  16384 rows x 4096 columns, bf16: 113 us, 5.9 TB/s of the 671 MB it has
// to move; the same formula as thirteen elementwise passes with fp32 intermediates took 1710 us.
template <int DT, int VEC>
__global__ __launch_bounds__(kRowThreads) void swiglu_backward_kernel(const uint16_t* gate_up, const uint16_t* grad,
                                                                      uint16_t* out, uint32_t cols, uint32_t items) {
  using V = Halves<VEC>;
  const uint32_t per_row = cols / VEC;
  for (uint32_t i = blockIdx.x * kRowThreads + threadIdx.x; i < items; i += gridDim.x * kRowThreads) {
    const uint32_t row = i / per_row, col = (i - row * per_row) * VEC;
    const uint64_t at = (uint64_t)row * (2 * (uint64_t)cols) + col;
    const V g = *reinterpret_cast<const V*>(gate_up + at);
    const V u = *reinterpret_cast<const V*>(gate_up + at + cols);
    const V d = *reinterpret_cast<const V*>(grad + (uint64_t)row * cols + col);
    V dg, du;
#pragma unroll
    for (int e = 0; e < VEC; ++e) {
      const float gate = widen<DT>(g.v[e]), up = widen<DT>(u.v[e]), up_grad = widen<DT>(d.v[e]);
      const float sig = 1.0f / (1.0f + __expf(-gate));
      dg.v[e] = narrow<DT>(up_grad * up * sig * (1.0f + gate * (1.0f - sig)));
      du.v[e] = narrow<DT>(up_grad * gate * sig);
    }
    *reinterpret_cast<V*>(out + at) = dg;
    *reinterpret_cast<V*>(out + at + cols) = du;
  }
}

uint32_t row_blocks(uint32_t items) {
  const uint32_t all = (items + kRowThreads - 1) / kRowThreads;
  return all < kRowBlocks ? all : kRowBlocks;
}

template <int DT>
hipError_t launch_swiglu_backward(const uint16_t* gate_up, const uint16_t* grad, uint16_t* out, int64_t rows,
                                  int64_t cols, int vec, hipStream_t stream) {
  // (32-bit item numbers: tensors of more than 2^30 items go in slabs of rows)
  const int64_t slab = (int64_t(1) << 30) / (cols / vec);
  for (int64_t row = 0; row < rows; row += slab) {
    const int64_t count = rows - row < slab ? rows - row : slab;
    const uint32_t items = (uint32_t)(count * (cols / vec));
    const uint16_t* gu = gate_up + row * 2 * cols;
    const uint16_t* gr = grad + row * cols;
    uint16_t* o = out + row * 2 * cols;
#define GG_LAUNCH(V)                                                                                            \
  hipLaunchKernelGGL((swiglu_backward_kernel<DT, V>), dim3(row_blocks(items)), dim3(kRowThreads), 0, stream, gu, \
                     gr, o, (uint32_t)cols, items)
    switch (vec) {
      case 8: GG_LAUNCH(8); break;
      case 4: GG_LAUNCH(4); break;
      case 2: GG_LAUNCH(2); break;
      default: GG_LAUNCH(1); break;
    }
#undef GG_LAUNCH
    const hipError_t err = hipGetLastError();
    if (err != hipSuccess) return err;
  }
  return hipSuccess;
}

}  // namespace

hipError_t swiglu_backward(const void* gate_up, const void* grad, void* out, int64_t rows, int64_t cols, int dt,
                           hipStream_t stream) {
  const uintptr_t bits = reinterpret_cast<uintptr_t>(gate_up) | reinterpret_cast<uintptr_t>(grad) |
                         reinterpret_cast<uintptr_t>(out) | (uintptr_t)(2 * cols);
  int vec = 8;
  while (vec > 1 && (bits & (uintptr_t)(2 * vec - 1))) vec >>= 1;
  auto launch = dt == kBF16 ? &launch_swiglu_backward<kBF16> : &launch_swiglu_backward<kF16>;
  return launch(static_cast<const uint16_t*>(gate_up), static_cast<const uint16_t*>(grad),
                static_cast<uint16_t*>(out), rows, cols, vec, stream);
}

}  // namespace gg
