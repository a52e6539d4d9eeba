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
// to move; the same formula as thirteen elementwise passes with fp32 intermediates took 1710 us.  The
// full exponential: the short one, whose error grows with |gate|, is 1 % faster here, 8 % at 4096 x 1408 (12 us).
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
      const float sig = 1.0f / (1.0f + expf(-gate));
      dg.v[e] = narrow<DT>(up_grad * up * sig * (1.0f + gate * (1.0f - sig)));
      du.v[e] = narrow<DT>(up_grad * gate * sig);
    }
    *reinterpret_cast<V*>(out + at) = dg;
    *reinterpret_cast<V*>(out + at + cols) = du;
  }
}

// Rows that name the same destination, summed: the inverse of a gather.  An index names each
// destination a few times (top-k routing), in any order, so its inverse is built on the way: per
// destination a count and kInlineRows slots for the rows that name it, filled with one atomic
// per row; rows past those (an index may name a row any number of times) hang on a list per
// destination.  The slots are put in ascending order by whoever sums them, so the sums of up to
// kInlineRows rows do not depend on timing.
//
// Bound by reading every row once: 49152 rows x 2048 columns onto 8192 destinations (six each), bf16:
// 51 us, 4.6 TB/s, and 9 us for the two kernels that build the inverse.  Adding the rows to a cleared
// fp32 tensor atom by atom, with a conversion on either side, took 481 us.
constexpr int kInlineRows = 8;

struct RowSumScratch {
  int32_t* count;       // [destinations] rows that name it; zero before use
  int32_t* list_head;   // [destinations] 1 + first row of its list, 0: none; zero before use
  int32_t* slots;       // [destinations][kInlineRows]
  int32_t* list_next;   // [rows] 1 + next row of the same list, 0: none
};

// (64-bit numbers: two words per destination may be close to 2^32, past which a step would wrap around)
__global__ __launch_bounds__(kRowThreads) void clear_words_kernel(int32_t* words, uint64_t n) {
  for (uint64_t i = blockIdx.x * kRowThreads + threadIdx.x; i < n; i += gridDim.x * kRowThreads) words[i] = 0;
}

__global__ __launch_bounds__(kRowThreads) void invert_index_kernel(const int32_t* row_index, uint32_t rows,
                                                                   uint32_t destinations, RowSumScratch s) {
  for (uint32_t r = blockIdx.x * kRowThreads + threadIdx.x; r < rows; r += gridDim.x * kRowThreads) {
    const uint32_t d = (uint32_t)row_index[r];
    if (d >= destinations) continue;   // names no row
    const int at = atomicAdd(&s.count[d], 1);
    if (at < kInlineRows) {
      s.slots[(uint64_t)d * kInlineRows + at] = (int32_t)r;
    } else {
      s.list_next[r] = atomicExch(&s.list_head[d], (int32_t)r + 1);
    }
  }
}

// One item: VEC columns of one destination row, summed in fp32 and rounded once; a destination
// that no row names gets zeros.  All loads of an item's rows are in flight together.
template <int DT, int VEC>
__global__ __launch_bounds__(kRowThreads) void sum_rows_kernel(const uint16_t* src, uint16_t* dst, uint32_t cols,
                                                               uint32_t first, uint32_t items, RowSumScratch s) {
  using V = Halves<VEC>;
  constexpr int32_t NONE = 0x7fffffff;
  const uint32_t per_row = cols / VEC;
  for (uint32_t i = blockIdx.x * kRowThreads + threadIdx.x; i < items; i += gridDim.x * kRowThreads) {
    const uint32_t d = first + i / per_row, col = i % per_row * VEC;
    const int count = s.count[d];
    int32_t row[kInlineRows];
#pragma unroll
    for (int k = 0; k < kInlineRows; ++k) {
      const int32_t r = s.slots[(uint64_t)d * kInlineRows + k];   // (not written past the count)
      row[k] = k < count ? r : NONE;
    }
    // ascending: odd-even transposition, kInlineRows rounds
#pragma unroll
    for (int round = 0; round < kInlineRows; ++round)
#pragma unroll
      for (int k = round & 1; k + 1 < kInlineRows; k += 2) {
        const int32_t lo = min(row[k], row[k + 1]), hi = max(row[k], row[k + 1]);
        row[k] = lo, row[k + 1] = hi;
      }
    V v[kInlineRows];
#pragma unroll
    for (int k = 0; k < kInlineRows; ++k)
      if (row[k] != NONE) v[k] = *reinterpret_cast<const V*>(src + (uint64_t)row[k] * cols + col);
    float sum[VEC];
#pragma unroll
    for (int e = 0; e < VEC; ++e) sum[e] = 0.0f;
#pragma unroll
    for (int k = 0; k < kInlineRows; ++k)
      if (row[k] != NONE)
#pragma unroll
        for (int e = 0; e < VEC; ++e) sum[e] += widen<DT>(v[k].v[e]);
    if (count > kInlineRows) {
      for (int32_t next = s.list_head[d]; next != 0; next = s.list_next[next - 1]) {
        const V more = *reinterpret_cast<const V*>(src + (uint64_t)(next - 1) * cols + col);
#pragma unroll
        for (int e = 0; e < VEC; ++e) sum[e] += widen<DT>(more.v[e]);
      }
    }
    V out;
#pragma unroll
    for (int e = 0; e < VEC; ++e) out.v[e] = narrow<DT>(sum[e]);
    *reinterpret_cast<V*>(dst + (uint64_t)d * cols + col) = out;
  }
}

// Rows of `cols` elements copied to rows of another length: operands whose rows do not start on
// 4-byte boundaries are laid out again, zero-padded, for the streaming kernels, and their results
// are taken back.  Bound by memory: one pass, 16 aligned bytes of the destination per item.  The
// source's alignment is any: the item's bytes are loaded as the dwords that hold them and shifted
// into place (CDNA has no narrower-than-dword alignment for wide loads).  An item that is not whole
// (the end of a padded row, or a chunk of a dense destination with a row boundary in it) moves element
// by element.
template <typename T>
__device__ __forceinline__ u32x4 load_unaligned_16(const T* from) {
  struct Words {
    uint32_t v[4];
  } __attribute__((aligned(4)));
  const uintptr_t at = reinterpret_cast<uintptr_t>(from);
  const uint32_t shift = at & 3;
  const uint32_t* aligned = reinterpret_cast<const uint32_t*>(at - shift);
  const Words w = *reinterpret_cast<const Words*>(aligned);
  // (the fifth dword holds the item's last bytes when it is needed, so it is never outside the tensor)
  const uint32_t last = shift != 0 ? aligned[4] : 0u;
  return u32x4{__builtin_amdgcn_alignbyte(w.v[1], w.v[0], shift), __builtin_amdgcn_alignbyte(w.v[2], w.v[1], shift),
               __builtin_amdgcn_alignbyte(w.v[3], w.v[2], shift), __builtin_amdgcn_alignbyte(last, w.v[3], shift)};
}

// dst: batches of dst_rows rows of dst_cols elements (16 bytes divide a row), zeros around the batch's
// src_rows rows of src_cols elements.  first_row: the first of dst's rows (over all batches) that
// this launch fills; row numbers and item numbers are 32-bit.
//
// A training step of 8192 rows, 8 experts, 2047 -> 5461, bf16 (five of these, three of the reverse):
// 319 us, 5.1 TB/s; torch's strided copies into cleared tensors, 11 copies and 8 fills, took 693.
template <typename T>
__global__ __launch_bounds__(kRowThreads) void pad_rows_kernel(const T* src, T* dst, uint32_t src_rows, uint32_t src_cols,
                                                               uint32_t dst_rows, uint32_t dst_cols, uint32_t first_row,
                                                               uint32_t items) {
  constexpr uint32_t VEC = 16 / sizeof(T);
  const uint32_t per_row = dst_cols / VEC;
  for (uint32_t i = blockIdx.x * kRowThreads + threadIdx.x; i < items; i += gridDim.x * kRowThreads) {
    const uint32_t down = i / per_row, col = (i - down * per_row) * VEC;
    const uint32_t row = first_row + down;
    const uint32_t batch = row / dst_rows, r = row - batch * dst_rows;
    u32x4 v = {0u, 0u, 0u, 0u};
    if (r < src_rows && col < src_cols) {
      const T* from = src + ((uint64_t)batch * src_rows + r) * src_cols + col;
      if (col + VEC <= src_cols) {
        v = load_unaligned_16(from);
      } else {
        T e[VEC];
#pragma unroll
        for (uint32_t k = 0; k < VEC; ++k) e[k] = col + k < src_cols ? from[k] : T(0);
        v = __builtin_bit_cast(u32x4, e);
      }
    }
    *reinterpret_cast<u32x4*>(dst + (uint64_t)row * dst_cols + col) = v;
  }
}

// The reverse: dst is dense, batches of dst_rows rows of dst_cols elements, the upper left parts of
// src's.  Item i covers elements 8 i - head .. + 7 of this launch's part of dst, which begins `lead`
// elements into row `first_row` (over all batches); `count` elements in all.
template <typename T>
__global__ __launch_bounds__(kRowThreads) void unpad_rows_kernel(const T* src, T* dst, uint32_t src_rows, uint32_t src_cols,
                                                                 uint32_t dst_rows, uint32_t dst_cols, uint32_t first_row,
                                                                 uint32_t lead, uint32_t head, uint32_t count, uint32_t items) {
  constexpr uint32_t VEC = 16 / sizeof(T);
  for (uint32_t i = blockIdx.x * kRowThreads + threadIdx.x; i < items; i += gridDim.x * kRowThreads) {
    const int64_t begin = (int64_t)i * VEC - head;   // in dst; below 0 in the first item only
    const uint32_t skip = begin < 0 ? head : 0;
    const uint32_t at = lead + (uint32_t)(begin + skip);
    uint32_t down = at / dst_cols, col = at - down * dst_cols;
    uint32_t row = first_row + down;
    uint32_t batch = row / dst_rows, r = row - batch * dst_rows;
    const T* from = src + ((uint64_t)batch * src_rows + r) * src_cols + col;
    T* to = dst + begin;
    if (skip == 0 && col + VEC <= dst_cols && begin + VEC <= count) {
      *reinterpret_cast<u32x4*>(to) = load_unaligned_16(from);
      continue;
    }
    for (uint32_t k = skip; k < VEC && begin + k < count; ++k) {
      to[k] = *from;
      ++from;
      if (++col == dst_cols) {
        col = 0, ++row;
        batch = row / dst_rows, r = row - batch * dst_rows;
        from = src + ((uint64_t)batch * src_rows + r) * src_cols;
      }
    }
  }
}

uint32_t row_blocks(uint64_t items) {
  const uint64_t all = (items + kRowThreads - 1) / kRowThreads;
  return all < kRowBlocks ? (uint32_t)all : kRowBlocks;
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

template <int DT>
hipError_t launch_sum_rows(const uint16_t* src, uint16_t* dst, int64_t destinations, int64_t cols, int vec,
                           const RowSumScratch& s, hipStream_t stream) {
  const int64_t slab = (int64_t(1) << 30) / (cols / vec);
  for (int64_t first = 0; first < destinations; first += slab) {
    const int64_t count = destinations - first < slab ? destinations - first : slab;
    const uint32_t items = (uint32_t)(count * (cols / vec));
#define GG_LAUNCH(V)                                                                                              \
  hipLaunchKernelGGL((sum_rows_kernel<DT, V>), dim3(row_blocks(items)), dim3(kRowThreads), 0, stream, src, dst, \
                     (uint32_t)cols, (uint32_t)first, items, s)
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

int access_width(uintptr_t bits) {   // elements per access that divide every address and pitch in `bits`
  int vec = 8;
  while (vec > 1 && (bits & (uintptr_t)(2 * vec - 1))) vec >>= 1;
  return vec;
}

}  // namespace

uint64_t sum_rows_scratch_bytes(int64_t rows, int64_t destinations) {
  return (uint64_t)(destinations * (2 + kInlineRows) + rows) * sizeof(int32_t);
}

hipError_t sum_rows(const void* src, const int32_t* row_index, void* dst, int64_t rows, int64_t destinations,
                    int64_t cols, int dt, void* scratch, hipStream_t stream) {
  RowSumScratch s;
  s.count = static_cast<int32_t*>(scratch);
  s.list_head = s.count + destinations;
  s.slots = s.list_head + destinations;
  s.list_next = s.slots + destinations * kInlineRows;
  const uint64_t words = 2 * (uint64_t)destinations;
  hipLaunchKernelGGL(clear_words_kernel, dim3(row_blocks(words)), dim3(kRowThreads), 0, stream, s.count, words);
  hipError_t err = hipGetLastError();
  if (err != hipSuccess) return err;
  if (rows > 0) {
    hipLaunchKernelGGL(invert_index_kernel, dim3(row_blocks((uint32_t)rows)), dim3(kRowThreads), 0, stream, row_index,
                       (uint32_t)rows, (uint32_t)destinations, s);
    err = hipGetLastError();
    if (err != hipSuccess) return err;
  }
  const int vec = access_width(reinterpret_cast<uintptr_t>(src) | reinterpret_cast<uintptr_t>(dst) | (uintptr_t)(2 * cols));
  auto launch = dt == kBF16 ? &launch_sum_rows<kBF16> : &launch_sum_rows<kF16>;
  return launch(static_cast<const uint16_t*>(src), static_cast<uint16_t*>(dst), destinations, cols, vec, s, stream);
}

hipError_t swiglu_backward(const void* gate_up, const void* grad, void* out, int64_t rows, int64_t cols, int dt,
                           hipStream_t stream) {
  const int vec = access_width(reinterpret_cast<uintptr_t>(gate_up) | reinterpret_cast<uintptr_t>(grad) |
                               reinterpret_cast<uintptr_t>(out) | (uintptr_t)(2 * cols));
  auto launch = dt == kBF16 ? &launch_swiglu_backward<kBF16> : &launch_swiglu_backward<kF16>;
  return launch(static_cast<const uint16_t*>(gate_up), static_cast<const uint16_t*>(grad),
                static_cast<uint16_t*>(out), rows, cols, vec, stream);
}

namespace {

template <typename T>
hipError_t launch_pad_rows(const T* src, T* dst, int64_t batches, int64_t src_rows, int64_t src_cols, int64_t dst_rows,
                           int64_t dst_cols, hipStream_t stream) {
  const int64_t per_row = dst_cols / (16 / (int64_t)sizeof(T)), rows = batches * dst_rows;
  // (32-bit item numbers: larger tensors go in slabs of rows)
  const int64_t slab = (int64_t(1) << 30) / per_row;
  for (int64_t first = 0; first < rows; first += slab) {
    const uint32_t items = (uint32_t)((rows - first < slab ? rows - first : slab) * per_row);
    hipLaunchKernelGGL((pad_rows_kernel<T>), dim3(row_blocks(items)), dim3(kRowThreads), 0, stream, src, dst,
                       (uint32_t)src_rows, (uint32_t)src_cols, (uint32_t)dst_rows, (uint32_t)dst_cols, (uint32_t)first, items);
    const hipError_t err = hipGetLastError();
    if (err != hipSuccess) return err;
  }
  return hipSuccess;
}

template <typename T>
hipError_t launch_unpad_rows(const T* src, T* dst, int64_t batches, int64_t src_rows, int64_t src_cols, int64_t dst_rows,
                             int64_t dst_cols, hipStream_t stream) {
  constexpr int64_t VEC = 16 / sizeof(T), SLAB = int64_t(1) << 30;
  const int64_t total = batches * dst_rows * dst_cols;
  for (int64_t first = 0; first < total; first += SLAB) {
    const int64_t count = total - first < SLAB ? total - first : SLAB;
    const int64_t row = first / dst_cols;
    T* to = dst + first;
    const int64_t head = (int64_t)(reinterpret_cast<uintptr_t>(to) % 16 / sizeof(T));
    const uint32_t items = (uint32_t)((head + count + VEC - 1) / VEC);
    hipLaunchKernelGGL((unpad_rows_kernel<T>), dim3(row_blocks(items)), dim3(kRowThreads), 0, stream, src, to,
                       (uint32_t)src_rows, (uint32_t)src_cols, (uint32_t)dst_rows, (uint32_t)dst_cols, (uint32_t)row,
                       (uint32_t)(first - row * dst_cols), (uint32_t)head, (uint32_t)count, items);
    const hipError_t err = hipGetLastError();
    if (err != hipSuccess) return err;
  }
  return hipSuccess;
}

}  // namespace

hipError_t pad_rows(const void* src, void* dst, int64_t batches, int64_t src_rows, int64_t src_cols, int64_t dst_rows,
                    int64_t dst_cols, int elem_bytes, hipStream_t stream) {
  if (elem_bytes == 1)
    return launch_pad_rows(static_cast<const uint8_t*>(src), static_cast<uint8_t*>(dst), batches, src_rows, src_cols,
                           dst_rows, dst_cols, stream);
  return launch_pad_rows(static_cast<const uint16_t*>(src), static_cast<uint16_t*>(dst), batches, src_rows, src_cols,
                         dst_rows, dst_cols, stream);
}

hipError_t unpad_rows(const void* src, void* dst, int64_t batches, int64_t src_rows, int64_t src_cols, int64_t dst_rows,
                      int64_t dst_cols, hipStream_t stream) {
  return launch_unpad_rows(static_cast<const uint16_t*>(src), static_cast<uint16_t*>(dst), batches, src_rows, src_cols,
                           dst_rows, dst_cols, stream);
}

}  // namespace gg
