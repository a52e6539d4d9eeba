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
// per row.  The slots are put in ascending order by whoever sums them, so the sums do not depend on timing.
//
// Bound by reading every row once: 49152 rows x 2048 columns onto 8192 destinations (six each), bf16: 48 us in
// five launches, 36 of them here where the rows still are in the Infinity Cache (in a training step 56); by atomics on a cleared fp32 tensor, with a conversion on
// either side, 484.  Sixteen rows each, 65536 onto 4096: 68 us.
//
// An index may name a row any number of times (padding rows that all name row 0).  Destinations of more
// rows than slots, the heavy ones, are left to two more kernels, which end at once where there are none
// (5 us of the 48): one lists their further rows, the other sums them.  65536 rows, 32 and 300 to a
// destination: 67 and 113 us (by atomics 604 and 587); 4096 of the 49152 rows on one destination: 136 (520), all of them:
// 394 (1356; as one chain of dependent loads 26000).
constexpr int kInlineRows = 16;
constexpr int kWaveRows = 64;       // heavy destinations of up to this many rows are summed by single waves,
constexpr int kListedRows = 1024;   // ... of up to this many by workgroups that sort the rows in LDS

struct RowSumScratch {
  int32_t* count;     // [destinations] rows that name it; zero before use
  int32_t* cursor;    // [kCursorWords] zero before use
  int32_t* slots;     // [destinations][kInlineRows] the first rows that name it
  int32_t* base;      // [destinations] heavy ones: where their further rows begin in `rest`
  int32_t* arrival;   // [rows] how many rows of the same destination were met before the row
  int32_t* rest;      // [rows] the further rows of heavy destinations, one destination after another
  int32_t* heavy;     // [2][most_heavy(rows)] heavy destinations: up to kWaveRows rows; up to kListedRows, others from the back
};
enum : int { kRestUsed = 0, kHeavyWave = 1, kHeavyListed = 2, kHeavyLong = 3, kCursorWords = 4 };
__host__ __device__ constexpr int64_t most_heavy(int64_t rows) { return rows / (kInlineRows + 1); }

// (64-bit numbers: the words may be close to 2^32, past which a step would wrap around)
__global__ __launch_bounds__(kRowThreads) void clear_words_kernel(int32_t* words, uint64_t n) {
  for (uint64_t i = blockIdx.x * kRowThreads + threadIdx.x; i < n; i += gridDim.x * kRowThreads) words[i] = 0;
}

__device__ __forceinline__ int lanes_below(uint64_t mask) {   // lanes of `mask` ahead of this one
  return __builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0));
}

// Atomics of one wave on one address follow each other at 11 ns: the rows of the destinations that the
// first lanes name are counted together (all 49152 rows on one destination: 559 -> 11 us), the others one by one.
__global__ __launch_bounds__(kRowThreads) void invert_index_kernel(const int32_t* row_index, uint32_t rows,
                                                                   uint32_t destinations, RowSumScratch s) {
  for (uint32_t r = blockIdx.x * kRowThreads + threadIdx.x; r < rows; r += gridDim.x * kRowThreads) {
    const uint32_t d = (uint32_t)row_index[r];
    int at = 0;
    bool counted = d >= destinations;   // names no row
#pragma unroll
    for (int round = 0; round < 2; ++round) {
      if (counted) continue;
      const uint32_t first = (uint32_t)__builtin_amdgcn_readfirstlane((int)d);   // of the lanes not counted yet
      const uint64_t same = __ballot(d == first);
      if (d == first) {
        const int before = lanes_below(same);
        int begin = 0;
        if (before == 0) begin = atomicAdd(&s.count[d], __popcll(same));
        at = __builtin_amdgcn_readfirstlane(begin) + before;   // (the lane ahead of all of `same`)
        counted = true;
      }
    }
    if (!counted) at = atomicAdd(&s.count[d], 1);
    s.arrival[r] = at;
    if (d < destinations && at < kInlineRows) s.slots[(uint64_t)d * kInlineRows + at] = (int32_t)r;
  }
}

// The VEC columns from `col` on of the up to N rows in `slots`, in ascending order of the rows; eight
// loads in flight.
template <int DT, int VEC, int N>
__device__ __forceinline__ void sum_few_rows(const uint16_t* src, const int32_t* slots, int count, uint32_t cols, uint32_t col,
                                             float* sum) {
  using V = Halves<VEC>;
  constexpr int32_t NONE = 0x7fffffff;
  constexpr int IN_FLIGHT = 8;
  int32_t row[N];
#pragma unroll
  for (int k = 0; k < N; ++k) {
    const int32_t r = slots[k];   // (not written past the count)
    row[k] = k < count ? r : NONE;
  }
  // odd-even transposition, N rounds
#pragma unroll
  for (int round = 0; round < N; ++round)
#pragma unroll
    for (int k = round & 1; k + 1 < N; k += 2) {
      const int32_t lo = min(row[k], row[k + 1]), hi = max(row[k], row[k + 1]);
      row[k] = lo, row[k + 1] = hi;
    }
#pragma unroll
  for (int at = 0; at < N; at += IN_FLIGHT) {
    V v[IN_FLIGHT];
#pragma unroll
    for (int k = 0; k < IN_FLIGHT; ++k)
      if (row[at + k] != NONE) v[k] = *reinterpret_cast<const V*>(src + (uint64_t)row[at + k] * cols + col);
#pragma unroll
    for (int k = 0; k < IN_FLIGHT; ++k)
      if (row[at + k] != NONE)
#pragma unroll
        for (int e = 0; e < VEC; ++e) sum[e] += widen<DT>(v[k].v[e]);
  }
}

// Enters the heavy ones of the destinations first .. first + number - 1 into the list; one
// atomic per wave and list, not one per destination.
__device__ __forceinline__ void list_heavy_destinations(uint32_t first, uint32_t number, uint32_t rows, const RowSumScratch& s) {
  const uint32_t step = gridDim.x * kRowThreads, lane = threadIdx.x & 63;
  for (uint32_t wave = blockIdx.x * kRowThreads + (threadIdx.x & ~63u); wave < number; wave += step) {   // (whole waves)
    const uint32_t d = first + wave + lane;
    const int count = wave + lane < number ? s.count[d] : 0;
    if (__ballot(count > kInlineRows) == 0) continue;
    const int list = count <= kInlineRows ? kRestUsed : (count <= kWaveRows ? kHeavyWave : (count <= kListedRows ? kHeavyListed : kHeavyLong));
    const int more = count > kInlineRows ? count - kInlineRows : 0;
    int upto = more;
#pragma unroll
    for (int distance = 1; distance < 64; distance <<= 1) {
      const int o = __shfl_up(upto, distance);
      if ((int)lane >= distance) upto += o;
    }
    int begin = lane == 63 ? atomicAdd(&s.cursor[kRestUsed], upto) : 0;
    begin = __shfl(begin, 63);
    if (more > 0) s.base[d] = begin + upto - more;
#pragma unroll
    for (int l = kHeavyWave; l <= kHeavyLong; ++l) {
      const uint64_t mask = __ballot(list == l);
      if (mask == 0) continue;
      begin = lane == 0 ? atomicAdd(&s.cursor[l], __popcll(mask)) : 0;
      const int64_t at = __shfl(begin, 0) + lanes_below(mask), most = most_heavy(rows);
      if (list == l) s.heavy[l == kHeavyWave ? at : (l == kHeavyListed ? most + at : 2 * most - 1 - at)] = (int32_t)d;
    }
  }
}

// One item: VEC columns of one destination row, summed in fp32 and rounded once; a destination
// that no row names gets zeros.
template <int DT, int VEC>
__global__ __launch_bounds__(kRowThreads) void sum_rows_kernel(const uint16_t* src, uint16_t* dst, uint32_t cols,
                                                               uint32_t first, uint32_t items, uint32_t rows, RowSumScratch s) {
  const uint32_t per_row = cols / VEC;
  if (rows > kInlineRows) list_heavy_destinations(first, items / per_row, rows, s);
  for (uint32_t i = blockIdx.x * kRowThreads + threadIdx.x; i < items; i += gridDim.x * kRowThreads) {
    const uint32_t d = first + i / per_row, col = i % per_row * VEC;
    const int count = s.count[d];
    const int32_t* slots = s.slots + (uint64_t)d * kInlineRows;
    float sum[VEC];
#pragma unroll
    for (int e = 0; e < VEC; ++e) sum[e] = 0.0f;
    if (count <= 8) {
      sum_few_rows<DT, VEC, 8>(src, slots, count, cols, col, sum);
    } else if (count <= kInlineRows) {
      sum_few_rows<DT, VEC, kInlineRows>(src, slots, count, cols, col, sum);
    } else {
      continue;
    }
    Halves<VEC> out;
#pragma unroll
    for (int e = 0; e < VEC; ++e) out.v[e] = narrow<DT>(sum[e]);
    *reinterpret_cast<Halves<VEC>*>(dst + (uint64_t)d * cols + col) = out;
  }
}

__global__ __launch_bounds__(kRowThreads) void list_heavy_rows_kernel(const int32_t* row_index, uint32_t rows, RowSumScratch s) {
  if (s.cursor[kRestUsed] == 0) return;
  for (uint32_t r = blockIdx.x * kRowThreads + threadIdx.x; r < rows; r += gridDim.x * kRowThreads) {
    const int at = s.arrival[r];
    if (at >= kInlineRows) s.rest[s.base[row_index[r]] + at - kInlineRows] = (int32_t)r;
  }
}

// The heavy destinations, eight loads in flight per thread.  Which rows a thread adds, and in which order,
// depends on the index alone.
//
// Up to kWaveRows rows: a wave takes 64 column items; each lane holds a row, counts the rows below it and
// hands it to the lane of that number.
//
// More rows: a workgroup takes ITEMS column items, its PARTS groups of ITEMS threads a share of the rows each,
// and the groups' sums are added up in order at the end.  Up to kListedRows rows are sorted in LDS (a thread
// counts the rows below its own) and dealt to the groups in turn.  Of more rows, those of a window of the
// index are marked in a bitmap in LDS, and the groups take its words (rows 32 w .. 32 w + 31) in turn.
template <int ITEMS>
struct HeavyTask {
  static constexpr int PARTS = kRowThreads / ITEMS;
  uint32_t d, slice, item, part;
  int count;
  __device__ __forceinline__ HeavyTask(uint32_t d_, uint32_t slice_, int count_)
      : d(d_), slice(slice_), item(slice_ * ITEMS + threadIdx.x % ITEMS), part(threadIdx.x / ITEMS), count(count_) {}
};
constexpr int kListedItems = 32, kLongItems = 4;
constexpr uint32_t kWindowWords = 4096, kWindowRows = 32 * kWindowWords;

template <int DT, int VEC>
struct HeavySum {
  static constexpr int IN_FLIGHT = 8;
  using V = Halves<VEC>;
  const uint16_t* src;
  uint16_t* dst;
  uint32_t cols;
  float sum[VEC];

  __device__ __forceinline__ void clear() {
#pragma unroll
    for (int e = 0; e < VEC; ++e) sum[e] = 0.0f;
  }
  __device__ __forceinline__ void add(const uint32_t* row, int have, uint32_t item) {
    V v[IN_FLIGHT];
#pragma unroll
    for (int k = 0; k < IN_FLIGHT; ++k)
      if (k < have) v[k] = *reinterpret_cast<const V*>(src + (uint64_t)row[k] * cols + item * VEC);
#pragma unroll
    for (int k = 0; k < IN_FLIGHT; ++k)
      if (k < have)
#pragma unroll
        for (int e = 0; e < VEC; ++e) sum[e] += widen<DT>(v[k].v[e]);
  }
  // The groups' sums in order, through `words`; ends with a barrier.
  template <int ITEMS>
  __device__ __forceinline__ void finish(const HeavyTask<ITEMS>& t, uint32_t* words) {
    constexpr int WIDTH = ITEMS * VEC, PARTS = HeavyTask<ITEMS>::PARTS;
    static_assert(kWindowWords >= PARTS * WIDTH && WIDTH <= kRowThreads, "");
    float* parts = reinterpret_cast<float*>(words);
    const int tid = threadIdx.x;
#pragma unroll
    for (int e = 0; e < VEC; ++e) parts[t.part * WIDTH + tid % ITEMS * VEC + e] = sum[e];
    __syncthreads();
    const uint32_t col = t.slice * WIDTH + tid;
    if (tid < WIDTH && col < cols) {
      float all = 0.0f;
#pragma unroll
      for (int k = 0; k < PARTS; ++k) all += parts[k * WIDTH + tid];
      dst[(uint64_t)t.d * cols + col] = narrow<DT>(all);
    }
    __syncthreads();
  }
};

template <int DT, int VEC>
__global__ __launch_bounds__(kRowThreads, 4) void sum_heavy_rows_kernel(const uint16_t* src, uint16_t* dst, uint32_t cols,
                                                                        uint32_t rows, RowSumScratch s) {
  using Sum = HeavySum<DT, VEC>;
  constexpr int IN_FLIGHT = Sum::IN_FLIGHT;
  __shared__ __attribute__((aligned(16))) uint32_t words[kWindowWords];
  static_assert(kWindowWords >= 2 * kListedRows, "");
  const int tid = threadIdx.x;
  const uint32_t per_row = cols / VEC;
  const int64_t most = most_heavy(rows);
  Sum sum{src, dst, cols};
  // the rows of destination d, in the order the device met them
  auto row_at = [&](uint32_t d, int base, int i) -> uint32_t {
    return i < kInlineRows ? s.slots[(uint64_t)d * kInlineRows + i] : s.rest[base + i - kInlineRows];
  };

  const uint32_t lane = tid & 63, groups = (per_row + 63) / 64;
  const uint64_t wave_tasks = (uint64_t)s.cursor[kHeavyWave] * groups;
  for (uint64_t task = blockIdx.x * (kRowThreads / 64) + tid / 64; task < wave_tasks; task += gridDim.x * (kRowThreads / 64)) {
    const uint32_t d = s.heavy[task / groups], item = (uint32_t)(task % groups) * 64 + lane;
    const int count = s.count[d];
    const int mine = (int)lane < count ? (int)row_at(d, s.base[d], lane) : 0x7fffffff;
    int below = 0;
    for (int k = 0; k < count; ++k) below += __shfl(mine, k) < mine ? 1 : 0;
    const int sorted = __builtin_amdgcn_ds_permute(4 * ((int)lane < count ? below : (int)lane), mine);
    sum.clear();
    for (int at = 0; at < count; at += IN_FLIGHT) {
      uint32_t row[IN_FLIGHT];
#pragma unroll
      for (int k = 0; k < IN_FLIGHT; ++k) row[k] = (uint32_t)__shfl(sorted, at + k);   // (past the count: not used)
      if (item < per_row) sum.add(row, min(IN_FLIGHT, count - at), item);
    }
    if (item >= per_row) continue;
    Halves<VEC> out;
#pragma unroll
    for (int e = 0; e < VEC; ++e) out.v[e] = narrow<DT>(sum.sum[e]);
    *reinterpret_cast<Halves<VEC>*>(dst + (uint64_t)d * cols + item * VEC) = out;
  }

  // (from here on every thread of a workgroup has the same tasks)
  const uint32_t listed_slices = (per_row + kListedItems - 1) / kListedItems;
  const uint64_t listed_tasks = (uint64_t)s.cursor[kHeavyListed] * listed_slices;
  for (uint64_t task = blockIdx.x; task < listed_tasks; task += gridDim.x) {
    const uint32_t d = s.heavy[most + (int64_t)(task / listed_slices)];
    const HeavyTask<kListedItems> t(d, (uint32_t)(task % listed_slices), s.count[d]);
    const int base = s.base[d];
    uint32_t *listed = words, *sorted = words + kListedRows;
    for (int i = tid; i < (t.count + 3) / 4 * 4; i += kRowThreads) listed[i] = i < t.count ? row_at(d, base, i) : ~0u;
    __syncthreads();
    for (int i = tid; i < t.count; i += kRowThreads) {
      const uint32_t mine = listed[i];
      int below = 0;
      for (int k = 0; k < t.count; k += 4) {
        const u32x4 other = *reinterpret_cast<const u32x4*>(listed + k);
        below += (other[0] < mine) + (other[1] < mine) + (other[2] < mine) + (other[3] < mine);
      }
      sorted[below] = mine;
    }
    __syncthreads();
    sum.clear();
    for (int at = t.part; at < t.count && t.item < per_row; at += t.PARTS * IN_FLIGHT) {
      uint32_t row[IN_FLIGHT];
      int have = 0;
#pragma unroll
      for (int k = 0; k < IN_FLIGHT; ++k)
        if (at + k * t.PARTS < t.count) row[k] = sorted[at + k * t.PARTS], have = k + 1;
      sum.add(row, have, t.item);
    }
    __syncthreads();   // (the sums go where the rows are)
    sum.finish(t, words);
  }

  const uint32_t long_slices = (per_row + kLongItems - 1) / kLongItems;
  const uint64_t long_tasks = (uint64_t)s.cursor[kHeavyLong] * long_slices;
  for (uint64_t task = blockIdx.x; task < long_tasks; task += gridDim.x) {
    const uint32_t d = s.heavy[2 * most - 1 - (int64_t)(task / long_slices)];
    const HeavyTask<kLongItems> t(d, (uint32_t)(task % long_slices), s.count[d]);
    const int base = s.base[d];
    sum.clear();
    for (uint32_t first = 0; first < rows; first += kWindowRows) {
      const uint32_t used = min(kWindowWords, (rows - first + 31) / 32);
      for (uint32_t w = tid; w < used; w += kRowThreads) words[w] = 0;
      __syncthreads();
      for (uint32_t i = tid; i < (uint32_t)t.count; i += kRowThreads * IN_FLIGHT) {
        uint32_t at[IN_FLIGHT];
#pragma unroll
        for (int k = 0; k < IN_FLIGHT; ++k)   // (rows ahead of the window, and no rows: far past its end)
          at[k] = i + k * kRowThreads < (uint32_t)t.count ? row_at(d, base, (int)(i + k * kRowThreads)) - first : ~0u;
#pragma unroll
        for (int k = 0; k < IN_FLIGHT; ++k)
          if (at[k] < kWindowRows) atomicOr(&words[at[k] / 32], 1u << (at[k] % 32));
      }
      __syncthreads();
      uint32_t w = t.part, bits = w < used ? words[w] : 0;
      while (w < used && t.item < per_row) {
        uint32_t row[IN_FLIGHT];
        int have = 0;
#pragma unroll
        for (int k = 0; k < IN_FLIGHT; ++k) {
          while (bits == 0 && w < used) {
            w += t.PARTS;
            bits = w < used ? words[w] : 0;
          }
          if (bits != 0) {
            row[k] = first + w * 32 + (__ffs(bits) - 1), have = k + 1;
            bits &= bits - 1;
          }
        }
        sum.add(row, have, t.item);
      }
      __syncthreads();
    }
    sum.finish(t, words);
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

// Workgroups of the kernel for heavy destinations, at most: four per compute unit.
constexpr int64_t kHeavyBlocks = 1024;

template <int DT, int VEC>
hipError_t launch_sum_rows(const uint16_t* src, uint16_t* dst, int64_t rows, int64_t destinations, int64_t cols,
                           const int32_t* row_index, const RowSumScratch& s, hipStream_t stream) {
  const int64_t per_row = cols / VEC, slab = (int64_t(1) << 30) / per_row;
  for (int64_t first = 0; first < destinations; first += slab) {
    const uint32_t items = (uint32_t)((destinations - first < slab ? destinations - first : slab) * per_row);
    hipLaunchKernelGGL((sum_rows_kernel<DT, VEC>), dim3(row_blocks(items)), dim3(kRowThreads), 0, stream, src, dst,
                       (uint32_t)cols, (uint32_t)first, items, (uint32_t)rows, s);
    const hipError_t err = hipGetLastError();
    if (err != hipSuccess) return err;
  }
  if (most_heavy(rows) == 0) return hipSuccess;
  hipLaunchKernelGGL(list_heavy_rows_kernel, dim3(row_blocks((uint32_t)rows)), dim3(kRowThreads), 0, stream, row_index,
                     (uint32_t)rows, s);
  hipError_t err = hipGetLastError();
  if (err != hipSuccess) return err;
  const int64_t tasks = most_heavy(rows) * ((per_row + kLongItems - 1) / kLongItems);   // no fewer than there can be
  hipLaunchKernelGGL((sum_heavy_rows_kernel<DT, VEC>), dim3(tasks < kHeavyBlocks ? (uint32_t)tasks : (uint32_t)kHeavyBlocks),
                     dim3(kRowThreads), 0, stream, src, dst, (uint32_t)cols, (uint32_t)rows, s);
  return hipGetLastError();
}

int access_width(uintptr_t bits) {   // elements per access that divide every address and pitch in `bits`
  int vec = 8;
  while (vec > 1 && (bits & (uintptr_t)(2 * vec - 1))) vec >>= 1;
  return vec;
}

}  // namespace

uint64_t sum_rows_scratch_bytes(int64_t rows, int64_t destinations) {
  return (uint64_t)(destinations * (2 + kInlineRows) + kCursorWords + 2 * rows + 2 * most_heavy(rows)) * sizeof(int32_t);
}

hipError_t sum_rows(const void* src, const int32_t* row_index, void* dst, int64_t rows, int64_t destinations,
                    int64_t cols, int dt, void* scratch, hipStream_t stream) {
  RowSumScratch s;
  s.count = static_cast<int32_t*>(scratch);
  s.cursor = s.count + destinations;
  s.slots = s.cursor + kCursorWords;
  s.base = s.slots + destinations * kInlineRows;
  s.arrival = s.base + destinations;
  s.rest = s.arrival + rows;
  s.heavy = s.rest + rows;
  const uint64_t words = (uint64_t)destinations + kCursorWords;
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
#define GG_LAUNCH(V)                                                                                  \
  (dt == kBF16 ? &launch_sum_rows<kBF16, V> : &launch_sum_rows<kF16, V>)(                             \
      static_cast<const uint16_t*>(src), static_cast<uint16_t*>(dst), rows, destinations, cols, row_index, s, stream)
  switch (vec) {
    case 8: return GG_LAUNCH(8);
    case 4: return GG_LAUNCH(4);
    case 2: return GG_LAUNCH(2);
    default: return GG_LAUNCH(1);
  }
#undef GG_LAUNCH
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

// Batches whose rows, `rows` each, are numbered in 32 bits together: what one launch may cover.
int64_t batches_of_a_launch(int64_t batches, int64_t rows) {
  const int64_t most = ((int64_t(1) << 32) - 1) / rows;
  return batches < most ? batches : most;
}

template <typename T>
hipError_t launch_pad_rows(const T* src, T* dst, int64_t batches, int64_t src_rows, int64_t src_cols, int64_t dst_rows,
                           int64_t dst_cols, hipStream_t stream) {
  const int64_t per_row = dst_cols / (16 / (int64_t)sizeof(T)), together = batches_of_a_launch(batches, dst_rows);
  // (32-bit item numbers: larger tensors go in slabs of rows)
  const int64_t slab = (int64_t(1) << 30) / per_row;
  for (int64_t batch = 0; batch < batches; batch += together) {
    const int64_t rows = (batches - batch < together ? batches - batch : together) * dst_rows;
    for (int64_t first = 0; first < rows; first += slab) {
      const uint32_t items = (uint32_t)((rows - first < slab ? rows - first : slab) * per_row);
      hipLaunchKernelGGL((pad_rows_kernel<T>), dim3(row_blocks(items)), dim3(kRowThreads), 0, stream,
                         src + batch * src_rows * src_cols, dst + batch * dst_rows * dst_cols, (uint32_t)src_rows,
                         (uint32_t)src_cols, (uint32_t)dst_rows, (uint32_t)dst_cols, (uint32_t)first, items);
      const hipError_t err = hipGetLastError();
      if (err != hipSuccess) return err;
    }
  }
  return hipSuccess;
}

template <typename T>
hipError_t launch_unpad_rows(const T* src, T* dst, int64_t batches, int64_t src_rows, int64_t src_cols, int64_t dst_rows,
                             int64_t dst_cols, hipStream_t stream) {
  constexpr int64_t VEC = 16 / sizeof(T), SLAB = int64_t(1) << 30;
  const int64_t together = batches_of_a_launch(batches, dst_rows);
  for (int64_t batch = 0; batch < batches; batch += together) {
    const int64_t total = (batches - batch < together ? batches - batch : together) * dst_rows * dst_cols;
    for (int64_t first = 0; first < total; first += SLAB) {
      const int64_t count = total - first < SLAB ? total - first : SLAB;
      const int64_t row = first / dst_cols;
      T* to = dst + batch * dst_rows * dst_cols + first;
      const int64_t head = (int64_t)(reinterpret_cast<uintptr_t>(to) % 16 / sizeof(T));
      const uint32_t items = (uint32_t)((head + count + VEC - 1) / VEC);
      hipLaunchKernelGGL((unpad_rows_kernel<T>), dim3(row_blocks(items)), dim3(kRowThreads), 0, stream,
                         src + batch * src_rows * src_cols, to, (uint32_t)src_rows, (uint32_t)src_cols, (uint32_t)dst_rows,
                         (uint32_t)dst_cols, (uint32_t)row, (uint32_t)(first - row * dst_cols), (uint32_t)head,
                         (uint32_t)count, items);
      const hipError_t err = hipGetLastError();
      if (err != hipSuccess) return err;
    }
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
