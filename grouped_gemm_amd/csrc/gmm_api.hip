// Host side of the C ABI declared in include/grouped_gemm_hip.h: argument checks,
// kernel selection and the launches.  No torch types, no allocation, no sync.
#include "../../include/grouped_gemm_hip.h"

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdarg>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <mutex>
#include <numeric>

#include "gmm_generic.hpp"
#include "gmm_variants.hpp"
#include "row_kernels.hpp"

namespace gg {
const GenericOps* generic_ops_0();
const GenericOps* generic_ops_1();
const GenericOps* generic_ops_2();
const GenericOps* generic_ops_3();
#define GG_VARIANT(index, DT_, LAYOUT_, SHAPE_, EPI_, INDEXED_) const VariantOps* variant_ops_##index();
#define GG_PAIR(index, DT_, LAYOUT_, SHAPE1_, SHAPE2_) const PairOps* pair_ops_##index();
#include "gmm_variants.def"
#undef GG_VARIANT
#undef GG_PAIR
}  // namespace gg

namespace {

using gg::Short;
using gg::Small;
using gg::SmallSquare;
using gg::Wide;
using gg::ShortRaggedDepth;
using gg::SmallRaggedDepth;
using gg::WideRaggedDepth;

thread_local char g_err[512] = "";

int fail(int code, const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_err, sizeof(g_err), fmt, ap);
  va_end(ap);
  return code;
}

#define GG_HIP(call)                                                                     \
  do {                                                                                   \
    hipError_t err__ = (call);                                                           \
    if (err__ != hipSuccess)                                                             \
      return fail(GG_EHIP, "%s failed: %s", #call, hipGetErrorString(err__));            \
  } while (0)

const gg::VariantOps* (*const kVariantGetters[])() = {
#define GG_VARIANT(index, DT_, LAYOUT_, SHAPE_, EPI_, INDEXED_) &gg::variant_ops_##index,
#include "gmm_variants.def"
#undef GG_VARIANT
};
const gg::PairOps* (*const kPairGetters[])() = {
#define GG_VARIANT(index, DT_, LAYOUT_, SHAPE_, EPI_, INDEXED_)
#define GG_PAIR(index, DT_, LAYOUT_, SHAPE1_, SHAPE2_) &gg::pair_ops_##index,
#include "gmm_variants.def"
#undef GG_VARIANT
#undef GG_PAIR
};
constexpr int kNumPairs = sizeof(kPairGetters) / sizeof(kPairGetters[0]);
constexpr int kNumVariants = sizeof(kVariantGetters) / sizeof(kVariantGetters[0]);

static_assert(GG_DTYPE_BF16 == gg::kBF16 && GG_DTYPE_F16 == gg::kF16 && GG_DTYPE_F8E4M3 == gg::kF8E4M3 &&
              GG_DTYPE_F8E5M2 == gg::kF8E5M2, "the header's element types are the kernels'");

const gg::GenericOps* generic_ops(int dt) {
  switch (dt) {
    case gg::kBF16: return gg::generic_ops_0();
    case gg::kF16: return gg::generic_ops_1();
    case gg::kF8E4M3: return gg::generic_ops_2();
    default: return gg::generic_ops_3();
  }
}

const gg::VariantOps* find_variant(int dt, int layout, int shape, int epilogue, int indexed) {
  for (int i = 0; i < kNumVariants; ++i) {
    const gg::VariantOps* v = kVariantGetters[i]();
    if (v->dt == dt && v->layout == layout && v->shape == shape && v->epilogue == epilogue &&
        v->indexed == indexed)
      return v;
  }
  return nullptr;
}

const gg::PairOps* find_pair(int dt, int layout, int shape1, int shape2) {
  for (int i = 0; i < kNumPairs; ++i) {
    const gg::PairOps* v = kPairGetters[i]();
    if (v->dt == dt && v->layout == layout && v->shape1 == shape1 && v->shape2 == shape2) return v;
  }
  return nullptr;
}

// Tile rows per band of the in-group tile order.  The weight-gradient layout with shallow groups
// is mostly output writes; there an odd band height measures 5-8 % faster than 4 (the bands then
// do not line up with the 32-tile runs the XCDs take, which spreads what is written at one time
// over more of the memory channels).
constexpr int kBandHeight = 4;
constexpr int kBandHeightShallow = 3;
constexpr int kShallowBelow = 1024;   // average rows per group below which the shallow height is used
constexpr int kShortBelow = 112;      // average rows per group below which the short tile shape is used

int band_height(int64_t num_groups, int64_t tokens, int trans_a) {
  return trans_a && tokens < (int64_t)kShallowBelow * num_groups ? kBandHeightShallow : kBandHeight;
}

bool use_short_shape(int64_t num_groups, int64_t tokens, int trans_a) {
  return !trans_a && num_groups > 0 && tokens < (int64_t)kShortBelow * num_groups;
}

// NN and NT layouts: whether the groups' tiles are handed out by ascending number of tile rows
// instead of in group order (the kernel still keeps the group order if it finds a group of more
// than 8 tile rows).  Where group sizes straddle a multiple of the tile height, groups of k and of
// k + 1 tile rows alternate at random; with equal groups side by side the launch is faster.
// Measured by permuting the groups, Poisson sizes, 7168 -> 2048, b stored transposed / as stored:
// 256 groups around 256 rows -3.2 / -2.3 %, 96 around 256 -4.8 / -3.6 %, 128 around 512 -1.8 /
// -2.2 %, around 768 -3.3 / -3.4 %, 64 around 1024 -1.2 / -1.6 %; around 128, 200, 320, 384, 640,
// 1536, 2048 rows within +-0.7 %; Zipf sizes with groups of up to 57 tile rows +0.8 / +1.7 %
// (hence the kernel's guard).  It pays with deep tiles only: the same 256 groups around 256 rows
// with hidden_in 4096 -2.6 / -1.9 %, 2048 +0.6 / -1.4 %, 1024 +1.6 / +0.7 %, 512 +8.9 / +7.4 %
// (the order itself, a counting sort and a second scan of the tile counts, is 5-8 us of a launch
// of 200 us there).
constexpr int kByTileRowsGroups = 32;         // at least this many groups
constexpr int kByTileRowsRowsBelow = 2048;    // ... of fewer rows than this on average
constexpr int kByTileRowsRounds = 4;          // ... at least this many rounds of tiles
constexpr int kByTileRowsDepth = 2048;        // ... and tiles at least this deep

bool order_by_tile_rows(int64_t num_groups, int64_t tokens, int64_t tiles_n, int bm, int grid, int64_t hidden_in) {
  return num_groups >= kByTileRowsGroups && tokens < (int64_t)kByTileRowsRowsBelow * num_groups &&
         hidden_in >= kByTileRowsDepth &&
         (tokens / bm + num_groups / 2) * tiles_n >= (int64_t)kByTileRowsRounds * grid;
}

// Whether the output goes out through L2 (kStoreMerging) instead of past it: where its rows do not start on
// 64-byte boundaries, so that stores meet inside sectors, and where the launch is bound by them.  Us per launch, past
// L2 / through it.  Weight gradients always are: 32 x 128 rows, 776 x 1032: 39.9 / 26.9; 64 x 128, 1032 x
// 2040: 174 / 104; 128 x 4, 2040 x 2040 (1.07 GB): 662 / 278; 8 x 2048, 2040 x 4088: 233 / 229; 32 x 128, 264 x 392: 12.5 / 13.0.
// Other layouts only if shallow and with many rows to a group, as L2 then does not hold what other tiles share, and
// what is left in it at the end of a launch is written then: 32 x 2048 rows, 392 -> 520: 72.8 / 61.7; 8 x
// 1024, 1048 -> 2040: 58.9 / 52.0; 32 x 512, 1000 -> 1000: 52.5 / 50.7; 64 x 128, 1000 -> 2000: 58.7 / 64.6; 8 x 2048, 2040 -> 4088:
// 254 / 265.  (Rows that do start there: 64 x 128, 1024 x 2048: 70 / 90.)
constexpr int64_t kShallowProduct = 1536;
bool merge_stores(const gg_gmm_args& g) {
  if ((reinterpret_cast<uintptr_t>(g.c) | (uint64_t)g.hidden_out * 2) % 64 == 0 || g.accumulate_f32) return false;
  return g.trans_a || (g.hidden_in <= kShallowProduct && 2 * g.tokens >= g.hidden_in * g.num_groups);
}

// Scratch of gg_gmm_no_alloc: the workspace of gg_gmm (arrival counters, then partial tiles) as a
// static array, one copy per device that loads this library, held until the process ends.  In
// host code `scratch` is only a handle for hipGetSymbolAddress; kernels get the address that
// call returns for the current device (DeviceInfo::scratch).
static __device__ __align__(256) unsigned char scratch[GG_WORKSPACE_BYTES];

// Most workgroups a launch may have for the static scratch to hold one partial tile each.
constexpr int kStaticScratchGrid = (GG_WORKSPACE_BYTES - gg::kWsCounterBytes) / (256 * 256 * 4);

// gg_size_status_word: zero when the library is loaded.
static __device__ int32_t size_status_word;

__global__ void clear_counters_kernel(int* counters) { counters[threadIdx.x] = 0; }

struct DeviceInfo {
  int cus = 0;
  bool ok = false;
  unsigned char* scratch = nullptr;   // device addresses of `scratch` and `size_status_word` on this device
  int32_t* size_status = nullptr;
};

// Per device, once: the architecture check and the LDS limit of every kernel variant.
int device_info(DeviceInfo* out) {
  static DeviceInfo cache[64];
  static std::mutex mu;
  int dev = 0;
  GG_HIP(hipGetDevice(&dev));
  if (dev < 0 || dev >= 64) return fail(GG_ELIMIT, "device index %d not supported", dev);
  std::lock_guard<std::mutex> lock(mu);
  if (!cache[dev].ok) {
    hipDeviceProp_t prop;
    GG_HIP(hipGetDeviceProperties(&prop, dev));
    if (strncmp(prop.gcnArchName, "gfx950", 6) != 0)
      return fail(GG_EHIP, "this library is built for gfx950 only, device is %s", prop.gcnArchName);
    for (int i = 0; i < kNumVariants; ++i) GG_HIP(kVariantGetters[i]()->prepare());
    for (int i = 0; i < kNumPairs; ++i) GG_HIP(kPairGetters[i]()->prepare());
    void* scratch_address = nullptr;
    GG_HIP(hipGetSymbolAddress(&scratch_address, HIP_SYMBOL(scratch)));
    void* status_address = nullptr;
    GG_HIP(hipGetSymbolAddress(&status_address, HIP_SYMBOL(size_status_word)));
    cache[dev].scratch = static_cast<unsigned char*>(scratch_address);
    cache[dev].size_status = static_cast<int32_t*>(status_address);
    cache[dev].cus = prop.multiProcessorCount;
    cache[dev].ok = true;
  }
  *out = cache[dev];
  return GG_OK;
}

template <typename S, int LAYOUT>
int launch_dump(const gg::GmmParams& p, const gg::HostSizes& hs, hipStream_t stream) {
  hipLaunchKernelGGL((gg::schedule_dump_kernel<LAYOUT, S::BM, S::BN>), dim3(1), dim3(64), 0, stream, p, hs);
  GG_HIP(hipGetLastError());
  return GG_OK;
}

int dispatch_dump(bool short_shape, int layout, const gg::GmmParams& p, const gg::HostSizes& hs,
                  hipStream_t stream) {
  if (layout == gg::kTN) return launch_dump<Wide, gg::kTN>(p, hs, stream);
  if (short_shape) {
    return layout == gg::kNN ? launch_dump<Short, gg::kNN>(p, hs, stream)
                             : launch_dump<Short, gg::kNT>(p, hs, stream);
  }
  return layout == gg::kNN ? launch_dump<Wide, gg::kNN>(p, hs, stream)
                           : launch_dump<Wide, gg::kNT>(p, hs, stream);
}

int check_common(const int64_t* batch_sizes, int64_t num_groups, int64_t tokens, int64_t hidden_in,
                 int64_t hidden_out, int trans_a, int trans_b) {
  if (trans_a && trans_b) return fail(GG_EINVAL, "trans_a and trans_b cannot both be set");
  if (num_groups < 0 || tokens < 0 || hidden_in < 0 || hidden_out < 0)
    return fail(GG_EINVAL, "negative dimension");
  if (num_groups > 0 && batch_sizes == nullptr) return fail(GG_EINVAL, "batch_sizes is null");
  if (hidden_in >= (1 << 22) || hidden_out >= (1 << 22))
    return fail(GG_ELIMIT, "hidden sizes must be below 2^22");
  if (tokens >= (int64_t(1) << 31)) return fail(GG_ELIMIT, "tokens must be below 2^31");
  return GG_OK;
}

// Which kernels a call runs on, from its sizes, element type and the operands' alignment.
struct Route {
  uintptr_t address_bits;
  int elem_bytes;
  bool indexed;        // any row index given
  bool indexed_fits;   // ... and a and c are within reach of the streaming kernels' 32-bit offsets
  bool relaxed;        // streaming kernel on operands that are only 4-byte aligned (see classify)
  bool ragged_width;   // ... with a width that is not a multiple of 8
  bool ragged_depth;   // ... with rows along a depth that is not a multiple of 8
  bool generic;        // the kernels of gmm_generic.hpp
  int vec;             // their vector width
  int64_t a_bytes, c_bytes;
};

Route classify(const gg_gmm_args& g) {
  Route r;
  const int64_t hidden_in = g.hidden_in, hidden_out = g.hidden_out, tokens = g.tokens;
  const bool trans_a = g.trans_a != 0, trans_b = g.trans_b != 0;
  const bool swiglu = g.epilogue == GG_EPILOGUE_SWIGLU;
  r.elem_bytes = g.dtype == GG_DTYPE_F8E4M3 || g.dtype == GG_DTYPE_F8E5M2 ? 1 : 2;
  r.address_bits =
      reinterpret_cast<uintptr_t>(g.a) | reinterpret_cast<uintptr_t>(g.b) | reinterpret_cast<uintptr_t>(g.c);
  // The streaming kernels fetch and store rows 16 bytes at a time: two-byte elements, hidden sizes
  // that are multiples of 8, operands on 16-byte boundaries, rows in place.  Everything else goes
  // to the kernels of gmm_generic.hpp, VEC elements at a time.
  r.indexed = g.a_row_index != nullptr || g.b_row_index != nullptr || g.c_row_index != nullptr;
  r.a_bytes = (g.a_num_rows > 0 ? g.a_num_rows : tokens) * hidden_in * r.elem_bytes;
  r.c_bytes = (g.c_num_rows > 0 ? g.c_num_rows : tokens) * hidden_out * 2;
  // with row indices the streaming kernels address a and c through 32-bit byte offsets
  r.indexed_fits = !trans_a && r.a_bytes < (int64_t)gg::kOutOfRangeIndexed && r.c_bytes < (int64_t)gg::kOutOfRangeIndexed;
  // (fp8 streams in 16-byte chunks like the rest: 16 elements, along whichever dimension is
  // contiguous in each operand)
  const bool f8_streams = r.elem_bytes == 1 && (!swiglu || (trans_b && !r.indexed)) &&
                          (trans_a ? hidden_in % 16 == 0 && hidden_out % 16 == 0
                                   : hidden_in % 16 == 0 && (trans_b || hidden_out % 16 == 0));
  // Two-byte elements with the plain store epilogue also stream from 4-byte boundaries: a 16-byte
  // access needs no more than that, and the end of a buffer descriptor clips it dword by dword.
  // Both hidden sizes have to be even (rows then start on 4-byte boundaries).  Along the width a
  // chunk may run past the row's end: what it picks up there lands in tile columns that are never
  // stored, and a row of c whose last chunk holds 2, 4 or 6 columns is finished with narrower
  // stores.  Along the depth (rows of a, and of b stored transposed; not in the weight-gradient
  // layout, where both operands run along their widths) such a chunk would add the next row's
  // first values to the sums: a kernel variant clears them in LDS before the slice is multiplied
  // (WideRaggedDepth and its like; plain rows only, no row indices).
  const bool aligned = hidden_in % 8 == 0 && hidden_out % 8 == 0 && (r.address_bits & 15) == 0;
  r.relaxed = !aligned && r.elem_bytes == 2 && !swiglu && !g.accumulate_f32 && (r.address_bits & 3) == 0 &&
              hidden_out % 2 == 0 && hidden_in % 2 == 0;
  r.ragged_width = r.relaxed && hidden_out % 8 != 0;
  r.ragged_depth = !trans_a && hidden_in % 8 != 0;
  if (r.ragged_depth && r.indexed) r.relaxed = false;
  r.ragged_depth = r.ragged_depth && r.relaxed;
  r.generic = !r.relaxed &&
              ((r.elem_bytes != 2 && !f8_streams) || hidden_in % 8 != 0 || hidden_out % 8 != 0 ||
               (r.address_bits & 15));
  r.generic = r.generic || (r.indexed && !r.indexed_fits);
  r.vec = 8;
  if (r.generic) {
    while (r.vec > 1 && (hidden_in % r.vec != 0 || hidden_out % r.vec != 0 ||
                         (r.address_bits & (uintptr_t)(r.vec * 2 - 1))))
      r.vec >>= 1;
  }
  return r;
}

// gg_gmm_strided: rows of a and b on 16-byte boundaries, further apart than they are long.
struct Strides {
  int64_t a, b;
};

bool strides_fit(const gg_gmm_args& g, const Strides& s) {
  if (g.dtype != GG_DTYPE_BF16 && g.dtype != GG_DTYPE_F16) return false;
  if (g.epilogue != GG_EPILOGUE_NONE || g.accumulate_f32 || g.a_row_index || g.b_row_index || g.c_row_index) return false;
  if ((reinterpret_cast<uintptr_t>(g.a) | reinterpret_cast<uintptr_t>(g.b)) & 15) return false;
  const int64_t b_row = g.trans_b ? g.hidden_in : g.hidden_out;
  // (whole chunks of 8: what a chunk reads past the end of a row is its padding)
  return s.a % 8 == 0 && s.b % 8 == 0 && s.a >= g.hidden_in && s.b >= b_row && s.a < (1 << 22) && s.b < (1 << 22);
}

Route strided_route(const gg_gmm_args& g) {
  gg_gmm_args aligned = g;   // (the streaming kernels' route, whatever the sizes and c)
  aligned.hidden_in = (g.hidden_in + 7) / 8 * 8;
  aligned.hidden_out = (g.hidden_out + 7) / 8 * 8;
  aligned.c = reinterpret_cast<void*>((reinterpret_cast<uintptr_t>(g.c) + 15) / 16 * 16);
  Route r = classify(aligned);
  r.address_bits = (r.address_bits & ~(uintptr_t)15) | (reinterpret_cast<uintptr_t>(g.c) & 15);
  return r;
}

// Rows of a, b and c in memory, the bounds a row index is held against: an index that names no
// row is a missing row (zeros on the way in, nothing stored on the way out) on every kernel.
struct IndexedRows {
  int64_t a, b, c;
};

IndexedRows indexed_rows(const gg_gmm_args& g) {
  IndexedRows r;
  r.a = g.a_num_rows > 0 ? g.a_num_rows : g.tokens;
  r.b = g.b_num_rows > 0 ? g.b_num_rows : g.tokens;
  r.c = g.c_num_rows > 0 ? g.c_num_rows : g.tokens;
  return r;
}

struct TileShape {
  int id, bm, bn;
};
template <typename S>
constexpr TileShape shape_of() {
  return TileShape{S::kId, S::BM, S::BN};
}

// Tiles of a call in a shape, as far as that can be told without the sizes, which may be on the
// device only.  Groups are ragged: each has on average half a tile row more than its rows fill (groups of
// 64 rows on average are as often 65 and more, two rows of 64 x 128 tiles, as 64 and fewer).
int64_t expected_tiles(const gg_gmm_args& g, int bm, int bn) {
  const int64_t tiles_n = (g.hidden_out + bn - 1) / bn;
  if (g.trans_a) return g.num_groups * ((g.hidden_in + bm - 1) / bm) * tiles_n;
  const int64_t tile_rows = (2 * g.tokens / bm + g.num_groups) / 2;
  return (tile_rows > g.num_groups ? tile_rows : g.num_groups) * tiles_n;
}

// Workgroups of a full launch of one workgroup per compute unit, for the rules below.
constexpr int kFullLaunch = 256;

// Whether the streaming kernel exists in a shape: the short and the small ones for two-byte elements
// and, with b stored transposed and the plain epilogue, fp8.
bool has_shape(const gg_gmm_args& g, const Route& r, int id) {
  const bool plain = g.epilogue == GG_EPILOGUE_NONE && !r.indexed;
  if (g.trans_a) return id == Wide::kId || (id == SmallSquare::kId && r.elem_bytes == 2);
  return id == Wide::kId || ((id == Short::kId || id == Small::kId) && (r.elem_bytes == 2 || (g.trans_b && plain)));
}

// The tile shape of a streaming call.
//
// NN and NT layouts: small tiles up to one and a half of them per compute unit (one for deep
// products, whose tiles suffer most from sharing): such a launch is bound by how long one tile takes,
// and by how many compute units pull data.  Short tiles where
// one round of them holds the launch, where groups average few rows (use_short_shape), and where few
// rows of deep products leave nothing to do but pull weights, for which their larger buffers are
// better than small tiles' (8 x 16, 14336 -> 4096, 128 short tiles in two depth pieces each: 152 us, 256
// small ones: 172 us).  Us per launch, bf16, NN layout, row counts drawn at random around the average,
// wide / short / small, and the expected number of small and of short tiles: 29 x 238 rows, 280 -> 152
// (244, 68): 11.8 / 10.6 / 9.5; 4 x 512, 512 -> 1024 (272, 72): 13.0 / 12.2 / 11.6; 8 x 700, 512 -> 512 (364, 94):
// 13.4 / 12.5 / 11.9; 16 x 200, 3072 -> 768 (348, 99): 38.3 / 32.8 / 35.3; 32 x 128, 2048 -> 768 (480, 144): 30.4 /
// 29.8 / 32.7; 16 x 256, 2048 -> 1024 (576, 160): 31.2 / 30.8 / 38.8; 64 x 64, 1024 -> 1024 (768, 256): 28.1 / 26.8 /
// 42.2; 32 x 250, 1024 -> 1024 (1256, 312): 30.2 / 32.6 / 42.3; 32 x 128, 768 -> 2048 (1280, 384): 24.3 / 29.9 / 36.9.
// Depths that are even but no multiples of 8 go by the same lines.  Full tiles / these, us: 28 Zipf (1.2) groups, 5434 rows, 13374 -> 272
// (short): 182 / 130, b stored transposed 201 / 174; 64 x 16, 6402 -> 518: 128 / 105; 128 x 2, 2046 -> 5462: 472 / 403; 32 x 94, 770 -> 2050:
// 34.1 / 32.1; small ones: 8 x 187, 1022 -> 1030: 16.2 / 12.7, in short ones 18.1; 4 x 75, 130 -> 262: 8.8 / 6.7 and 9.2.
// (The line of one round of short tiles is not sharp: 5 x 409, 272 -> 3520 (952, 252), b stored transposed: 16.7 / 17.8.)
// Weight gradients: small tiles up to two rounds of them.  Wide / small, groups of even and of Zipf (0.8)
// depths: 8 x 512 rows, 512 x 1024 (256 small tiles): 19.4 / 12.4 and 30.8 / 17.3; 16 x 512, 768 x 640 (480): 19.4 /
// 18.1 and 39.0 / 24.9; 16 x 1024, 512 x 1024 (512): 28.3 / 25.2 and 70.7 / 40.6 (the deepest group's tiles set the
// length of the launch: four times as many take a quarter of the time each); past that line even
// depths lose: 64 x 256, 256 x 768 (768): 18.3 / 20.0; 16 x 256, 1024 x 1024 (1024): 19.7 / 22.6.  Groups of
// kMiddlingGroups rows gain up to four rounds of small tiles (not accumulated in fp32, where full tiles add atomically:
// 19 x 1896, 640 x 1024 (760): 115 / 91, but 10 x 2383, 184 x 5592 (880): 128 / 149), where the depth of a tile counts for more than its
// traffic (both gradients in one launch): 9 x 613, 1792 x 960 (1008): 79 / 66; 11 x 980, 1088 x 1088 (891): 82 / 73; 6 x 1784, 1792 x 1088
// (756): 120 / 111; 15 x 1627, 2368 x 256 (570): 91 / 96; of fewer rows 26 x 318, 192 x 1312 (572): 30 / 38.  Groups of
// kDeepGroups rows and more keep the wide ones where these fill the device: where a few of them are much deeper than
// the rest, those are cut along the depth (plan_pieces_by_length).  Where wide tiles leave half of it idle, small
// ones, and pieces of them, which pay from 16 slices on, put the rest to work.  Wide / small and the number of
// wide ones: 19 x 2569 rows, 384 x 128 (38): 53 / 25; 5 x 3106, 608 x 240 (15): 60 / 24; 3 x 4000, 1024 x 1024, Zipf 1.2 (48):
// 82 / 53; 4 x 15000, 1024 x 512 (32): 101 / 72; 6 x 5000, 768 x 1024 (72): 89 / 64; 8 x 5000, 1024 x 1024 (128): 89 / 84; with fp32
// accumulation 98 / 70 and 108 / 94; but 4 x 10000, 2048 x 1024 (128): 154 / 170.  Only where the caller says so
// (GG_FLAG_FEW_TILES, as the PyTorch binding always does): of the rules here the only one that is an option of the C ABI.
// Without it the groups' depths are cut by plan_deep_tiles, into as many pieces of every tile that is cut.
constexpr int64_t kDeepGroups = 2560;
constexpr int64_t kMiddlingGroups = 512;
constexpr int64_t kVeryDeepGroups = 8192;
constexpr int64_t kDeepProduct = 6144;       // weights are pulled through short tiles
constexpr int64_t kDeepForSharing = 3072;    // small tiles one to a compute unit

TileShape pick_shape(const gg_gmm_args& g, const Route& r) {
  const int halves = g.epilogue == GG_EPILOGUE_SWIGLU ? 2 : 1;   // of a tile's width: gate and up
  if (g.trans_a) {
    const int64_t small_tiles = expected_tiles(g, SmallSquare::BM, SmallSquare::BN);
    const int64_t wide_tiles = expected_tiles(g, Wide::BM, Wide::BN);
    const bool few = (g.flags & GG_FLAG_FEW_TILES) &&
                     wide_tiles <= (g.tokens < kVeryDeepGroups * g.num_groups ? kFullLaunch / 2 : kFullLaunch / 4);
    const bool small = has_shape(g, r, SmallSquare::kId) &&
                       (few || (g.tokens < kDeepGroups * g.num_groups &&
                                small_tiles <= (g.tokens >= kMiddlingGroups * g.num_groups && !g.accumulate_f32 ? 4 : 2) * kFullLaunch));
    return small ? shape_of<SmallSquare>() : shape_of<Wide>();
  }
  const int64_t short_tiles = expected_tiles(g, Short::BM, Short::BN / halves);
  const bool streams_weights = g.tokens <= Small::BM * g.num_groups && g.hidden_in >= kDeepProduct && 2 * short_tiles >= kFullLaunch;
  const int64_t most_small = g.hidden_in >= kDeepForSharing ? kFullLaunch : kFullLaunch * 3 / 2;
  if (has_shape(g, r, Small::kId) && !streams_weights && expected_tiles(g, Small::BM, Small::BN / halves) <= most_small)
    return r.ragged_depth ? shape_of<SmallRaggedDepth>() : shape_of<Small>();
  if (has_shape(g, r, Short::kId) && (use_short_shape(g.num_groups, g.tokens, 0) ||
                                      short_tiles <= kFullLaunch))
    return r.ragged_depth ? shape_of<ShortRaggedDepth>() : shape_of<Short>();
  return r.ragged_depth ? shape_of<WideRaggedDepth>() : shape_of<Wide>();
}

// Whether tiles of a call may be cut along the depth: what gg_workspace_bytes_for promises and what a launch is
// allowed.  Judged as for a crowded device (the sizes, and so the tiles of the last round, may be known on the
// device only): a call that could be cut only where its last round holds few tiles does without.
bool may_cut_depth(const gg_gmm_args& g, const Route& r, const TileShape& shape) {
  // (the fix-up of depth pieces stores 4 columns at a time where rows go through indices: whole tiles and row pieces
  // for ragged widths then)
  if (r.generic || (r.ragged_width && r.indexed) || g.num_groups <= 0) return false;
  if (g.flags & (GG_FLAG_WHOLE_TILES | GG_FLAG_ROW_PIECES)) return false;
  // (callers that bring a workspace to every call may share one where these sizes had no use for it)
  if ((r.ragged_width || r.ragged_depth) && !(g.flags & GG_FLAG_EVEN_PIECES)) return false;
  const bool scattered = r.indexed || g.epilogue == GG_EPILOGUE_SWIGLU;
  if (scattered && shape.id == Wide::kId) return false;
  const int64_t slice = r.elem_bytes == 1 ? 2 * gg::BK : gg::BK;   // depth elements per slice
  // (weight-gradient layout: the depth is a group's row count, and one group may hold all rows:
  // the kernel cuts the tiles of groups much deeper than the rest, plan_deep_tiles)
  const int64_t depth = g.trans_a ? g.tokens : g.hidden_in;
  const int slices = (int)std::min<int64_t>((depth + slice - 1) / slice, 1 << 16);
  if (g.trans_a && slices >= 2 * gg::min_slices_per_piece(shape.bm * shape.bn)) return true;
  const int rows = g.trans_a || g.tokens >= g.num_groups * shape.bm ? shape.bm : (int)((g.tokens / g.num_groups + 31) / 32 * 32);
  return gg::best_depth_pieces(slices, rows, shape.bn, kFullLaunch, 2 * kFullLaunch, gg::kMaxDepthPieces) > 1;
}

// A call that has been checked, and how it is launched.
struct Plan {
  bool empty = true;   // nothing to write
  gg::GmmParams p{};
  Route route;
  TileShape shape;
  const gg::VariantOps* variant = nullptr;   // nullptr: the general kernels
  IndexedRows index_rows;
  int epilogue, layout, cus;
  int bn;              // output columns per tile
};

// static_scratch: use the device's static scratch array as the workspace (gg_gmm_no_alloc).
// gate_up: where gate | up are kept beside c (SwiGLU epilogue), or nullptr.
// strides: where rows of a and b are further apart than they are long (gg_gmm_strided).
// assumed: a device to plan for instead of the current one.
int plan_call(const gg_gmm_args& g, bool static_scratch, Plan* out, void* gate_up = nullptr, const Strides* strides = nullptr,
              const DeviceInfo* assumed = nullptr) {
  const int64_t num_groups = g.num_groups, tokens = g.tokens;
  const int64_t hidden_in = g.hidden_in, hidden_out = g.hidden_out;
  const int trans_a = g.trans_a != 0, trans_b = g.trans_b != 0;
  const bool out_f32 = g.accumulate_f32 != 0;
  int rc = check_common(g.batch_sizes, num_groups, tokens, hidden_in, hidden_out, trans_a, trans_b);
  if (rc != GG_OK) return rc;
  if (g.dtype < GG_DTYPE_BF16 || g.dtype > GG_DTYPE_F8E5M2)
    return fail(GG_EINVAL, "dtype must be one of GG_DTYPE_*");
  const int elem_bytes = g.dtype == GG_DTYPE_F8E4M3 || g.dtype == GG_DTYPE_F8E5M2 ? 1 : 2;
  if (g.epilogue != GG_EPILOGUE_NONE && g.epilogue != GG_EPILOGUE_SWIGLU)
    return fail(GG_EINVAL, "epilogue must be one of GG_EPILOGUE_*");
  const bool swiglu = g.epilogue == GG_EPILOGUE_SWIGLU;
  if (swiglu && (trans_a || out_f32))
    return fail(GG_EINVAL, "the SwiGLU epilogue is for the layouts with a row of c per token and a c of the element type");
  if (swiglu && hidden_in * hidden_out >= (int64_t(1) << 28))
    return fail(GG_ELIMIT, "hidden_in * hidden_out must be below 2^28 with the SwiGLU epilogue");
  if (g.a_num_rows < 0 || g.b_num_rows < 0 || g.c_num_rows < 0) return fail(GG_EINVAL, "negative row count");
  if (trans_a && g.c_row_index != nullptr)
    return fail(GG_EINVAL, "c_row_index scatters output rows; the trans_a output has none per token");
  if (!trans_a && g.b_row_index != nullptr)
    return fail(GG_EINVAL, "b_row_index gathers rows of b; only the trans_a layout has a row per token in b");
  if (out_f32 && !trans_a)
    return fail(GG_EINVAL, "the fp32-accumulated output exists for the trans_a layout only");
  if (out_f32 && (hidden_in >= (1 << 20) || hidden_out >= (1 << 20)))
    return fail(GG_ELIMIT, "hidden sizes must be below 2^20 for the accumulating form");
  if (num_groups == 0) return GG_OK;
  // nothing to write
  if (hidden_out == 0 || (trans_a ? hidden_in == 0 : tokens == 0)) return GG_OK;
  if (g.c == nullptr) return fail(GG_EINVAL, "c is null");
  if (tokens > 0 && (g.a == nullptr || g.b == nullptr)) return fail(GG_EINVAL, "a or b is null");
  if (strides != nullptr && !strides_fit(g, *strides)) return fail(GG_EINVAL, "row strides do not fit the call (gg_gmm_strided)");
  const Route route = strides != nullptr ? strided_route(g) : classify(g);
  const uintptr_t address_bits = route.address_bits;
  if (address_bits & (uintptr_t)(elem_bytes - 1) || reinterpret_cast<uintptr_t>(g.c) & (out_f32 ? 3 : 1))
    return fail(GG_ELIMIT, "a, b and c must be aligned to their element size");
  const bool indexed = route.indexed, indexed_fits = route.indexed_fits, generic = route.generic;
  const int64_t a_bytes = route.a_bytes, c_bytes = route.c_bytes;
  const int vec = route.vec;

  // Host-resident sizes are validated here; they travel in the kernel argument block.
  if (!g.batch_sizes_on_device) {
    int64_t row = 0;
    for (int64_t e = 0; e < num_groups; ++e) {
      if (g.batch_sizes[e] < 0) return fail(GG_EINVAL, "batch_sizes[%lld] is negative", (long long)e);
      if (g.batch_sizes[e] > tokens - row)
        return fail(GG_EINVAL, "batch_sizes sum past the %lld rows of a", (long long)tokens);
      row += g.batch_sizes[e];
    }
  }

  DeviceInfo info;
  if (assumed != nullptr) {
    info = *assumed;
  } else {
    rc = device_info(&info);
    if (rc != GG_OK) return rc;
  }
  hipStream_t stream = static_cast<hipStream_t>(g.stream);
  const int layout = trans_a ? gg::kTN : (trans_b ? gg::kNT : gg::kNN);
  const int epilogue = out_f32 ? gg::kEpiAccF32 : (gate_up != nullptr ? gg::kEpiSwiGLUKeep : (swiglu ? gg::kEpiSwiGLU : gg::kEpiStore));
  const TileShape shape = generic ? TileShape{-1, gg::kGenericTileM, gg::kGenericTileN} : pick_shape(g, route);
  // deep groups: the launch is bound by the matrix pipe, and atomic additions to c cost less of
  // its time than reading, adding and writing; shallow groups: bound by the traffic of c, the reverse
  // (small tiles: launches too short for the difference, read-add-write only)
  const int variant_epilogue = out_f32 && shape.id == Wide::kId && tokens >= (int64_t)kShallowBelow * num_groups
                                   ? gg::kEpiAccF32Atomic : epilogue;
  const int bm = shape.bm;
  // output columns per tile: half the tile's width when it holds gate and up columns
  const int bn = shape.bn / (swiglu ? 2 : 1);
  const gg::VariantOps* variant = nullptr;
  if (!generic) {
    variant = find_variant(g.dtype, layout, shape.id, variant_epilogue, indexed ? 1 : 0);
    if (variant == nullptr) return fail(GG_EINVAL, "no kernel for this combination of arguments");
  }

  gg::GmmParams& p = out->p;
  p.a = static_cast<const char*>(g.a);
  p.b = static_cast<const char*>(g.b);
  p.c = static_cast<char*>(g.c);
  p.gate_up = static_cast<char*>(gate_up);
  p.tokens = tokens;
  p.hidden_in = (int32_t)hidden_in;
  p.hidden_out = (int32_t)hidden_out;
  p.b_cols = (int32_t)(swiglu ? 2 * hidden_out : hidden_out);
  p.lda = (int32_t)(strides != nullptr ? strides->a : hidden_in);
  p.ldb = (int32_t)(strides != nullptr ? strides->b : (trans_a ? hidden_out : (trans_b ? hidden_in : p.b_cols)));
  p.a_rows = g.a_row_index;
  p.c_rows = g.c_row_index;
  static_assert(GG_STATUS_NEGATIVE_SIZE == gg::kStatusNegativeSize && GG_STATUS_ROWS_PAST_END == gg::kStatusRowsPastEnd,
                "the header's status bits are the kernel's");
  p.status = g.batch_sizes_on_device ? g.size_status : nullptr;
  p.a_bytes = (uint32_t)(indexed_fits ? a_bytes : 0);
  p.c_bytes = (uint32_t)(indexed_fits ? c_bytes : 0);
  const IndexedRows index_rows = indexed_rows(g);
  p.a_index_rows = (uint32_t)(indexed_fits ? index_rows.a : 0);
  p.c_index_rows = (uint32_t)(indexed_fits ? index_rows.c : 0);
  p.group_m = band_height(num_groups, tokens, trans_a);
  static_assert(GG_FLAG_WHOLE_TILES == gg::kFlagWholeTiles && GG_FLAG_ONE_CLASS == gg::kFlagOneClass &&
                GG_FLAG_ROW_PIECES == gg::kFlagRowPieces && GG_FLAG_GROUP_ORDER == gg::kFlagGroupOrder,
                "the header's flags are the kernel's");
  p.flags = g.flags & (GG_FLAG_WHOLE_TILES | GG_FLAG_ONE_CLASS | GG_FLAG_ROW_PIECES | GG_FLAG_GROUP_ORDER);
  if (merge_stores(g)) p.flags |= gg::kFlagMergeStores;
  if (trans_a && (g.flags & GG_FLAG_FEW_TILES)) p.flags |= gg::kFlagPiecesByLength;
  if (strides != nullptr && (hidden_out % 8 != 0 || (reinterpret_cast<uintptr_t>(g.c) & 15))) p.flags |= gg::kFlagAnyRows;
  const bool depth_pieces = !generic && may_cut_depth(g, route, shape);
  p.sched_out = nullptr;
  if (static_scratch) {
    if (g.workspace != nullptr)
      return fail(GG_EINVAL, "gg_gmm_no_alloc brings its own scratch: workspace must be NULL");
    if (info.cus > kStaticScratchGrid)
      return fail(GG_ELIMIT, "the static scratch serves launches of up to %d workgroups, this device has %d "
                  "compute units", kStaticScratchGrid, info.cus);
    p.workspace = reinterpret_cast<char*>(info.scratch);
    p.ws_slots = (int32_t)(((uint64_t)GG_WORKSPACE_BYTES - gg::kWsCounterBytes) /
                           ((uint64_t)bm * bn * (swiglu ? 2 : 1) * 4));
    if (p.ws_slots > 1024) p.ws_slots = 1024;
    if (!depth_pieces) p.ws_slots = 0;
    // Every call on this device shares the array and finds what the last call left: the arrival
    // counters must start at zero (a fill kernel, not a memset: callers may be capturing a graph).
    hipLaunchKernelGGL(clear_counters_kernel, dim3(1), dim3(gg::kWsCounterBytes / 4), 0, stream,
                       reinterpret_cast<int*>(info.scratch));
    GG_HIP(hipGetLastError());
  } else if (g.workspace != nullptr && !generic) {
    const bool ragged = route.ragged_width || route.ragged_depth;   // (takes any workspace; one that does not fit is not used)
    const bool misaligned = (reinterpret_cast<uintptr_t>(g.workspace) & 255) != 0;
    if (misaligned && !ragged) return fail(GG_ELIMIT, "the workspace must be 256-byte aligned");
    const uint64_t slot_bytes = (uint64_t)bm * bn * (swiglu ? 2 : 1) * 4;
    // (one tile of the wide shape, or of the short one where groups average few rows: what a caller can tell
    // without the rules of pick_shape, whose tiles are no larger)
    const bool few_rows = !swiglu && !indexed && elem_bytes == 2 && use_short_shape(num_groups, tokens, trans_a);
    const uint64_t least = gg::kWsCounterBytes + (few_rows ? (uint64_t)Short::BM * Short::BN : (uint64_t)Wide::BM * Wide::BN) * 4;
    if (g.workspace_bytes < least && !ragged)
      return fail(GG_ELIMIT, "the workspace holds %llu bytes, the smallest useful one %llu",
                  (unsigned long long)g.workspace_bytes, (unsigned long long)least);
    const uint64_t slots = misaligned || g.workspace_bytes < least ? 0 : (g.workspace_bytes - gg::kWsCounterBytes) / slot_bytes;
    p.workspace = static_cast<char*>(g.workspace);
    // one arrival counter per tile of the last round: at most grid / 2 of them, 1024 fit
    p.ws_slots = !depth_pieces ? 0 : (slots > 1024 ? 1024 : (int32_t)slots);
  }

  out->route = route;
  out->shape = shape;
  out->variant = variant;
  out->index_rows = index_rows;
  out->epilogue = epilogue;
  out->layout = layout;
  out->cus = info.cus;
  out->bn = bn;
  out->empty = false;
  return GG_OK;
}

// The part of a call that one launch takes, groups first .. first + count - 1: into plan->p (and hs: their
// host-resident sizes, which start at row *row).  *tiles: how many there are, at most.
int plan_launch(const gg_gmm_args& g, Plan* plan, int64_t first, int64_t count, int64_t* row, gg::HostSizes* hs, int64_t* tiles) {
  gg::GmmParams& p = plan->p;
  const int bm = plan->shape.bm;
  const int64_t tiles_n = (g.hidden_out + plan->bn - 1) / plan->bn;
  const int64_t tiles_m_fixed = (g.hidden_in + bm - 1) / bm;   // weight-gradient layout
  p.first_group = (int32_t)first;
  p.num_groups = (int32_t)count;
  if (g.batch_sizes_on_device) {
    p.sizes_dev = g.batch_sizes;
    p.row_base = 0;
    // upper bound for any size vector (the device clips rows to `tokens`)
    *tiles = g.trans_a ? count * tiles_m_fixed * tiles_n : (g.tokens / bm + count) * tiles_n;
  } else {
    p.sizes_dev = nullptr;
    p.row_base = *row;
    *tiles = 0;
    for (int64_t i = 0; i < count; ++i) {
      const int64_t m = g.batch_sizes[first + i];
      hs->v[i] = (int32_t)m;
      *row += m;
      *tiles += g.trans_a ? tiles_m_fixed * tiles_n : ((m + bm - 1) / bm) * tiles_n;
    }
  }
  if (*tiles >= (int64_t(1) << 31)) return fail(GG_ELIMIT, "too many output tiles for one launch");
  p.flags &= ~gg::kFlagByTileRows;
  if (plan->variant != nullptr && !g.trans_a && !(p.flags & gg::kFlagGroupOrder) && count >= kByTileRowsGroups &&
      order_by_tile_rows(g.num_groups, g.tokens, tiles_n, bm, plan->cus, g.hidden_in))
    p.flags |= gg::kFlagByTileRows;
  return GG_OK;
}

int launch_call(const gg_gmm_args& g, Plan* plan) {
  if (plan->empty) return GG_OK;
  hipStream_t stream = static_cast<hipStream_t>(g.stream);
  // At most GG_MAX_GROUPS_PER_LAUNCH groups per launch.  A launch sees all operands and the rows
  // its groups start at: handed over by the host for host-resident sizes, summed up by the kernel
  // itself from the sizes of the groups before it for device-resident ones.
  int64_t row = 0;
  for (int64_t first = 0; first < g.num_groups; first += GG_MAX_GROUPS_PER_LAUNCH) {
    const int64_t count = g.num_groups - first < GG_MAX_GROUPS_PER_LAUNCH
                              ? g.num_groups - first : GG_MAX_GROUPS_PER_LAUNCH;
    gg::HostSizes hs;
    int64_t tiles;
    const int rc = plan_launch(g, plan, first, count, &row, &hs, &tiles);
    if (rc != GG_OK) return rc;
    if (tiles == 0) continue;
    // the full grid also for few tiles: the last round's tiles may be cut into pieces for
    // the workgroups that would otherwise idle
    if (plan->variant == nullptr) {
      gg::GenericParams gp;
      gp.p = plan->p;
      gp.p.workspace = nullptr;
      gp.p.ws_slots = 0;
      gp.a_rows = g.a_row_index;
      gp.b_rows = g.b_row_index;
      gp.c_rows = g.c_row_index;
      const IndexedRows& index_rows = plan->index_rows;
      gp.a_num_rows = index_rows.a;
      gp.b_num_rows = index_rows.b;
      gp.c_num_rows = index_rows.c;
      // light workgroups (28 KiB of LDS): two per compute unit
      const int64_t grid = tiles < 2 * plan->cus ? tiles : 2 * plan->cus;
      GG_HIP(generic_ops(g.dtype)->launch(plan->layout, plan->route.vec, plan->epilogue, gp, hs, (int)grid, stream));
    } else {
      GG_HIP(plan->variant->launch(plan->p, hs, plan->cus * plan->variant->workgroups_per_cu, stream));
    }
  }
  return GG_OK;
}

int gmm_impl(const gg_gmm_args& g, bool static_scratch = false) {
  Plan plan;
  const int rc = plan_call(g, static_scratch, &plan);
  return rc != GG_OK ? rc : launch_call(g, &plan);
}

// Groups of few rows and large weights: the first product does nothing but read weights, the second nothing but
// write gradients, and reads queue behind writes.  Two launches' time over one's, geometric mean, least and most of 110 products drawn
// over 2 - 105 rows to a group, 6 - 200 groups, 128 - 7168 -> 128 - 10000, by MB of weights: below 64 1.09 (1.00 - 1.17), to
// 128 1.07 (1.02 - 1.17), to 384 1.03 (0.97 - 1.07), to 700 1.00 (0.90 - 1.10), to 900 0.97 (0.86 - 1.03), to 1500 0.99 (0.90 - 1.02).
// Us: 48 x 65 rows, 3600 -> 1184 (390): 211 in two, 202 in one; 13 x 9, 3856 -> 4744 (454): 233 / 252; 20 x 6, 2504 -> 9016 (861): 408 /
// 466; 108 x 23, 3792 x 9328 (7290): 3295 / 3356.
constexpr int64_t kPairWeightBytes = int64_t(384) << 20;
constexpr int64_t kLongRounds = 8;   // (see pair_kernel)
bool reads_then_writes(const gg_gmm_args& g) {
  return use_short_shape(g.num_groups, g.tokens, 0) && g.num_groups * g.hidden_in * g.hidden_out * 2 > kPairWeightBytes;
}

// The kernel that runs both calls in one launch, or nullptr: a product with plain rows and epilogue and a weight
// gradient, over the same groups, in tile shapes of about the same weight, sharing no workspace.
const gg::PairOps* pair_kernel(const gg_gmm_args& g1, const Plan& p1, const gg_gmm_args& g2, const Plan& p2) {
  if (p1.empty || p2.empty || p1.variant == nullptr || p2.variant == nullptr) return nullptr;
  if (g1.trans_a || !g2.trans_a || p1.epilogue != gg::kEpiStore || p2.epilogue != gg::kEpiStore) return nullptr;
  if (p1.route.indexed || p2.route.indexed || g1.dtype != g2.dtype || g1.stream != g2.stream) return nullptr;
  if (g1.batch_sizes != g2.batch_sizes || g1.batch_sizes_on_device != g2.batch_sizes_on_device ||
      g1.num_groups != g2.num_groups || g1.tokens != g2.tokens || g1.num_groups > GG_MAX_GROUPS_PER_LAUNCH)
    return nullptr;
  if (p1.p.ws_slots > 0 && p2.p.ws_slots > 0 && p1.p.workspace == p2.p.workspace) return nullptr;
  if (reads_then_writes(g1)) return nullptr;
  // (launches of many rounds have little to gain.  Two launches' time over one's by the rounds of the shorter product, geometric mean,
  // least and most of 50 products of 120 - 6000 rows to a group: 2 to 5 rounds 1.03 (0.98 - 1.09), 5 to 8 1.026 (1.013 - 1.042), 8 to 10
  // 1.008 (1.000 - 1.016), 10 to 24 1.002 (0.994 - 1.010); 8 x 4096 rows, 4096 -> 14336 (8.25), forward and gradients: 8383 us
  // in two, 8457 in one; 256 x 256, 7168 -> 2048 (42): 6753 / 6777)
  if (expected_tiles(g1, p1.shape.bm, p1.shape.bn) >= kLongRounds * kFullLaunch &&
      expected_tiles(g2, p2.shape.bm, p2.shape.bn) >= kLongRounds * kFullLaunch)
    return nullptr;
  // (small tiles have a compute unit each to themselves here, half as many as alone: too few to pull the weights of
  // deep products.  14 x 221 rows, 11392 -> 384: 118 / 130)
  if (p1.shape.id == Small::kId && g1.hidden_in > kDeepForSharing) return nullptr;
  return find_pair(g1.dtype, p1.layout, p1.shape.id, p2.shape.id);
}

// Both calls of a pair, planned.
struct PairPlan {
  Plan first, second;
  const gg::PairOps* pair = nullptr;   // the kernel that runs both in one launch; nullptr: one after the other
  gg::HostSizes sizes;                 // (pair)
};

int plan_pair(const gg_gmm_args* first, const Strides* strides1, const gg_gmm_args* second, const Strides* strides2,
              PairPlan* out, const DeviceInfo* assumed = nullptr) {
  if (first == nullptr || second == nullptr) return fail(GG_EINVAL, "args is null");
  if (first->struct_bytes != sizeof(gg_gmm_args) || second->struct_bytes != sizeof(gg_gmm_args))
    return fail(GG_EINVAL, "gg_gmm_args.struct_bytes is not the %zu this library expects", sizeof(gg_gmm_args));
  Plan &p1 = out->first, &p2 = out->second;
  int rc = plan_call(*first, false, &p1, nullptr, strides1, assumed);
  if (rc == GG_OK) rc = plan_call(*second, false, &p2, nullptr, strides2, assumed);
  if (rc != GG_OK) return rc;
  // (also one after the other: the partial tiles of the first would be left where the second's counters have to be zero)
  if (p1.p.ws_slots > 0 && p2.p.ws_slots > 0 && p1.p.workspace != p2.p.workspace &&
      p1.p.workspace < p2.p.workspace + second->workspace_bytes && p2.p.workspace < p1.p.workspace + first->workspace_bytes) {
    // (ragged sizes take any workspace, see plan_call)
    const bool ragged1 = p1.route.ragged_width || p1.route.ragged_depth, ragged2 = p2.route.ragged_width || p2.route.ragged_depth;
    if (!ragged1 && !ragged2) return fail(GG_EINVAL, "the workspaces of the two calls overlap in part");
    (ragged1 ? p1 : p2).p.ws_slots = 0;
  }
  out->pair = pair_kernel(*first, p1, *second, p2);
  if (out->pair != nullptr) {
    int64_t row1 = 0, row2 = 0, tiles1, tiles2;
    rc = plan_launch(*first, &p1, 0, first->num_groups, &row1, &out->sizes, &tiles1);
    if (rc == GG_OK) rc = plan_launch(*second, &p2, 0, second->num_groups, &row2, &out->sizes, &tiles2);
    if (rc != GG_OK) return rc;
    if (tiles1 == 0 || tiles2 == 0) out->pair = nullptr;
  }
  return GG_OK;
}

int run_pair(const gg_gmm_args* first, const Strides* strides1, const gg_gmm_args* second, const Strides* strides2) {
  PairPlan plan;
  int rc = plan_pair(first, strides1, second, strides2, &plan);
  if (rc != GG_OK) return rc;
  if (plan.pair != nullptr) {
    GG_HIP(plan.pair->launch(plan.first.p, plan.second.p, plan.sizes, plan.first.cus * plan.pair->workgroups_per_cu,
                             static_cast<hipStream_t>(first->stream)));
    return GG_OK;
  }
  rc = launch_call(*first, &plan.first);
  return rc == GG_OK ? launch_call(*second, &plan.second) : rc;
}

}  // namespace

extern "C" {

const char* gg_last_error(void) { return g_err; }

int gg_version(void) { return 200; }

int gg_init(void) {
  DeviceInfo info;
  return device_info(&info);
}

int32_t* gg_size_status_word(void) {
  DeviceInfo info;
  return device_info(&info) == GG_OK ? info.size_status : nullptr;
}

int gg_tile_shape(int64_t num_groups, int64_t tokens, int trans_a, int trans_b, int* bm, int* bn,
                  int* bk) {
  if (trans_a && trans_b) return fail(GG_EINVAL, "trans_a and trans_b cannot both be set");
  const bool s = use_short_shape(num_groups, tokens, trans_a);
  if (bm) *bm = s ? Short::BM : Wide::BM;
  if (bn) *bn = s ? Short::BN : Wide::BN;
  if (bk) *bk = gg::BK;
  return GG_OK;
}

int gg_debug_tile(const gg_gmm_args* args, int* bm, int* bn) {
  if (args == nullptr || args->struct_bytes != sizeof(gg_gmm_args) || args->num_groups <= 0 || args->hidden_out <= 0)
    return fail(GG_EINVAL, "args do not describe a call with an output");
  const Route route = classify(*args);
  const TileShape shape = route.generic ? TileShape{-1, 0, 0} : pick_shape(*args, route);
  if (bm) *bm = shape.bm;
  if (bn) *bn = shape.bn / (args->epilogue == GG_EPILOGUE_SWIGLU ? 2 : 1);
  return GG_OK;
}

int gg_debug_pair(const gg_gmm_args* first, const gg_gmm_args* second, const int64_t* strides, int* shapes) {
  if (shapes == nullptr) return fail(GG_EINVAL, "shapes is null");
  const Strides strides1{strides ? strides[0] : 0, strides ? strides[1] : 0};
  const Strides strides2{strides ? strides[2] : 0, strides ? strides[3] : 0};
  DeviceInfo device;
  device.cus = kFullLaunch;
  PairPlan plan;
  const int rc = plan_pair(first, strides ? &strides1 : nullptr, second, strides ? &strides2 : nullptr, &plan, &device);
  if (rc != GG_OK) return rc;
  const bool one = plan.pair != nullptr;
  shapes[0] = one ? plan.first.shape.bm : 0;
  shapes[1] = one ? plan.first.shape.bn : 0;
  shapes[2] = one ? plan.second.shape.bm : 0;
  shapes[3] = one ? plan.second.shape.bn : 0;
  return GG_OK;
}

int gg_debug_deep_cut(const int64_t* batch_sizes, int64_t num_groups, int64_t tiles_per_group, int workgroups,
                      int partial_tiles, int tile_outputs, int* pieces, int* tiles) {
  if (batch_sizes == nullptr || num_groups < 1 || num_groups > GG_MAX_GROUPS_PER_LAUNCH || tiles_per_group < 1 ||
      tiles_per_group > (1 << 20) || workgroups < 1 || partial_tiles < 0 || pieces == nullptr || tiles == nullptr)
    return fail(GG_EINVAL, "bad argument");
  int64_t rows[GG_MAX_GROUPS_PER_LAUNCH];
  std::copy(batch_sizes, batch_sizes + num_groups, rows);
  std::sort(rows, rows + num_groups, std::greater<int64_t>());
  if (rows[num_groups - 1] < 0 || rows[0] >= (int64_t(1) << 31) / num_groups)
    return fail(GG_EINVAL, "batch_sizes are negative or too large");
  const int64_t all = std::accumulate(rows, rows + num_groups, int64_t(0));
  const gg::DeepCut cut = gg::cut_deep_tiles([&](int q) { return (int)((rows[q] + gg::BK - 1) / gg::BK); }, (int)num_groups, all,
                                             (int)tiles_per_group, workgroups, partial_tiles,
                                             gg::min_slices_per_piece(tile_outputs), gg::BK);
  *pieces = cut.pieces;
  *tiles = cut.tiles;
  return GG_OK;
}

int gg_debug_pieces(const int64_t* batch_sizes, int64_t num_groups, int64_t tiles_per_group, int workgroups, int units,
                    int partial_tiles, int tile_outputs, int tail_pieces, int32_t* pieces, int32_t* places, int64_t capacity) {
  if (batch_sizes == nullptr || num_groups < 1 || num_groups > GG_MAX_GROUPS_PER_LAUNCH || tiles_per_group < 1 ||
      tiles_per_group > (1 << 20) || workgroups < 1 || units < 1 || partial_tiles < 0 || tail_pieces < 1 || pieces == nullptr)
    return fail(GG_EINVAL, "bad argument");
  int64_t rows[GG_MAX_GROUPS_PER_LAUNCH];
  std::copy(batch_sizes, batch_sizes + num_groups, rows);
  std::sort(rows, rows + num_groups, std::greater<int64_t>());
  if (rows[num_groups - 1] < 0 || rows[0] >= (int64_t(1) << 31) / num_groups)
    return fail(GG_EINVAL, "batch_sizes are negative or too large");
  struct {
    uint32_t groups, depth[GG_MAX_GROUPS_PER_LAUNCH], upto[GG_MAX_GROUPS_PER_LAUNCH + 1];
    uint32_t at(uint32_t q) const { return q < groups ? depth[q] : 0; }
    uint32_t first(uint32_t n) const { return upto[std::min(n, groups)]; }
  } depths;
  depths.groups = (uint32_t)num_groups;
  depths.upto[0] = 0;
  for (int64_t q = 0; q < num_groups; ++q) {
    depths.depth[q] = (uint32_t)((rows[q] + gg::BK - 1) / gg::BK);
    depths.upto[q + 1] = depths.upto[q] + depths.depth[q];
  }
  const gg::PieceLaunch launch{(int)(num_groups * tiles_per_group), (int)tiles_per_group, workgroups, units, partial_tiles};
  auto choose = [&](auto outputs) {   // length in slices, 0: nothing is cut
    using Costs = gg::PieceCosts<decltype(outputs)::value>;
    const int deepest = (int)depths.at(0);
    if (partial_tiles == 0 || deepest < 4 * Costs::SHORTEST) return 0;
    const float share = ((float)depths.first((uint32_t)num_groups) * launch.per_group + Costs::TILE * launch.tiles) / workgroups;
    float best = gg::kPiecesPay * gg::uncut_end<Costs::OUT>(depths, launch, tail_pieces, share);
    int chosen = 0;
    for (int k = 0; k < gg::kPieceLengths; ++k) {
      const int n = gg::piece_count<Costs::OUT>(k), length = (deepest + n - 1) / n;
      int cut = 0, all = 0;
      for (; gg::is_cut(depths.at((uint32_t)cut), length); ++cut) all += ((int)depths.at((uint32_t)cut) + length - 1) / length;
      const float end = gg::pieces_end<Costs::OUT>(depths, launch, n, length, cut, all, share);
      if (end < best) best = end, chosen = length;
    }
    return chosen;
  };
  const int length = tile_outputs > Small::BM * Small::BN * 2 ? choose(std::integral_constant<int, Wide::BM * Wide::BN>{})
                                                              : choose(std::integral_constant<int, SmallSquare::BM * SmallSquare::BN>{});
  int64_t index = 0;
  for (int64_t q = 0; q < num_groups; ++q) {
    const uint32_t d = depths.at((uint32_t)q);
    pieces[q] = length > 0 && gg::is_cut(d, length) ? (int32_t)((d + length - 1) / length) : 0;
    const int64_t first = index;
    for (; index < first + pieces[q] * tiles_per_group; ++index) {
      if (places == nullptr) continue;
      if (index >= capacity) return fail(GG_EINVAL, "more than %lld pieces", (long long)capacity);
      const gg::PieceAt at = gg::piece_at((int)index, (int)first, (int)tiles_per_group);
      const int32_t place[4] = {(int32_t)(q * tiles_per_group) + at.tile, at.piece, pieces[q],
                                at.slot + at.piece * (int)tiles_per_group};
      std::copy(place, place + 4, places + 4 * index);
    }
  }
  return GG_OK;
}

int gg_gmm(const gg_gmm_args* args) {
  if (args == nullptr) return fail(GG_EINVAL, "args is null");
  if (args->struct_bytes != sizeof(gg_gmm_args))
    return fail(GG_EINVAL, "gg_gmm_args.struct_bytes is %u, this library expects %zu", args->struct_bytes,
                sizeof(gg_gmm_args));
  return gmm_impl(*args);
}

int gg_keeps_gate_up(const gg_gmm_args* args) {
  if (args == nullptr || args->struct_bytes != sizeof(gg_gmm_args)) return 0;
  if (args->epilogue != GG_EPILOGUE_SWIGLU || (args->dtype != GG_DTYPE_BF16 && args->dtype != GG_DTYPE_F16)) return 0;
  const Route r = classify(*args);
  return !r.generic && !r.indexed ? 1 : 0;
}

int gg_gmm_keep_gate_up(const gg_gmm_args* args, void* gate_up) {
  if (!gg_keeps_gate_up(args)) return fail(GG_EINVAL, "gate | up cannot be kept by this call (gg_keeps_gate_up)");
  if (gate_up == nullptr || (reinterpret_cast<uintptr_t>(gate_up) & 15))
    return fail(GG_EINVAL, "gate_up must be on a 16-byte boundary");
  Plan plan;
  const int rc = plan_call(*args, false, &plan, gate_up);
  return rc != GG_OK ? rc : launch_call(*args, &plan);
}

int gg_gmm_strided(const gg_gmm_args* args, int64_t a_row, int64_t b_row) {
  if (args == nullptr || args->struct_bytes != sizeof(gg_gmm_args)) return fail(GG_EINVAL, "args is null or of another size");
  const Strides strides{a_row, b_row};
  Plan plan;
  const int rc = plan_call(*args, false, &plan, nullptr, &strides);
  return rc != GG_OK ? rc : launch_call(*args, &plan);
}

int gg_gmm_pair(const gg_gmm_args* first, const gg_gmm_args* second) { return run_pair(first, nullptr, second, nullptr); }

int gg_gmm_pair_strided(const gg_gmm_args* first, int64_t a_row1, int64_t b_row1, const gg_gmm_args* second, int64_t a_row2,
                        int64_t b_row2) {
  const Strides strides1{a_row1, b_row1}, strides2{a_row2, b_row2};
  return run_pair(first, &strides1, second, &strides2);
}

uint64_t gg_workspace_bytes_for(const gg_gmm_args* args) {
  if (args == nullptr || args->struct_bytes != sizeof(gg_gmm_args)) return 0;
  const gg_gmm_args& g = *args;
  if (g.dtype < GG_DTYPE_BF16 || g.dtype > GG_DTYPE_F8E5M2 || g.hidden_in <= 0 || g.hidden_out <= 0) return 0;
  const Route r = classify(g);
  return !r.generic && may_cut_depth(g, r, pick_shape(g, r)) ? GG_WORKSPACE_BYTES : 0;
}

uint64_t gg_workspace_bytes_for_strided(const gg_gmm_args* args, int64_t a_row, int64_t b_row) {
  if (args == nullptr || args->struct_bytes != sizeof(gg_gmm_args)) return 0;
  const gg_gmm_args& g = *args;
  if (g.hidden_in <= 0 || g.hidden_out <= 0 || !strides_fit(g, Strides{a_row, b_row})) return 0;
  const Route r = strided_route(g);
  return may_cut_depth(g, r, pick_shape(g, r)) ? GG_WORKSPACE_BYTES : 0;
}

int gg_gmm_no_alloc(const gg_gmm_args* args) {
  if (args == nullptr) return fail(GG_EINVAL, "args is null");
  if (args->struct_bytes != sizeof(gg_gmm_args))
    return fail(GG_EINVAL, "gg_gmm_args.struct_bytes is %u, this library expects %zu", args->struct_bytes,
                sizeof(gg_gmm_args));
  return gmm_impl(*args, /*static_scratch=*/true);
}

int gg_gmm_bf16(const void* a, const void* b, void* c, const int64_t* batch_sizes,
                int batch_sizes_on_device, int64_t num_groups, int64_t tokens, int64_t hidden_in,
                int64_t hidden_out, int trans_a, int trans_b, void* stream) {
  gg_gmm_args g{};
  g.struct_bytes = sizeof(g);
  g.dtype = GG_DTYPE_BF16;
  g.a = a, g.b = b, g.c = c;
  g.batch_sizes = batch_sizes, g.batch_sizes_on_device = batch_sizes_on_device;
  g.num_groups = num_groups, g.tokens = tokens, g.hidden_in = hidden_in, g.hidden_out = hidden_out;
  g.trans_a = trans_a, g.trans_b = trans_b;
  g.stream = stream;
  return gmm_impl(g);
}

int gg_gmm_bf16_acc_f32(const void* a, const void* b, float* c, const int64_t* batch_sizes,
                        int batch_sizes_on_device, int64_t num_groups, int64_t tokens,
                        int64_t hidden_in, int64_t hidden_out, void* stream) {
  gg_gmm_args g{};
  g.struct_bytes = sizeof(g);
  g.dtype = GG_DTYPE_BF16;
  g.a = a, g.b = b, g.c = c;
  g.batch_sizes = batch_sizes, g.batch_sizes_on_device = batch_sizes_on_device;
  g.num_groups = num_groups, g.tokens = tokens, g.hidden_in = hidden_in, g.hidden_out = hidden_out;
  g.trans_a = 1, g.accumulate_f32 = 1;
  g.stream = stream;
  return gmm_impl(g);
}

int gg_swiglu_backward(const void* gate_up, const void* grad, void* out, int64_t rows, int64_t cols, int dtype,
                       void* stream) {
  if (dtype != GG_DTYPE_BF16 && dtype != GG_DTYPE_F16) return fail(GG_EINVAL, "dtype must be GG_DTYPE_BF16 or GG_DTYPE_F16");
  if (rows < 0 || cols < 0) return fail(GG_EINVAL, "negative dimension");
  if (rows >= (int64_t(1) << 31) || cols >= (1 << 22)) return fail(GG_ELIMIT, "rows must be below 2^31, cols below 2^22");
  if (rows == 0 || cols == 0) return GG_OK;
  if (gate_up == nullptr || grad == nullptr || out == nullptr) return fail(GG_EINVAL, "gate_up, grad or out is null");
  GG_HIP(gg::swiglu_backward(gate_up, grad, out, rows, cols, dtype, static_cast<hipStream_t>(stream)));
  return GG_OK;
}

uint64_t gg_sum_rows_scratch_bytes(int64_t rows, int64_t num_dst) {
  return rows < 0 || num_dst < 0 ? 0 : gg::sum_rows_scratch_bytes(rows, num_dst);
}

int gg_sum_rows(const void* src, const int32_t* row_index, void* dst, int64_t rows, int64_t num_dst, int64_t cols,
                int dtype, void* scratch, void* stream) {
  if (dtype != GG_DTYPE_BF16 && dtype != GG_DTYPE_F16) return fail(GG_EINVAL, "dtype must be GG_DTYPE_BF16 or GG_DTYPE_F16");
  if (rows < 0 || num_dst < 0 || cols < 0) return fail(GG_EINVAL, "negative dimension");
  if (rows >= (int64_t(1) << 31) || num_dst >= (int64_t(1) << 31) || cols >= (1 << 22))
    return fail(GG_ELIMIT, "rows must be below 2^31, cols below 2^22");
  if (num_dst == 0 || cols == 0) return GG_OK;
  if (dst == nullptr || scratch == nullptr || (rows > 0 && (src == nullptr || row_index == nullptr)))
    return fail(GG_EINVAL, "src, row_index, dst or scratch is null");
  GG_HIP(gg::sum_rows(src, row_index, dst, rows, num_dst, cols, dtype, scratch, static_cast<hipStream_t>(stream)));
  return GG_OK;
}

static int check_repitch(const void* src, const void* dst, int64_t batches, int64_t small_rows, int64_t small_cols,
                         int64_t large_rows, int64_t large_cols, int elem_bytes) {
  if (batches < 0 || small_rows < 0 || small_cols < 0) return fail(GG_EINVAL, "negative dimension");
  if (large_rows < small_rows || large_cols < small_cols) return fail(GG_EINVAL, "the padded tensor must be the larger one");
  if (large_cols >= (int64_t(1) << 23) || large_rows >= (int64_t(1) << 31))
    return fail(GG_ELIMIT, "a batch's rows must be below 2^31, columns below 2^23");
  if (elem_bytes != 1 && elem_bytes != 2) return fail(GG_EINVAL, "elements of 1 or 2 bytes");
  if (src == nullptr || dst == nullptr) return fail(GG_EINVAL, "src or dst is null");
  return GG_OK;
}

int gg_pad_rows(const void* src, void* dst, int64_t batches, int64_t src_rows, int64_t src_cols, int64_t dst_rows,
                int64_t dst_cols, int elem_bytes, void* stream) {
  const int rc = check_repitch(src, dst, batches, src_rows, src_cols, dst_rows, dst_cols, elem_bytes);
  if (rc != GG_OK) return rc;
  if ((dst_cols * elem_bytes) % 16 != 0 || (reinterpret_cast<uintptr_t>(dst) & 15))
    return fail(GG_ELIMIT, "dst must have rows of whole 16-byte chunks, on a 16-byte boundary");
  if (reinterpret_cast<uintptr_t>(src) & (uintptr_t)(elem_bytes - 1)) return fail(GG_ELIMIT, "src must be aligned to its elements");
  if (batches == 0 || dst_rows == 0 || dst_cols == 0) return GG_OK;
  GG_HIP(gg::pad_rows(src, dst, batches, src_rows, src_cols, dst_rows, dst_cols, elem_bytes, static_cast<hipStream_t>(stream)));
  return GG_OK;
}

int gg_unpad_rows(const void* src, void* dst, int64_t batches, int64_t src_rows, int64_t src_cols, int64_t dst_rows,
                  int64_t dst_cols, void* stream) {
  const int rc = check_repitch(src, dst, batches, dst_rows, dst_cols, src_rows, src_cols, 2);
  if (rc != GG_OK) return rc;
  if ((reinterpret_cast<uintptr_t>(src) | reinterpret_cast<uintptr_t>(dst)) & 1)
    return fail(GG_ELIMIT, "src and dst must be aligned to their elements");
  if (batches == 0 || dst_rows == 0 || dst_cols == 0) return GG_OK;
  GG_HIP(gg::unpad_rows(src, dst, batches, src_rows, src_cols, dst_rows, dst_cols, static_cast<hipStream_t>(stream)));
  return GG_OK;
}

int gg_debug_schedule(const int64_t* batch_sizes, int batch_sizes_on_device, int64_t num_groups,
                      int64_t tokens, int64_t hidden_in, int64_t hidden_out, int trans_a,
                      int trans_b, int64_t* table_out, void* stream_) {
  int rc = check_common(batch_sizes, num_groups, tokens, hidden_in, hidden_out, trans_a, trans_b);
  if (rc != GG_OK) return rc;
  if (num_groups > GG_MAX_GROUPS_PER_LAUNCH)
    return fail(GG_ELIMIT, "at most %d groups per schedule", GG_MAX_GROUPS_PER_LAUNCH);
  if (num_groups == 0) return GG_OK;
  if (table_out == nullptr) return fail(GG_EINVAL, "table_out is null");
  DeviceInfo info;
  rc = device_info(&info);
  if (rc != GG_OK) return rc;
  hipStream_t stream = static_cast<hipStream_t>(stream_);
  gg::GmmParams p{};
  p.tokens = tokens;
  p.hidden_in = (int32_t)hidden_in;
  p.hidden_out = (int32_t)hidden_out;
  p.group_m = band_height(num_groups, tokens, trans_a);
  p.num_groups = (int32_t)num_groups;
  p.b_cols = (int32_t)hidden_out;
  p.lda = (int32_t)hidden_in;
  p.ldb = (int32_t)(trans_b ? hidden_in : hidden_out);
  p.sched_out = table_out;
  const int layout = trans_a ? gg::kTN : (trans_b ? gg::kNT : gg::kNN);
  const bool short_shape = use_short_shape(num_groups, tokens, trans_a);
  {
    const int bm = short_shape ? Short::BM : Wide::BM, bn = short_shape ? Short::BN : Wide::BN;
    if (!trans_a && num_groups >= kByTileRowsGroups &&
        order_by_tile_rows(num_groups, tokens, (hidden_out + bn - 1) / bn, bm, info.cus, hidden_in))
      p.flags |= gg::kFlagByTileRows;
  }
  gg::HostSizes hs;
  if (batch_sizes_on_device) {
    p.sizes_dev = batch_sizes;
  } else {
    // the table shows what the kernel would do with these sizes: clamped like device-resident ones
    for (int64_t i = 0; i < num_groups; ++i) {
      const int64_t v = batch_sizes[i];
      hs.v[i] = (int32_t)(v < 0 ? 0 : (v > tokens ? tokens : v));
    }
  }
  return dispatch_dump(short_shape, layout, p, hs, stream);
}

}  // extern "C"
