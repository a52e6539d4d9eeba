// What the host side (gmm_api.hip) and the kernel translation units (gmm_variant.hip) share:
// tile shapes, epilogue kinds and the table entry through which a variant is prepared and launched.
#pragma once

#include <hip/hip_runtime.h>

#include "gmm_kernel.hpp"

namespace gg {

constexpr int BK = 64, STAGES = 2;

// Tile shapes; which one a call runs on is decided in gmm_api.hip (pick_shape), where both sides of each line are.
// Wide: 256 x 256 outputs per workgroup, 2 x 2 waves of 128 x 128.  Short: 128 x 256, 1 x 4 waves of 128 x 64, in
// the layouts with a row of c per token, for calls whose groups average few rows (with at most 128 rows per
// group all four waves then share the rows instead of two of them idling: 4-7 % faster below about 100 rows per
// group, slower from 128 on) and for launches that one round of short tiles holds.
struct Wide {
  static constexpr int kId = 0, BM = 256, BN = 256, WAVES_M = 2, WAVES_N = 2;
  static constexpr bool RAGGED_DEPTH = false;
};
struct Short {
  static constexpr int kId = 1, BM = 128, BN = 256, WAVES_M = 1, WAVES_N = 4;
  static constexpr bool RAGGED_DEPTH = false;
};
// The wide, the short and the small shape for a hidden_in that is even but no multiple of 8, in the layouts whose rows run
// along the depth: the kernel then clears, in LDS, what the last 16-byte chunk of a row picks up
// from the next row (DepthMajor::clear_depth_tail).
struct WideRaggedDepth : Wide {
  static constexpr int kId = 2;
  static constexpr bool RAGGED_DEPTH = true;
};
struct ShortRaggedDepth : Short {
  static constexpr int kId = 5;
  static constexpr bool RAGGED_DEPTH = true;
};

// Small tiles, for launches that have too few wide ones to fill the device: 64 x 128 outputs, two
// workgroups per compute unit, in the layouts with a row of c per token; 128 x 128 for weight
// gradients (whose operands run along both widths, at least 128 of each).
struct Small {
  static constexpr int kId = 3, BM = 64, BN = 128, WAVES_M = 2, WAVES_N = 2;
  static constexpr bool RAGGED_DEPTH = false;
};
struct SmallRaggedDepth : Small {
  static constexpr int kId = 6;
  static constexpr bool RAGGED_DEPTH = true;
};
struct SmallSquare {
  static constexpr int kId = 4, BM = 128, BN = 128, WAVES_M = 2, WAVES_N = 2;
  static constexpr bool RAGGED_DEPTH = false;
};

struct VariantOps {
  int dt, layout, shape, epilogue, indexed;
  int lds_bytes;
  int workgroups_per_cu;
  // raises the kernel's dynamic LDS limit on the current device
  hipError_t (*prepare)();
  hipError_t (*launch)(const GmmParams& p, const HostSizes& hs, int grid, hipStream_t stream);
};

// Both gradients of a product in one launch (gmm_pair_kernel).
struct PairOps {
  int dt, layout, shape1, shape2;
  int workgroups_per_cu;
  hipError_t (*prepare)();
  // grid: workgroups of each of the two products
  hipError_t (*launch)(const GmmParams& p1, const GmmParams& p2, const HostSizes& hs, int grid, hipStream_t stream);
};

// The kernels of gmm_generic.hpp for one element type (gmm_generic_variant.hip).
struct GenericParams;
struct GenericOps {
  int dt;
  hipError_t (*launch)(int layout, int vec, int epilogue, const GenericParams& gp, const HostSizes& hs,
                       int grid, hipStream_t stream);
};

constexpr int kGenericTileM = 128, kGenericTileN = 128;
constexpr int kNumElementTypes = 4;   // bf16, f16, f8 e4m3, f8 e5m2

}  // namespace gg
