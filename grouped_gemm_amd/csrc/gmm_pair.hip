// One pair kernel of the library: the instantiation of gmm_pair_kernel named by -DGG_PAIR_INDEX=<n> (an index of
// the pairs in gmm_variants.def) and the two host functions that prepare and launch it.
#include "gmm_variants.hpp"

#ifndef GG_PAIR_INDEX
#error "compile with -DGG_PAIR_INDEX=<index of a GG_PAIR in gmm_variants.def>"
#endif

namespace gg {
namespace {

template <int INDEX>
struct PairDef;
#define GG_VARIANT(index, DT_, LAYOUT_, SHAPE_, EPI_, INDEXED_)
#define GG_PAIR(index, DT_, LAYOUT_, SHAPE1_, SHAPE2_)   \
  template <>                                            \
  struct PairDef<index> {                                \
    static constexpr int DT = DT_, LAYOUT = LAYOUT_;     \
    using First = SHAPE1_;                               \
    using Second = SHAPE2_;                              \
  };
#include "gmm_variants.def"
#undef GG_VARIANT
#undef GG_PAIR

using V = PairDef<GG_PAIR_INDEX>;
using S1 = V::First;
using S2 = V::Second;
using Cfg = PairConfig<V::LAYOUT, S1, S2, BK, STAGES>;

const void* kernel_address() {
  return reinterpret_cast<const void*>(&gmm_pair_kernel<V::DT, V::LAYOUT, S1, S2, BK, STAGES>);
}

hipError_t prepare() {
  return hipFuncSetAttribute(kernel_address(), hipFuncAttributeMaxDynamicSharedMemorySize, Cfg::LDS_BYTES);
}

hipError_t launch(const GmmParams& p1, const GmmParams& p2, const HostSizes& hs, int grid, hipStream_t stream) {
  GmmParams first = p1, second = p2;
  HostSizes sizes = hs;
  void* args[3] = {&first, &second, &sizes};
  return hipLaunchKernel(kernel_address(), dim3(2 * grid), dim3(Cfg::NT), args, Cfg::LDS_BYTES, stream);
}

const PairOps kOps = {V::DT, V::LAYOUT, S1::kId, S2::kId, Cfg::WORKGROUPS_PER_CU, &prepare, &launch};

}  // namespace

#define GG_CAT2(a, b) a##b
#define GG_CAT(a, b) GG_CAT2(a, b)
const PairOps* GG_CAT(pair_ops_, GG_PAIR_INDEX)() { return &kOps; }

}  // namespace gg
