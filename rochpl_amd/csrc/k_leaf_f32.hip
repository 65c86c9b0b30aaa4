// Instantiations of the cooperative panel leaf: float registers over float
// storage (the FP32 panel of the mixed-precision factorisation).
#include "leaf.hpp"

namespace hplx {
namespace {
template <int RPT, bool SINGLE>
const void* entry() {
  return reinterpret_cast<const void*>(
      &leaf::leaf_kernel<float, float, kLeafThreads, RPT, SINGLE>);
}
}  // namespace
template <>
const void* leaf_kernel_ptr<float>(int rpt, bool single) {
  if(single) return rpt == 1 ? entry<1, true>() : entry<kLeafRPT, true>();
  return rpt == 1 ? entry<1, false>() : entry<kLeafRPT, false>();
}
}  // namespace hplx
