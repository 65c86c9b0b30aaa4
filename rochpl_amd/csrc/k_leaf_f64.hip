// Instantiations of the cooperative panel leaf: double registers over double
// storage.
#include "leaf.hpp"

namespace hplx {
namespace {
template <int RPT, bool SINGLE>
const void* entry() {
  return reinterpret_cast<const void*>(
      &leaf::leaf_kernel<double, double, kLeafThreads, RPT, SINGLE>);
}
}  // namespace
template <>
const void* leaf_kernel_ptr<double>(int rpt, bool single) {
  if(single) return rpt == 1 ? entry<1, true>() : entry<kLeafRPT, true>();
  return rpt == 1 ? entry<1, false>() : entry<kLeafRPT, false>();
}
}  // namespace hplx
