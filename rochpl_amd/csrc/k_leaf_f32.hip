// Instantiations of the cooperative panel leaf: float registers over float
// storage (the FP32 panel of the mixed-precision factorisation).
#include "leaf.hpp"

namespace hplx {
template <>
const void* leaf_kernel_ptr<float>(int rpt) {
  return rpt == 1 ? reinterpret_cast<const void*>(
                        &leaf::leaf_kernel<float, float, kLeafThreads, 1>)
                  : reinterpret_cast<const void*>(
                        &leaf::leaf_kernel<float, float, kLeafThreads, kLeafRPT>);
}
}  // namespace hplx
