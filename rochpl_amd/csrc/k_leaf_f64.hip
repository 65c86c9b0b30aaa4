// Instantiations of the cooperative panel leaf: double registers over double
// storage.
#include "leaf.hpp"

namespace hplx {
template <>
const void* leaf_kernel_ptr<double>(int rpt) {
  return rpt == 1 ? reinterpret_cast<const void*>(
                        &leaf::leaf_kernel<double, double, kLeafThreads, 1>)
                  : reinterpret_cast<const void*>(
                        &leaf::leaf_kernel<double, double, kLeafThreads, kLeafRPT>);
}
}  // namespace hplx
