// Triangular solves on one diagonal block (k <= 1024), 16 right-hand sides per
// workgroup:  T x = b in place.
//
// Used for the unit-lower L11 solves of the panel recursion and of the
// trailing update (rocblas_dtrsm at src/pfact/HPL_pdrpanrlT.cpp:124-135 and
// src/pgesv/HPL_pdupdateTT.cpp:95-106), for the explicit inverse of L11, and
// for the FP32 or FP64 inverses of the diagonal blocks of the mixed-precision
// factors.
//
// The solve itself is tri_block.hpp's.
#include "mxp.hpp"
#include "pipid.hpp"
#include "stamp.hpp"
#include "tri_block.hpp"

namespace hplx {
namespace {

using namespace tri;

// Problem blockIdx.y: T and X advance by t_step and x_step.
template <typename MT, typename V, bool LOWER, bool IDENTITY, int KM>
__global__ __launch_bounds__(kTriThreads) void tri_kernel(int k, int n, const MT* T, int ldt,
                                                          size_t t_step, V* X, int ldx,
                                                          size_t x_step) {
  __shared__ TriShared<V, KM> sh;
  tri_block<MT, V, LOWER, IDENTITY, KM>(k, n, T + blockIdx.y * t_step, ldt,
                                        X + blockIdx.y * x_step, ldx, blockIdx.x, sh);
}

// What follows a panel: block 0 composes its interchanges (pipid.hpp), the
// others form the inverse of L11, 16 columns each.
template <typename V, int KM>
__global__ __launch_bounds__(kTriThreads) void panel_tail_kernel(
    int jb, const int* ipiv, int base, int* permU, const V* L, int ldl, V* Linv, int ldi,
    Stamps st) {
  __shared__ union Shared {
    __device__ Shared() {}
    TriShared<V, KM> tri;
    PipidShared      pipid;
  } sh;
  stamp_now(st);
  if(blockIdx.x == 0)
    pipid_block(jb, ipiv, base, permU, sh.pipid);
  else
    tri_block<V, V, true, true, KM>(jb, jb, L, ldl, Linv, ldi, blockIdx.x - 1, sh.tri);
}

template <typename V>
hipError_t panel_tail(hipStream_t s, int jb, const int* ipiv, int base, int* permU,
                      const V* L, int ldl, V* Linv, int ldi, Stamps st) {
  if(jb <= 0) return hipSuccess;
  if(jb > kMaxNB) return hipErrorInvalidValue;
  const dim3 g(1 + (jb + 15) / 16), b(kTriThreads);
  if(jb <= 128)
    hipLaunchKernelGGL((panel_tail_kernel<V, 128>), g, b, 0, s, jb, ipiv, base, permU, L,
                       ldl, Linv, ldi, st);
  else if(jb <= 512)
    hipLaunchKernelGGL((panel_tail_kernel<V, 512>), g, b, 0, s, jb, ipiv, base, permU, L,
                       ldl, Linv, ldi, st);
  else
    hipLaunchKernelGGL((panel_tail_kernel<V, 1024>), g, b, 0, s, jb, ipiv, base, permU, L,
                       ldl, Linv, ldi, st);
  return hipGetLastError();
}

// The instance with the least LDS: more workgroups to a CU.
template <bool LOWER, bool IDENTITY, typename MT, typename V>
hipError_t tri_solve(hipStream_t s, int k, int n, int blocks, const MT* T, int ldt,
                     size_t t_step, V* X, int ldx, size_t x_step) {
  if(k <= 0 || n <= 0 || blocks <= 0) return hipSuccess;
  if(k > kMaxNB || blocks > 65535) return hipErrorInvalidValue;
  const dim3 g((n + 15) / 16, blocks), b(kTriThreads);
  static_assert(kMaxNB <= 1024, "tri_kernel's largest instance");
  if(k <= 128)
    hipLaunchKernelGGL((tri_kernel<MT, V, LOWER, IDENTITY, 128>), g, b, 0, s, k, n, T, ldt,
                       t_step, X, ldx, x_step);
  else if(k <= 512)
    hipLaunchKernelGGL((tri_kernel<MT, V, LOWER, IDENTITY, 512>), g, b, 0, s, k, n, T, ldt,
                       t_step, X, ldx, x_step);
  else
    hipLaunchKernelGGL((tri_kernel<MT, V, LOWER, IDENTITY, 1024>), g, b, 0, s, k, n, T, ldt,
                       t_step, X, ldx, x_step);
  return hipGetLastError();
}

}  // namespace

hipError_t launch_linv(hipStream_t s, int jb, const double* L, int ldl,
                       double* Linv, int ldi) {
  return tri_solve<true, true>(s, jb, jb, 1, L, ldl, 0, Linv, ldi, 0);
}

hipError_t launch_panel_tail(hipStream_t s, int jb, const int* ipiv, int ipiv_base,
                             int* permU, const double* L, int ldl, double* Linv,
                             int ldi, Stamps st) {
  return panel_tail(s, jb, ipiv, ipiv_base, permU, L, ldl, Linv, ldi, st);
}

hipError_t launch_panel_tail(hipStream_t s, int jb, const int* ipiv, int ipiv_base,
                             int* permU, const float* L, int ldl, float* Linv,
                             int ldi, Stamps st) {
  return panel_tail(s, jb, ipiv, ipiv_base, permU, L, ldl, Linv, ldi, st);
}

// Block J starts at T[J kb, J kb], its inverse (leading dimension kb) at Inv +
// J kb kb.
template <typename MT, typename V>
static hipError_t diag_inverse(hipStream_t s, bool lower, int nblk, int kb, const MT* T,
                               int ldt, V* Inv) {
  if(nblk <= 0 || kb <= 0) return hipSuccess;
  const size_t t_step = kb * (1 + static_cast<size_t>(ldt));
  const size_t x_step = kb * static_cast<size_t>(kb);
  return lower ? tri_solve<true, true>(s, kb, kb, nblk, T, ldt, t_step, Inv, kb, x_step)
               : tri_solve<false, true>(s, kb, kb, nblk, T, ldt, t_step, Inv, kb, x_step);
}

hipError_t launch_diag_inverse(hipStream_t s, bool lower, int nblk, int kb,
                               const float* T, int ldt, double* Inv) {
  return diag_inverse(s, lower, nblk, kb, T, ldt, Inv);
}

hipError_t launch_diag_inverse(hipStream_t s, bool lower, int nblk, int kb,
                               const __half* T, int ldt, double* Inv) {
  return diag_inverse(s, lower, nblk, kb, T, ldt, Inv);
}

hipError_t launch_diag_inverse(hipStream_t s, bool lower, int nblk, int kb,
                               const float* T, int ldt, float* Inv) {
  return diag_inverse(s, lower, nblk, kb, T, ldt, Inv);
}

hipError_t launch_diag_inverse(hipStream_t s, bool lower, int nblk, int kb,
                               const __half* T, int ldt, float* Inv) {
  return diag_inverse(s, lower, nblk, kb, T, ldt, Inv);
}

hipError_t launch_trsm_colsweep(hipStream_t s, int k, int n, const double* L,
                                int ldl, double* B, int ldb) {
  return tri_solve<true, false>(s, k, n, 1, L, ldl, 0, B, ldb, 0);
}

hipError_t launch_trsm_colsweep(hipStream_t s, int k, int n, const float* L,
                                int ldl, float* B, int ldb) {
  return tri_solve<true, false>(s, k, n, 1, L, ldl, 0, B, ldb, 0);
}

}  // namespace hplx
