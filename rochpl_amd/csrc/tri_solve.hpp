// Unit lower triangular solve of one right-hand-side column on one workgroup,
// for the persistent panel kernel (k_panel_kernel.hip), whose workgroups take
// the columns in turn.  x lives in LDS; wave 0 solves 64 rows at a time with
// their triangle in registers (one row per lane) and x broadcast by lane
// shuffles, then every thread applies the 64 columns to the rows still to be
// solved, with all 64 loads of a row issued before the first product.  Any
// workgroup size that is a multiple of 64 works; each row's sum is formed by
// one thread in the same order whatever the size.
#pragma once

#include <hip/hip_runtime.h>

#include "hplx_internal.hpp"

namespace hplx {
namespace trs {

__device__ inline void tri_solve_col(int k, const double* __restrict__ T, int ldt,
                                     double* __restrict__ xc) {
  __shared__ double sx[kMaxNB];
  const int t    = threadIdx.x;
  const int lane = t & 63;
  for(int i = t; i < k; i += blockDim.x) sx[i] = xc[i];
  __syncthreads();
  for(int c0 = 0; c0 < k; c0 += 64) {
    const int w = min(64, k - c0);
    if(t < 64) {
      const int i  = c0 + lane;
      double    xi = lane < w ? sx[i] : 0.0;
      double    e[64];
#pragma unroll
      for(int j = 0; j < 64; ++j)
        e[j] = j < w && lane < w && j < lane ? T[i + static_cast<size_t>(c0 + j) * ldt] : 0.0;
#pragma unroll
      for(int j = 0; j < 64; ++j) {
        if(j < w) {
          const double xj = __shfl(xi, j);
          if(lane > j) xi = fma(-e[j], xj, xi);
        }
      }
      if(lane < w) sx[i] = xi;
    }
    __syncthreads();
    if(w == 64) {
      // full chunk: the row's 64 entries are loaded before the first use, so
      // their latencies overlap
      for(int r = c0 + w + t; r < k; r += blockDim.x) {
        double tv[64];
#pragma unroll
        for(int j = 0; j < 64; ++j) tv[j] = T[r + static_cast<size_t>(c0 + j) * ldt];
        double acc = 0.0;
#pragma unroll
        for(int j = 0; j < 64; ++j) acc = fma(tv[j], sx[c0 + j], acc);
        sx[r] -= acc;
      }
    }
    __syncthreads();
  }
  for(int i = t; i < k; i += blockDim.x) xc[i] = sx[i];
}

}  // namespace trs
}  // namespace hplx
