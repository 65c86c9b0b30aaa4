// Device HPL_pipid: compose jb interchanges (row i <-> ipiv[i]-base) into
// permU[0:jb] (source of each top row) and permU[jb:2jb] (destination of
// each displaced top row, or -1), without a serial pass:
//   position i < jb is last written at step i, with what position p_i held
//   just before step i; a position q is written before step i only by the
//   latest earlier step i' with p_i' = q, which moved there what position i'
//   held just before step i'.  With g(i) = content of position i just before
//   step i:
//     g(i)       = g(last i' < i with p_i' = i), or i if none
//     top[i]     = g(i) if p_i == i, else g(last i' < i with p_i' = p_i), or
//                  p_i if none
//     a position q >= jb ends with g(last i with p_i = q).
//   Chains of g only go to smaller indices and are followed per thread.  The
//   steps that share a target are found through a hash table of the targets,
//   each with a list of its steps (nearly always one): with every step
//   compared to every other it took 81 us for 1024 steps; now it ends well
//   before the inverse of L11 that is formed beside it (97).
#pragma once

#include <hip/hip_runtime.h>

#include "hplx_internal.hpp"

namespace hplx {

struct PipidShared {
  static constexpr int kSlots = 2 * kMaxNB;
  int p[kMaxNB];
  int next[kMaxNB];  // another step with the same target, or -1
  int slot[kMaxNB];
  int to[kMaxNB];    // last i' < i with p_i' == i, or -1
  int g[kMaxNB];
  int out[2 * kMaxNB];
  int key[kSlots], head[kSlots];
};

// One workgroup of any size.
__device__ inline void pipid_block(int jb, const int* __restrict__ ipiv, int base,
                                   int* __restrict__ permU, PipidShared& sh) {
  const int t = threadIdx.x, nt = blockDim.x;
  // an interchange must target a row at or below its own; anything else is
  // treated as no interchange so that every LDS index stays in range
  for(int i = t; i < jb; i += nt) {
    const int p = ipiv[i] - base;
    sh.p[i]     = p < i ? i : p;
    sh.to[i]    = -1;
  }
  for(int i = t; i < PipidShared::kSlots; i += nt) sh.key[i] = sh.head[i] = -1;
  __syncthreads();
  for(int i = t; i < jb; i += nt) {
    const int p = sh.p[i];
    if(p == i) continue;
    if(p < jb) atomicMax(&sh.to[p], i);
    int h = static_cast<int>((static_cast<uint32_t>(p) * 2654435769u) >> 21);
    for(;; h = (h + 1) & (PipidShared::kSlots - 1)) {
      const int old = atomicCAS(&sh.key[h], -1, p);
      if(old == -1 || old == p) break;
    }
    sh.slot[i] = h;
    sh.next[i] = atomicExch(&sh.head[h], i);
  }
  __syncthreads();
  for(int i = t; i < jb; i += nt) {
    int j = i;
    while(sh.to[j] >= 0) j = sh.to[j];  // strictly decreasing chain
    sh.g[i] = j;
  }
  __syncthreads();
  for(int i = t; i < jb; i += nt) {
    const int p    = sh.p[i];
    int       prev = -1;
    bool      last = true;
    if(p != i)
      for(int j = sh.head[sh.slot[i]]; j >= 0; j = sh.next[j]) {
        if(j < i && j > prev) prev = j;
        if(j > i) last = false;
      }
    sh.out[i]      = p == i ? sh.g[i] : prev >= 0 ? sh.g[prev] : p;
    sh.out[jb + i] = -1;
    sh.slot[i]     = p >= jb && last ? p : -1;  // its own entry: read above
  }
  __syncthreads();
  for(int i = t; i < jb; i += nt)
    if(sh.slot[i] >= 0) sh.out[jb + sh.g[i]] = sh.slot[i];
  __syncthreads();
  for(int i = t; i < 2 * jb; i += nt) permU[i] = sh.out[i];
}
static_assert(PipidShared::kSlots == 2048, "the hash keeps the upper 11 bits");

}  // namespace hplx
