// A triangular solve on one diagonal block (k <= KM), 16 right-hand sides per
// workgroup: the kernels of k_trsm.hip and the persistent panel kernel's solves
// (k_panel_kernel.hip).
//
// x lives in LDS.  The block is processed in 64-row chunks along the sweep
// direction: 4 of the waves solve the chunk's triangle for 4 right-hand sides
// each (tri_chain.hpp), then all apply the chunk's 64 columns to the
// rows still to be solved, 16 rows at a time, by 16 x 16 x 4 MFMAs, T straight
// from memory into the operand registers.  An MFMA's result is the chain of
// its four FMAs in order, so a row's sum over a chunk has the bits of the plain
// loop over the 64 columns.  Two workgroup barriers per 64 rows; the next
// triangle and the first rows' operands are loaded while a triangle is solved.
//
// Bound by latency: a chunk costs a substitution, a product and the barriers,
// 6 us with 1024 rows.  With one workgroup per right-hand side each of them
// read all of T; us then and now: the inverse of 1024 x 1024 in FP32 357, 97;
// FP64 256 x 256 35, 20; FP64 896 x 896 on the CUs beside an update 462, 138;
// a solve with 32 x 32 and 32 right-hand sides 9.5, 6; all inverses for the
// correction solves of N = 32768 with FP16 factors 8490, 1460.
#pragma once

#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>

#include "hplx_internal.hpp"
#include "tri_chain.hpp"

namespace hplx {
namespace tri {

template <typename V>
using vec4_t = V __attribute__((ext_vector_type(4)));

template <typename V>
__device__ inline vec4_t<V> mfma16x16x4(V a, V b, vec4_t<V> c) {
  if constexpr(sizeof(V) == 8)
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

template <typename V, typename MT>
__device__ inline V to_v(MT x) {
  if constexpr(sizeof(MT) == 2)
    return static_cast<V>(__half2float(x));
  else
    return static_cast<V>(x);
}

template <typename V>
constexpr V kLargest = sizeof(V) == 8 ? V(1.7976931348623157e308) : V(3.40282347e38);

constexpr int kTriThreads = 512;

// Columns [16 block, 16 block + 16) of X on one workgroup.  LOWER: unit lower triangle, forward; else upper,
// backward.  IDENTITY: the right-hand sides are the identity's columns (X is
// only written).  V: element type of X and of the arithmetic; MT: of T.  KM:
// the largest k.
template <typename V, int KM>
struct TriShared {
  alignas(16) V tri[kTri];
  V sx[16 * (KM + 1)];
  V sd[64];
};

template <typename MT, typename V, bool LOWER, bool IDENTITY, int KM>
__device__ __forceinline__ void tri_block(int k, int n, const MT* __restrict__ T, int ldt,
                                          V* __restrict__ X, int ldx, int block,
                                          TriShared<V, KM>& sh) {
  constexpr int LX = KM + 1, NC = 16, NW = kTriThreads / 64;
  V* const tri = sh.tri;
  V* const sx  = sh.sx;
  V* const sd  = sh.sd;
  const int t = threadIdx.x, lane = t & 63, m = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int col0 = block * NC, nc = min(NC, n - col0);
  const int nchunk = (k + 63) / 64;
  // with the identity, the rows before its columns in sweep order stay zero
  const int first =
      IDENTITY ? (LOWER ? col0 / 64 : nchunk - 1 - min(col0 + NC - 1, k - 1) / 64) : 0;
  auto chunk_row = [&](int s) { return 64 * (LOWER ? s : nchunk - 1 - s); };
  auto row       = [&](int p) { return LOWER ? p : 63 - p; };
  // a chunk's triangle: lane = position, the wave's columns NW q + wave (clamped
  // into the block), and its diagonal
  constexpr int QT = 64 / NW;
  MT   tr[QT], td;
  auto load_triangle = [&](int c0) {
    const int i = min(c0 + row(lane), k - 1);
#pragma unroll
    for(int q = 0; q < QT; ++q)
      tr[q] = T[i + static_cast<size_t>(min(c0 + row(NW * q + wave), k - 1)) * ldt];
    if(!LOWER) td = T[i + static_cast<size_t>(i) * ldt];
  };
  // rows [r, r + 16) of the chunk's columns as an MFMA operand
  auto load_rows = [&](int r, int c0, MT(&a)[16]) {
    const int i = min(r + m, k - 1);
#pragma unroll
    for(int q = 0; q < 16; ++q)
      a[q] = T[i + static_cast<size_t>(min(c0 + 4 * q + g, k - 1)) * ldt];
  };
  load_triangle(chunk_row(first));
  for(int c = wave; c < NC; c += NW)
    for(int i = lane; i < k; i += 64)
      sx[c * LX + i] = IDENTITY   ? (i == col0 + c ? V(1) : V(0))
                       : c < nc ? X[i + static_cast<size_t>(col0 + c) * ldx]
                                : V(0);
  for(int s = first; s < nchunk; ++s) {
    const int c0 = chunk_row(s), w = min(64, k - c0);
#pragma unroll
    for(int q = 0; q < QT; ++q) {
      const int c = NW * q + wave;  // column and row of the triangle: positions
      if(lane >= (c & ~15))
        tri[tri_col(c) + 2 * lane] =
            lane > c && row(lane) < w && row(c) < w ? -to_v<V>(tr[q]) : V(0);
    }
    if(!LOWER && wave == 0) sd[lane] = row(lane) < w ? to_v<V>(td) : V(1);
    __syncthreads();
    if(s + 1 < nchunk) load_triangle(chunk_row(s + 1));
    const int r0 = LOWER ? c0 + w : 0, r1 = LOWER ? k : c0;
    MT        a[16], an[16];
    if(r0 + 16 * wave < r1) load_rows(r0 + 16 * wave, c0, an);
    if(wave < 4) {
      V*       xc = sx + (4 * wave + g) * LX + c0;
      const V* p  = tri + 2 * m;
      V        v[4], d[4];
#pragma unroll
      for(int q = 0; q < 4; ++q) {
        const int i = row(16 * q + m);
        v[q]        = i < w ? xc[i] : V(0);
        d[q]        = LOWER ? V(1) : sd[16 * q + m];
      }
      tri_columns<0, LOWER>(v, p, d[0]);
      if(!LOWER || w > 16) tri_columns<1, LOWER>(v, p, d[1]);
      if(!LOWER || w > 32) tri_columns<2, LOWER>(v, p, d[2]);
      if(!LOWER || w > 48) tri_columns<3, LOWER>(v, p, d[3]);
      bool fine = true;
#pragma unroll
      for(int q = 0; q < 4; ++q) fine = fine && fabs(v[q]) <= kLargest<V>;
      const unsigned long long bad = __ballot(!fine);
      if((bad >> (lane & 48)) & 0xffff) {
        // values that are not finite, whose products with the triangle's zeros
        // are not zero: the substitution as it is written
        V u[4];
#pragma unroll
        for(int q = 0; q < 4; ++q) {
          const int i = row(16 * q + m);
          u[q]        = i < w ? xc[i] : V(0);
        }
        for(int pj = 0; pj < 64; ++pj) {
          const int j = row(pj);
          if(j >= w) continue;
          V xj = V(0);
#pragma unroll
          for(int q = 0; q < 4; ++q)
            if((pj >> 4) == q) {
              xj = __shfl(u[q], pj & 15, 16);
              if(!LOWER) xj = xj / sd[pj];
              if(m == (pj & 15)) u[q] = xj;
            }
#pragma unroll
          for(int q = 0; q < 4; ++q) {
            const int pi = 16 * q + m, i = row(pi);
            if(pi > pj && i < w)
              u[q] = fma(-to_v<V>(T[c0 + i + static_cast<size_t>(c0 + j) * ldt]), xj, u[q]);
          }
        }
#pragma unroll
        for(int q = 0; q < 4; ++q) v[q] = u[q];
      }
#pragma unroll
      for(int q = 0; q < 4; ++q) {
        const int i = row(16 * q + m);
        if(i < w) xc[i] = v[q];
      }
    }
    __syncthreads();
    // the chunk's columns times x, off the rows still to be solved
    if(r0 + 16 * wave < r1) {
      V xb[16];
#pragma unroll
      for(int q = 0; q < 16; ++q)
        xb[q] = 4 * q + g < w ? sx[m * LX + c0 + 4 * q + g] : V(0);
      for(int r = r0 + 16 * wave; r < r1; r += 16 * NW) {
#pragma unroll
        for(int q = 0; q < 16; ++q) a[q] = an[q];
        if(r + 16 * NW < r1) load_rows(r + 16 * NW, c0, an);
        vec4_t<V> acc{0, 0, 0, 0};
#pragma unroll
        for(int q = 0; q < 16; ++q)
          acc = mfma16x16x4<V>(4 * q + g < w ? to_v<V>(a[q]) : V(0), xb[q], acc);
#pragma unroll
        for(int e = 0; e < 4; ++e) {
          const int i = r + (sizeof(V) == 8 ? 4 * e + g : 4 * g + e);
          if(i < r1) sx[m * LX + i] -= acc[e];
        }
      }
    }
  }
  __syncthreads();
  for(int c = wave; c < nc; c += NW)
    for(int i = lane; i < k; i += 64)
      X[i + static_cast<size_t>(col0 + c) * ldx] = sx[c * LX + i];
}

}  // namespace tri
}  // namespace hplx
