// A small tile of a GEMM on 256 threads, for k_gemm.hip (tile_kernel) and the
// persistent panel kernel (k_panel_kernel.hip).
#pragma once

#include <hip/hip_runtime.h>

#include "hplx_internal.hpp"

namespace hplx {
namespace gemm {

constexpr int kGroupM      = 8;
constexpr int kTileThreads = 256;
constexpr int kTileK       = 32;

template <typename V>
using vec4_t = V __attribute__((ext_vector_type(4)));
template <typename V>
using vec2_t = V __attribute__((ext_vector_type(2)));

// V_MFMA_F64_16X16X4_F64 / V_MFMA_F32_16X16X4_F32 operand layout (lane l):
//   a-operand: X[l % 16][l / 16]   (16 x 4)
//   b-operand: Y[l / 16][l % 16]   (4 x 16)
//   result:    D[4*r + l / 16][l % 16], r = 0..3         (f64)
//              D[4*(l / 16) + r][l % 16], r = 0..3       (f32)
template <typename V>
__device__ inline int dl_row(int r, int lane) {
  if constexpr(sizeof(V) == 8)
    return 4 * r + (lane >> 4);
  else
    return 4 * (lane >> 4) + r;
}

template <typename V>
__device__ inline vec4_t<V> mfma16x16x4(V a, V b, vec4_t<V> c) {
  if constexpr(sizeof(V) == 8)
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

template <typename V, int BM, int BN>
struct TileShared {
  alignas(16) V a[kTileK * (BM + 2)];
  alignas(16) V b[kTileK * (BN + 2)];
};

// Tile `tile` (rows first within groups of kGroupM tile rows) of C (M x N) =
// beta C + alpha A B, BM x BN on 4 waves in 2 x 2 (t: the thread among them),
// for 16-byte aligned operands with even leading dimensions that are not
// transposed: K in 32-deep stages through one LDS buffer (the next stage's
// loads are in flight in registers meanwhile), C loaded along with the first
// stage.  Every element is the sum over the same MFMA steps as in
// k_gemm.hip's dgemm_kernel, so the two give the same bits (but for zeros of
// op(A)'s upper triangle times values that are not finite).  Not `live`:
// nothing is stored (its barriers are).
//
// Bound by latency (a load, a stage's MFMAs and the store, one after the
// other) or, tall and thin, by C's and A's traffic.
template <typename V, bool BETA0, bool NEG, bool LOWER_A, int BM, int BN>
__device__ __forceinline__ void gemm_tile(int t, int tile, bool live, int M, int N, int K,
                                          const V* __restrict__ A, int lda,
                                          const V* __restrict__ B, int ldb,
                                          V* __restrict__ C, int ldc, int tiles_m,
                                          int tiles_n, TileShared<V, BM, BN>& sh) {
  constexpr int NT = kTileThreads, BKS = kTileK, LA = BM + 2, LB = BN + 2;
  constexpr int TM = BM / 32, TN = BN / 32;
  constexpr int QA = BM * BKS / 2 / NT, QB = BN * BKS / 2 / NT;  // pairs per thread
  constexpr int KA = 2 * NT / BM, OB = 2 * NT / BKS;  // k / columns per pass
  const int width  = kGroupM * tiles_n;
  const int group  = tile / width;
  const int firstm = group * kGroupM;
  const int gsz    = min(tiles_m - firstm, kGroupM);
  const int within = tile - group * width;
  const int m0     = (firstm + within % gsz) * BM;
  const int n0     = within / gsz * BN;
  const int kend   = LOWER_A ? min(K, m0 + BM) : K;

  const int lane = t & 63, wave = t >> 6;
  const int l16 = lane & 15, lk = lane >> 4;
  const int wm0 = (wave & 1) * (BM / 2), wn0 = (wave >> 1) * (BN / 2);

  // out-of-range elements are read from a clamped address and replaced by
  // zero at the LDS store
  const int ao = 2 * (t % (BM / 2)), ak = t / (BM / 2);
  const int bk = 2 * (t % (BKS / 2)), bo = t / (BKS / 2);
  vec2_t<V> ra[QA], rb[QB];
  // pairs that lie inside, one by one at the edge of an odd extent
  const bool pairs_a = M % 2 == 0 || m0 + BM <= M;
  const V*   pa0     = A + min(m0 + ao, pairs_a ? M - 2 : M - 1);
  const V*   pa1     = A + min(m0 + ao + 1, M - 1);
  auto load_stage = [&](int k0) {
    if(pairs_a) {
#pragma unroll
      for(int q = 0; q < QA; ++q)
        ra[q] = *reinterpret_cast<const vec2_t<V>*>(
            pa0 + static_cast<size_t>(min(k0 + ak + KA * q, kend - 1)) * lda);
    } else {
#pragma unroll
      for(int q = 0; q < QA; ++q) {
        const size_t c = static_cast<size_t>(min(k0 + ak + KA * q, kend - 1)) * lda;
        ra[q].x        = pa0[c];
        ra[q].y        = pa1[c];
      }
    }
    if(kend % 2 == 0 || k0 + BKS <= kend) {
      const V* pb = B + min(k0 + bk, kend - 2);
#pragma unroll
      for(int q = 0; q < QB; ++q)
        rb[q] = *reinterpret_cast<const vec2_t<V>*>(
            pb + static_cast<size_t>(min(n0 + bo + OB * q, N - 1)) * ldb);
    } else {
      const int b0 = min(k0 + bk, kend - 1), b1 = min(k0 + bk + 1, kend - 1);
#pragma unroll
      for(int q = 0; q < QB; ++q) {
        const V* c = B + static_cast<size_t>(min(n0 + bo + OB * q, N - 1)) * ldb;
        rb[q].x    = c[b0];
        rb[q].y    = c[b1];
      }
    }
  };
  auto store_stage = [&](int k0) {
#pragma unroll
    for(int q = 0; q < QA; ++q) {
      const int  k  = ak + KA * q;
      const bool in = k0 + k < kend;
      vec2_t<V>  x;
      x.x = in && m0 + ao < M ? (NEG ? -ra[q].x : ra[q].x) : V(0);
      x.y = in && m0 + ao + 1 < M ? (NEG ? -ra[q].y : ra[q].y) : V(0);
      *reinterpret_cast<vec2_t<V>*>(sh.a + k * LA + ao) = x;
    }
#pragma unroll
    for(int q = 0; q < QB; ++q) {
      const int  o  = bo + OB * q;
      const bool in = n0 + o < N;
      sh.b[bk * LB + o]       = in && k0 + bk < kend ? rb[q].x : V(0);
      sh.b[(bk + 1) * LB + o] = in && k0 + bk + 1 < kend ? rb[q].y : V(0);
    }
  };

  load_stage(0);
  V cv[TM][TN][4];
  if(!BETA0) {
#pragma unroll
    for(int i = 0; i < TM; ++i)
#pragma unroll
      for(int j = 0; j < TN; ++j)
#pragma unroll
        for(int r = 0; r < 4; ++r)
          cv[i][j][r] =
              C[min(m0 + wm0 + i * 16 + l16, M - 1) +
                static_cast<size_t>(min(n0 + wn0 + j * 16 + dl_row<V>(r, lane), N - 1)) * ldc];
  }
  vec4_t<V> acc[TM][TN];
#pragma unroll
  for(int i = 0; i < TM; ++i)
#pragma unroll
    for(int j = 0; j < TN; ++j) acc[i][j] = vec4_t<V>{0, 0, 0, 0};
  for(int k0 = 0; k0 < kend; k0 += BKS) {
    if(k0 > 0) __syncthreads();
    store_stage(k0);
    __syncthreads();
    if(k0 + BKS < kend) load_stage(k0 + BKS);
    const V* a_s = sh.a + lk * LA + wm0 + l16;
    const V* b_s = sh.b + lk * LB + wn0 + l16;
#pragma unroll
    for(int ks = 0; ks < BKS / 4; ++ks) {
      V fa[TM], fb[TN];
#pragma unroll
      for(int i = 0; i < TM; ++i) fa[i] = a_s[ks * 4 * LA + i * 16];
#pragma unroll
      for(int j = 0; j < TN; ++j) fb[j] = b_s[ks * 4 * LB + j * 16];
#pragma unroll
      for(int i = 0; i < TM; ++i)
#pragma unroll
        for(int j = 0; j < TN; ++j) acc[i][j] = mfma16x16x4<V>(fb[j], fa[i], acc[i][j]);
    }
  }
#pragma unroll
  for(int i = 0; i < TM; ++i) {
    const int row = m0 + wm0 + i * 16 + l16;
    if(row >= M) continue;
#pragma unroll
    for(int j = 0; j < TN; ++j)
#pragma unroll
      for(int r = 0; r < 4; ++r) {
        const int col = n0 + wn0 + j * 16 + dl_row<V>(r, lane);
        if(live && col < N)
          C[row + static_cast<size_t>(col) * ldc] =
              BETA0 ? acc[i][j][r] : cv[i][j][r] + acc[i][j][r];
      }
  }
}

}  // namespace gemm
}  // namespace hplx
