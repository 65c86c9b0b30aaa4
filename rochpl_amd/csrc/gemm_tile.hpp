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

// One operand of a tile, BO outer indices (rows of C for A, columns for B) by
// kTileK of k, staged as S[k][o] with pitch BO + 2.  KFAST: k is the contiguous
// index in memory, else o.  Pairs are loaded whole where they lie inside and
// one by one at the edge of an odd extent; out-of-range elements are read from
// a clamped address and replaced by zero at the store.
template <typename V, int BO, bool KFAST>
struct TileOperand {
  static constexpr int Q    = BO * kTileK / 2 / kTileThreads;  // pairs per thread
  static constexpr int LD   = BO + 2;
  static constexpr int STEP = 2 * kTileThreads / (KFAST ? kTileK : BO);
  const V* __restrict__ P;
  int       ld, o0, O, o, k;
  vec2_t<V> r[Q];

  __device__ __forceinline__ TileOperand(const V* P_, int ld_, int o0_, int O_, int t)
      : P(P_), ld(ld_), o0(o0_), O(O_),
        o(KFAST ? t / (kTileK / 2) : 2 * (t % (BO / 2))),
        k(KFAST ? 2 * (t % (kTileK / 2)) : t / (BO / 2)) {}

  __device__ __forceinline__ void load(int k0, int kend) {
    if constexpr(!KFAST) {
      if(O % 2 == 0 || o0 + BO <= O) {
        const V* p = P + min(o0 + o, O % 2 == 0 ? O - 2 : O - 1);
#pragma unroll
        for(int q = 0; q < Q; ++q)
          r[q] = *reinterpret_cast<const vec2_t<V>*>(
              p + static_cast<size_t>(min(k0 + k + STEP * q, kend - 1)) * ld);
      } else {
        const V *p0 = P + min(o0 + o, O - 1), *p1 = P + min(o0 + o + 1, O - 1);
#pragma unroll
        for(int q = 0; q < Q; ++q) {
          const size_t c = static_cast<size_t>(min(k0 + k + STEP * q, kend - 1)) * ld;
          r[q].x         = p0[c];
          r[q].y         = p1[c];
        }
      }
    } else {
      if(kend % 2 == 0 || k0 + kTileK <= kend) {
        const V* p = P + min(k0 + k, kend - 2);
#pragma unroll
        for(int q = 0; q < Q; ++q)
          r[q] = *reinterpret_cast<const vec2_t<V>*>(
              p + static_cast<size_t>(min(o0 + o + STEP * q, O - 1)) * ld);
      } else {
        const int c0 = min(k0 + k, kend - 1), c1 = min(k0 + k + 1, kend - 1);
#pragma unroll
        for(int q = 0; q < Q; ++q) {
          const V* c = P + static_cast<size_t>(min(o0 + o + STEP * q, O - 1)) * ld;
          r[q].x     = c[c0];
          r[q].y     = c[c1];
        }
      }
    }
  }

  template <bool NEG>
  __device__ __forceinline__ void store(V* S, int k0, int kend) const {
#pragma unroll
    for(int q = 0; q < Q; ++q) {
      const int  kq = KFAST ? k : k + STEP * q, oq = KFAST ? o + STEP * q : o;
      const bool ix = o0 + oq < O && k0 + kq < kend;
      const bool iy = KFAST ? o0 + oq < O && k0 + kq + 1 < kend
                            : o0 + oq + 1 < O && k0 + kq < kend;
      vec2_t<V>  x;
      x.x = ix ? (NEG ? -r[q].x : r[q].x) : V(0);
      x.y = iy ? (NEG ? -r[q].y : r[q].y) : V(0);
      if constexpr(KFAST) {
        S[kq * LD + oq]       = x.x;
        S[(kq + 1) * LD + oq] = x.y;
      } else {
        *reinterpret_cast<vec2_t<V>*>(S + kq * LD + oq) = x;
      }
    }
  }
};

template <typename V, int BM, int BN>
struct TileShared {
  alignas(16) V a[kTileK * (BM + 2)];
  alignas(16) V b[kTileK * (BN + 2)];
};

// Tile `tile` (rows first within groups of kGroupM tile rows; of a LOWER_A product,
// whose row tiles have K bounds of their own, the longest first) of C (M x N) =
// beta C + alpha op(A) op(B), BM x BN on 4 waves in 2 x 2 (t: the thread among
// them), for 16-byte aligned operands with even leading dimensions (TA / TB:
// stored transposed): K in 32-deep stages through one LDS buffer (the next stage's
// loads are in flight in registers meanwhile), C loaded along with the first
// stage.  Every element is the sum over the same MFMA steps as in
// k_gemm.hip's dgemm_kernel, so the two give the same bits (but for zeros of
// op(A)'s upper triangle times values that are not finite).  Not `live`:
// nothing is stored (its barriers are).
//
// Bound by latency (a load, a stage's MFMAs and the store, one after the
// other) or, tall and thin, by C's and A's traffic.
template <typename V, bool BETA0, bool NEG, bool LOWER_A, int BM, int BN, bool TA = false,
          bool TB = false>
__device__ __forceinline__ void gemm_tile(int t, int tile, bool live, int M, int N, int K,
                                          const V* __restrict__ A, int lda,
                                          const V* __restrict__ B, int ldb,
                                          V* __restrict__ C, int ldc, int tiles_m,
                                          int tiles_n, TileShared<V, BM, BN>& sh) {
  constexpr int BKS = kTileK, LA = BM + 2, LB = BN + 2;
  constexpr int TM = BM / 32, TN = BN / 32;
  int m0, n0;
  if constexpr(LOWER_A) {
    m0 = (tiles_m - 1 - tile / tiles_n) * BM;
    n0 = tile % tiles_n * BN;
  } else {
    const int width  = kGroupM * tiles_n;
    const int group  = tile / width;
    const int firstm = group * kGroupM;
    const int gsz    = min(tiles_m - firstm, kGroupM);
    const int within = tile - group * width;
    m0 = (firstm + within % gsz) * BM;
    n0 = within / gsz * BN;
  }
  const int kend   = LOWER_A ? min(K, m0 + BM) : K;

  const int lane = t & 63, wave = t >> 6;
  const int l16 = lane & 15, lk = lane >> 4;
  const int wm0 = (wave & 1) * (BM / 2), wn0 = (wave >> 1) * (BN / 2);

  TileOperand<V, BM, TA>  la(A, lda, m0, M, t);
  TileOperand<V, BN, !TB> lb(B, ldb, n0, N, t);
  la.load(0, kend);
  lb.load(0, kend);
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
    la.template store<NEG>(sh.a, k0, kend);
    lb.template store<false>(sh.b, k0, kend);
    __syncthreads();
    if(k0 + BKS < kend) {
      la.load(k0 + BKS, kend);
      lb.load(k0 + BKS, kend);
    }
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
