// A 64 x 64 triangle solved for 4 right-hand sides by one wave, by
// substitution: lane (m, g) = (lane % 16, lane / 16) holds rows m, 16 + m, 32 +
// m and 48 + m of the g-th right-hand side, a solved value reaches the other
// rows by a broadcast within each 16 lanes that is part of the FMA (DPP), and
// the triangle comes from LDS.  Every row takes its FMAs in the order of the
// columns, one after the other, as in a substitution written out.
//
// Bound by the chain of 64 dependent FMAs and the 96 others in between, about
// 0.7 us; with the broadcasts as lane shuffles and one right-hand side a wave
// it was four times that for each.
//
// The triangle's zeros take part: a solved value that is exactly -0 may become +0
// (no other value changes, and what is not finite is solved again without them).
//
// "Positions" are rows in the order they are solved (from the last row for a
// backward solve).
#pragma once

#include <hip/hip_runtime.h>

#include <utility>

namespace hplx {
namespace tri {

// The triangle in LDS holds, of its columns in pairs, the positions from 16 (c
// / 16) on; the index of the entry at position p is tri_col(c) + 2 p.
__host__ __device__ constexpr int tri_col(int c) {
  const int b = c / 16;  // 16 columns of 64, of 48, of 32, of 16 entries
  return 16 * (64 * b - 8 * b * (b - 1)) + (c - 16 * b) / 2 * 2 * (64 - 16 * b) -
         32 * b + (c & 1);
}
constexpr int kTri = 16 * (64 + 48 + 32 + 16);

// x[s] += u_J m[s], s = S .. 3, for column 16 S + J: u_J is lane J's of each 16
// lanes, m is -T(., column), zero up to the diagonal.  One asm per column, the
// rows further on first: s_nop covers a VALU write of u just before.  Every
// lane has to be active.  The second form takes x[S] itself for u.
#define HPLX_FMA(type, y, x, m, j) \
  "v_fmac_" type "_dpp %" #y ", %" #x ", %" #m \
  " row_newbcast:%" #j " row_mask:0xf bank_mask:0xf\n\t"
#define HPLX_TRI_COLUMN(V, type)                                                  \
  template <int S, int J>                                                        \
  __device__ __forceinline__ void tri_column(V(&x)[4], V u, const V(&m)[4]) {    \
    if constexpr(S == 0)                                                         \
      asm("s_nop 1\n\t" HPLX_FMA(type, 1, 8, 5, 9) HPLX_FMA(type, 2, 8, 6, 9)    \
              HPLX_FMA(type, 3, 8, 7, 9) HPLX_FMA(type, 0, 8, 4, 9)              \
          : "+v"(x[0]), "+v"(x[1]), "+v"(x[2]), "+v"(x[3])                       \
          : "v"(m[0]), "v"(m[1]), "v"(m[2]), "v"(m[3]), "v"(u), "n"(J));         \
    if constexpr(S == 1)                                                         \
      asm("s_nop 1\n\t" HPLX_FMA(type, 1, 6, 4, 7) HPLX_FMA(type, 2, 6, 5, 7)    \
              HPLX_FMA(type, 0, 6, 3, 7)                                         \
          : "+v"(x[1]), "+v"(x[2]), "+v"(x[3])                                   \
          : "v"(m[1]), "v"(m[2]), "v"(m[3]), "v"(u), "n"(J));                    \
    if constexpr(S == 2)                                                         \
      asm("s_nop 1\n\t" HPLX_FMA(type, 1, 4, 3, 5) HPLX_FMA(type, 0, 4, 2, 5)    \
          : "+v"(x[2]), "+v"(x[3])                                               \
          : "v"(m[2]), "v"(m[3]), "v"(u), "n"(J));                               \
    if constexpr(S == 3)                                                         \
      asm("s_nop 1\n\t" HPLX_FMA(type, 0, 2, 1, 3)                               \
          : "+v"(x[3])                                                           \
          : "v"(m[3]), "v"(u), "n"(J));                                          \
  }                                                                              \
  template <int S, int J>                                                        \
  __device__ __forceinline__ void tri_column(V(&x)[4], const V(&m)[4]) {         \
    if constexpr(S == 0)                                                         \
      asm("s_nop 1\n\t" HPLX_FMA(type, 1, 0, 5, 8) HPLX_FMA(type, 2, 0, 6, 8)    \
              HPLX_FMA(type, 3, 0, 7, 8) HPLX_FMA(type, 0, 0, 4, 8)              \
          : "+v"(x[0]), "+v"(x[1]), "+v"(x[2]), "+v"(x[3])                       \
          : "v"(m[0]), "v"(m[1]), "v"(m[2]), "v"(m[3]), "n"(J));                 \
    if constexpr(S == 1)                                                         \
      asm("s_nop 1\n\t" HPLX_FMA(type, 1, 0, 4, 6) HPLX_FMA(type, 2, 0, 5, 6)    \
              HPLX_FMA(type, 0, 0, 3, 6)                                         \
          : "+v"(x[1]), "+v"(x[2]), "+v"(x[3])                                   \
          : "v"(m[1]), "v"(m[2]), "v"(m[3]), "n"(J));                            \
    if constexpr(S == 2)                                                         \
      asm("s_nop 1\n\t" HPLX_FMA(type, 1, 0, 3, 4) HPLX_FMA(type, 0, 0, 2, 4)    \
          : "+v"(x[2]), "+v"(x[3])                                               \
          : "v"(m[2]), "v"(m[3]), "n"(J));                                       \
    if constexpr(S == 3)                                                         \
      asm("s_nop 1\n\t" HPLX_FMA(type, 0, 0, 1, 2)                               \
          : "+v"(x[3])                                                           \
          : "v"(m[3]), "n"(J));                                                  \
  }
HPLX_TRI_COLUMN(double, "f64")
HPLX_TRI_COLUMN(float, "f32")
#undef HPLX_TRI_COLUMN
#undef HPLX_FMA

// Columns 16 S + 2 J2 and the next; p: the triangle + 2 (lane % 16).  UNIT: the
// diagonal is one (or the rows are already divided by it); else d is its value
// in this lane's row 16 S + lane % 16 and every solved value is divided by it.
template <int S, bool UNIT, int J2, typename V>
__device__ __forceinline__ void tri_pair(V (&x)[4], const V* p, V d) {
  constexpr int c = tri_col(16 * S + 2 * J2);
  typedef V     V2 __attribute__((ext_vector_type(2)));
  V             m0[4], m1[4];
#pragma unroll
  for(int s = S; s < 4; ++s) {
    const V2 v = *reinterpret_cast<const V2*>(p + c + 32 * s);
    m0[s]      = v.x;
    m1[s]      = v.y;
  }
  if constexpr(UNIT) {
    tri_column<S, 2 * J2>(x, m0);
    tri_column<S, 2 * J2 + 1>(x, m1);
  } else {
    const int m = threadIdx.x & 15;
    V         u = x[S] / d;
    tri_column<S, 2 * J2>(x, u, m0);
    x[S] = m == 2 * J2 ? u : x[S];
    V w  = x[S] / d;
    tri_column<S, 2 * J2 + 1>(x, w, m1);
    x[S] = m == 2 * J2 + 1 ? w : x[S];
  }
}
template <int S, bool UNIT, typename V, int... J2>
__device__ __forceinline__ void tri_pairs(V (&x)[4], const V* p, V d,
                                          std::integer_sequence<int, J2...>) {
  (tri_pair<S, UNIT, J2>(x, p, d), ...);
}
// Columns 16 S .. 16 S + 15.
template <int S, bool UNIT = true, typename V>
__device__ __forceinline__ void tri_columns(V (&x)[4], const V* p, V d = V(1)) {
  tri_pairs<S, UNIT>(x, p, d, std::make_integer_sequence<int, 8>());
}

}  // namespace tri
}  // namespace hplx
