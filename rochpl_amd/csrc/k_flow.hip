// Triangular solves with a whole matrix of right-hand sides, as a dataflow of
// 128-row blocks: one launch per panel of L (whose interchanges separate the
// panels) and one per up to kFlowBlocks blocks of U, instead of a solve of
// every diagonal block by one workgroup per right-hand side and a product
// after it (HPL_pdtrsv, src/pgesv/HPL_pdtrsv_device.cpp:169-332, and the
// solves hplx_pdgetrs and hplx_pdgesv_adjoint add).
//
// A workgroup owns a block of 128 rows and a slice of 16 or 4 right-hand
// sides.  It keeps its block of B in MFMA accumulators, subtracts op(T)_ij x_j
// for the solved 64-row halves j in dependency order as they appear
// (V_MFMA_F64_16X16X4_F64 or _4X4X4_4B_F64, T straight from memory into the operand
// registers, one half ahead), and, if the block lies on the diagonal, solves
// its two 64 x 64 triangles by substitution, with the product between them,
// and publishes x_i.  (Products with the triangles' inverses take about as
// long, but their errors grow with the triangles' condition: the factors of a
// Gaussian kernel matrix of order 1000 gave a backward error of 8e-6 with
// them, 1.4e-16 with the substitution.)
//
// Progress.  A workgroup waits only for blocks of smaller index, and the
// dispatcher hands out workgroups in index order on every XCD, so the
// unfinished workgroup of the smallest index never waits: the grid need not
// be resident at once.  The waits are bounded all the same: past the limit of
// one wait a workgroup raises *err and goes on with NaNs.
//
// x_i travels through an exchange buffer that the call fills with a NaN of a
// payload of its own first (fill_kernel), and then a flag is raised.  The
// next block of the chain polls the values themselves, by device-scope
// accesses, until none is that NaN: a step needs one store-to-load trip
// through memory and no cache write-back or invalidation.  The blocks
// further on are not in a hurry: they poll the flag at leisure and then read
// x_i through their L2 (U of N = 16384 with 64 right-hand sides in 64-row
// blocks: 2243 us with all of them polling the values, 1220 us so).  The flag
// is a hint only: nothing orders it with what a block's L2 may hold, so what
// they read is checked for that NaN like a poll, and polled for if it is there.
// Nothing outlives the call, so the launches can be captured and replayed.
//
// Bound by latency: a step of the chain is two substitutions of 64 rows (each
// 64 dependent FMAs on broadcast values), two products of 64 columns and that
// trip, 4.6 us in all for narrow slices, 8.7 for wide ones.  128-row blocks
// rather than 64-row ones: half the trips (that U 1115 us).
//
// hplx_pdgetrs, before and now: N = 16384, NB = 512, 64 right-hand sides 9.50
// -> 2.70 ms (transposed 8.92 -> 3.45), one 9.27 -> 1.58, 512 15.2 -> 8.0;
// N = 5000, NB = 128, one 2.87 -> 0.70 ms.  The floor is one read of the
// factors (2.1 GB, 0.4 ms).
#include "hplx_internal.hpp"
#include "lds_stream.hpp"
#include "tri_chain.hpp"

namespace hplx {
namespace {

using namespace tri;

typedef double ud4 __attribute__((ext_vector_type(4)));
// two neighbouring doubles at any 8-byte address
typedef double d2u __attribute__((ext_vector_type(2), aligned(8)));

constexpr int kFB  = 128;  // rows of a block
constexpr int kFH  = 64;   // and of its halves
constexpr int kXcdBits = 3;
constexpr int kFLd = 66;   // LDS pitch of a right-hand side of a half
constexpr int kNext = 1;   // blocks ahead in the chain that poll the values
// Narrow slices (4 right-hand sides) while at most this many workgroups come
// of it, 2 per CU: a step takes 4.6 instead of 8.7 us, but every slice reads
// all of T (N = 16384: 16 right-hand sides 2.04 against 2.21 ms, 24 2.31
// against 2.21).
constexpr int kNarrowGrid = 512;
// From this many right-hand sides on the rows off the diagonal blocks of
// kSplitRows rows are updated by a GEMM, which reads T once per 64 of them.
constexpr int kSplitRhs = 192, kSplitRows = 512;
struct FlowArgs {
  const double* T;
  int           ldt;
  double*       B;
  int           ldb, nrhs;
  int           d0, d1;  // rows of the diagonal blocks
  int           o0, o1;  // rows of the others, updated only
  int           nd, nt;  // blocks on the diagonal, in all
  int           ns;      // slices of 16 or 4 right-hand sides
  int           xcd_bits;  // 2^these XCDs take turns at the blocks
  unsigned long long* x;      // nd x ns blocks of 2 halves of 16 x 64 values
  int*                flags;  // nd x ns
  int*                err;    // FlowScratch's
  uint32_t            polls;
  // The interchanges of a panel of L, applied as B is loaded (null: none): perm
  // as launch_pipid composes it, relative to d0; top: the panel's rows of B as
  // they were before it (leading dimension d1 - d0), whose places in B the
  // solved blocks take; next: where the first rows below go for the next panel
  // (next_rows of them; null: nowhere).
  const int*    perm;
  const double* top;
  double*       next;
  int           next_rows;
};

// The exchange buffer's filling: a NaN no computed value has (those that
// would be published are replaced by the plain quiet NaN).
constexpr unsigned long long kEmpty = 0x7ff8b10cffffb10cull;

// None of a wave's values is the filling.
template <int W>
__device__ __forceinline__ bool all_there(const unsigned long long (&v)[W]) {
  bool in = true;
#pragma unroll
  for(int q = 0; q < W; ++q) in = in && v[q] != kEmpty;
  return __all(in);
}

// Also copies the first `rows` rows of B's nrhs columns to top, if it is not
// null.
__global__ __launch_bounds__(256) void fill_kernel(unsigned long long* p, int n,
                                                   int* flags, int nf, int raised,
                                                   const double* B, int ldb, int nrhs,
                                                   double* top, int rows) {
  const int i0 = blockIdx.x * 256 + threadIdx.x;
  for(int i = i0; i < n; i += gridDim.x * 256) p[i] = kEmpty;
  if(i0 < nf) flags[i0] = raised;
  if(top)
    for(int i = i0; i < rows * nrhs; i += gridDim.x * 256)
      top[i] = B[i % rows + static_cast<size_t>(i / rows) * ldb];
}

// A wave's 16 rows x 64 columns of op(T): lane (m, g) holds T(row0 + m,
// col0 + 16 g + s), s = 0 .. 15 (the MFMA's k index is 4 s' + g in any
// order, as long as both operands agree).  nr / nc: rows and columns inside;
// the others are zero and read nothing.
template <bool TRANS>
__device__ __forceinline__ void load_block(const double* __restrict__ T, int ldt,
                                           int row0, int nr, int col0, int nc,
                                           double (&t)[16]) {
  const int lane = threadIdx.x & 63, m = lane & 15, g = lane >> 4;
  if(nr >= 16 && nc >= kFH) {
    if(TRANS) {
      const double* p = T + col0 + 16 * g + static_cast<size_t>(row0 + m) * ldt;
#pragma unroll
      for(int s = 0; s < 16; s += 2) {
        const d2u v = *reinterpret_cast<const d2u*>(p + s);
        t[s]     = v.x;
        t[s + 1] = v.y;
      }
    } else {
      // uniform column starts plus one 32-bit offset per lane
      const double*  p   = T + row0 + static_cast<size_t>(col0) * ldt;
      const uint32_t off = static_cast<uint32_t>(m + 16 * g * ldt);
#pragma unroll
      for(int s = 0; s < 16; ++s) t[s] = (p + static_cast<size_t>(s) * ldt)[off];
    }
    return;
  }
  if(nr <= 0 || nc <= 0) {
#pragma unroll
    for(int s = 0; s < 16; ++s) t[s] = 0.0;
    return;
  }
  // an edge: clamped addresses, then zeros
  const double* p  = T + (TRANS ? col0 + static_cast<size_t>(row0) * ldt
                                : row0 + static_cast<size_t>(col0) * ldt);
  const int     mr = m < nr ? m : nr - 1;
#pragma unroll
  for(int s = 0; s < 16; ++s) {
    const int c  = 16 * g + s, cr = c < nc ? c : nc - 1;
    const double v = p[static_cast<uint32_t>(TRANS ? cr + mr * ldt : mr + cr * ldt)];
    t[s] = m < nr && c < nc ? v : 0.0;
  }
}

// T x for the wave's 16 rows and a slice of right-hand sides (xs: [column]
// [row], 64 rows).  Wide: 16 columns, V_MFMA_F64_16X16X4_F64; narrow: 4
// columns, V_MFMA_F64_4X4X4_4B_F64 (its four blocks four rows each), a
// quarter of the time.  A lane holds kE values: row(e), col().
template <bool WIDE>
struct Product;
template <>
struct Product<true> {
  static constexpr int kR = 16, kE = 4;
  typedef ud4          Acc;
  __device__ static int row(int e) { return 4 * e + ((threadIdx.x & 63) >> 4); }
  __device__ static int col() { return threadIdx.x & 15; }
  __device__ static ud4 zero() { return ud4{0.0, 0.0, 0.0, 0.0}; }
  __device__ static ud4 mfma(double t, double x, ud4 acc) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(t, x, acc, 0, 0, 0);
  }
};
typedef double ud1 __attribute__((ext_vector_type(1)));
template <>
struct Product<false> {
  static constexpr int kR = 4, kE = 1;
  typedef ud1          Acc;
  __device__ static int row(int) {
    return 4 * ((threadIdx.x >> 2) & 3) + ((threadIdx.x & 63) >> 4);
  }
  __device__ static int col() { return threadIdx.x & 3; }
  __device__ static ud1 zero() { return ud1{0.0}; }
  __device__ static ud1 mfma(double t, double x, ud1 acc) {
    return ud1{__builtin_amdgcn_mfma_f64_4x4x4f64(t, x, acc.x, 0, 0, 0)};
  }
};

template <bool WIDE>
__device__ __forceinline__ typename Product<WIDE>::Acc block_product(
    const double (&t)[16], const double* xs) {
  typedef Product<WIDE> P;
  const double* x = xs + P::col() * kFLd + 16 * ((threadIdx.x & 63) >> 4);
  double        xf[16];
#pragma unroll
  for(int s = 0; s < 16; ++s) xf[s] = x[s];
  typename P::Acc acc = P::zero();
#pragma unroll
  for(int s = 0; s < 16; ++s) acc = P::mfma(t[s], xf[s], acc);
  return acc;
}

constexpr double kHuge = 1.7976931348623157e308;

// The triangles of a diagonal block's two halves, in the order they are
// solved, as tri_columns takes them: divided by the diagonal and negated,
// zero up to the diagonal.  scale: the diagonal's reciprocals.  rare is set
// if one of them is not an ordinary number.  t: the block's first entry, w
// its rows.  L (its unit diagonal is not read) is what is solved forward as it
// lies or backward transposed.
template <bool TRANS, bool BACK>
__device__ __forceinline__ void stage_triangle(const double* __restrict__ t, int ldt, int w,
                                               double* tri, double* scale, int* rare) {
  constexpr bool UNIT = TRANS == BACK;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int h = wave >> 2, r0 = kFH * (BACK ? 1 - h : h);
  auto row = [&](int p) { return r0 + (BACK ? kFH - 1 - p : p); };
  auto at  = [&](int i, int j) {  // of a row and a column inside
    i = min(i, w - 1), j = min(j, w - 1);
    return t[TRANS ? j + static_cast<size_t>(i) * ldt : i + static_cast<size_t>(j) * ldt];
  };
  // a line of op(T) along memory per wave: a column, or a row of the
  // transposed
  double v[16];
#pragma unroll
  for(int q = 0; q < 16; ++q) {
    const int k = 4 * q + (wave & 3);
    v[q]        = TRANS ? at(row(k), row(lane)) : at(row(lane), row(k));
  }
  const int    mr = row(lane);
  const double d  = UNIT || mr >= w ? 1.0 : at(mr, mr);
  if((wave & 3) == 0) {
    scale[kFH * h + lane] = 1.0 / d;
    if(!(fabs(d) >= 0x1p-1000 && fabs(d) <= 0x1p1000)) *rare = 1;
  }
#pragma unroll
  for(int q = 0; q < 16; ++q) {
    const int    k = 4 * q + (wave & 3);
    const int    p = TRANS ? k : lane, c = TRANS ? lane : k;
    const double e = UNIT ? v[q] : v[q] / (TRANS ? __shfl(d, k) : d);
    if(p >= (c & ~15))
      tri[h * kTri + tri_col(c) + 2 * p] = p > c && row(p) < w && row(c) < w ? -e : 0.0;
  }
}

// A half by plain substitution, for what tri_columns cannot take: a diagonal
// whose reciprocal is not an ordinary number, or values that are not finite
// (whose products with its zeros are not zero).
template <bool TRANS, bool BACK>
__device__ __forceinline__ void solve_half(const double* __restrict__ t, int ldt, int r0,
                                        int left, const double* xc, double (&v)[4]) {
  constexpr bool UNIT = TRANS == BACK;
  const int lane = threadIdx.x & 63, m = lane & 15;
#pragma unroll
  for(int s = 0; s < 4; ++s) v[s] = xc[BACK ? kFH - 1 - (16 * s + m) : 16 * s + m];
  for(int p = 0; p < kFH; ++p) {
    const int j = BACK ? kFH - 1 - p : p;
    if(j >= left) continue;
    const double* tj = t + r0 + static_cast<size_t>(r0) * ldt;
    double        xj = 0.0;
#pragma unroll
    for(int s = 0; s < 4; ++s)
      if((p >> 4) == s) {
        xj = __shfl(v[s], p & 15, 16);
        if(!UNIT) xj = xj / tj[j + static_cast<size_t>(j) * ldt];
        if(m == (p & 15)) v[s] = xj;
      }
#pragma unroll
    for(int s = 0; s < 4; ++s) {
      const int q = 16 * s + m, i = BACK ? kFH - 1 - q : q;
      if(q > p && i < left)
        v[s] = fma(-tj[TRANS ? j + static_cast<size_t>(i) * ldt
                             : i + static_cast<size_t>(j) * ldt],
                   xj, v[s]);
    }
  }
}

// TRANS: op(T) = T^T.  BACK: the diagonal blocks are solved from the last.
template <bool TRANS, bool BACK, bool WIDE>
__global__ __launch_bounds__(512) void flow_kernel(FlowArgs a) {
  typedef Product<WIDE> P;
  constexpr int         R = P::kR, E = P::kE, W = (R + 7) / 8;
  constexpr bool        UNIT = TRANS == BACK;
  __shared__ __attribute__((aligned(16))) double xs[2][R * kFLd];
  __shared__ __attribute__((aligned(16))) double tri[2 * kTri];
  __shared__ double scale[2 * kFH];
  __shared__ int    rare;
  __shared__ int    from[kFB];  // where the block's rows of B come from
  // blocks in index order; the slices of a block on one XCD (they read the same
  // rows of T), unless the blocks are too few for all XCDs (N = 100 with
  // 1000 right-hand sides, one block: 144 us a call on one XCD, 44 spread)
  const int xb  = a.xcd_bits;
  const int per = a.ns << xb, bg = blockIdx.x / per, br = blockIdx.x - bg * per;
  const int sl = br >> xb, i = (bg << xb) + (br & ((1 << xb) - 1));
  if(i >= a.nt) return;
  const int t = threadIdx.x, lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int ac = P::col();  // this lane's right-hand side
  const int c0 = sl * R, nc = min(R, a.nrhs - c0);
  auto diag_row = [&](int k) { return a.d0 + kFB * (BACK ? a.nd - 1 - k : k); };
  const bool diag = i < a.nd;
  const int  r = diag ? diag_row(i) : a.o0 + kFB * (i - a.nd);
  const int  w = min(kFB, (diag ? a.d1 : a.o1) - r);
  const int  r0 = r + 16 * wave, nr = w - 16 * wave;  // this wave's rows
  // the solved halves in the order they appear: half h of block k is rows
  // [half_row, + 64)
  const int steps = 2 * (diag ? i : a.nd);
  auto half_row = [&](int st) {
    return diag_row(st >> 1) + kFH * (BACK ? 1 - (st & 1) : st & 1);
  };

  double*         Bc = a.B + r0 + static_cast<size_t>(c0 + ac) * a.ldb;
  // the products are summed by themselves and added to B at the end
  typename P::Acc acc = P::zero(), b = P::zero();
  bool swap = false;
  if constexpr(!TRANS && !BACK) swap = a.perm != nullptr;
  if(swap) {
    // from: a row of top (>= 0) or of B (< 0: minus the row from d0, minus 1)
    const int jb = a.d1 - a.d0;
    if(t < kFB) {
      const int q = r - a.d0 + t;  // the row, from d0
      const int f = diag ? (t < w ? a.perm[q] : 0) : q;
      from[t]     = f < jb ? f : -f - 1;
    }
    __syncthreads();
    if(!diag)  // the panel's rows that were moved into this block
      for(int k = t; k < jb; k += 512) {
        const int q = a.perm[jb + k] - (r - a.d0);
        if(q >= 0 && q < w) from[q] = k;
      }
    __syncthreads();
#pragma unroll
    for(int e = 0; e < E; ++e)
      if(P::row(e) < nr && ac < nc) {
        const int f = from[16 * wave + P::row(e)];
        b[e]        = f >= 0 ? a.top[f + static_cast<size_t>(c0 + ac) * jb]
                             : a.B[a.d0 - f - 1 + static_cast<size_t>(c0 + ac) * a.ldb];
      }
  } else {
#pragma unroll
    for(int e = 0; e < E; ++e)
      if(P::row(e) < nr && ac < nc) b[e] = Bc[P::row(e)];
  }
  double tv[16], tn[16];
  if(diag) {
    if(t == 0) rare = 0;
    __syncthreads();
    stage_triangle<TRANS, BACK>(a.T + r + static_cast<size_t>(r) * a.ldt, a.ldt, w, tri,
                                scale, &rare);
  }
  // the second half of a block on the diagonal has one more product to form,
  // with its own first half
  const bool second = diag && (BACK ? wave < 4 : wave >= 4);
  const int  mine   = steps + (second ? 1 : 0);
  if(mine > 0) {
    const int cj = half_row(0);
    load_block<TRANS>(a.T, a.ldt, r0, nr, cj, min(kFH, a.d1 - cj), tn);
  }
  bool dead = false;
  for(int st = 0; st < steps; ++st) {
#pragma unroll
    for(int s = 0; s < 16; ++s) tv[s] = tn[s];
    // x of this half into LDS: wave w columns w, w + 8
    const int           j  = st >> 1;
    unsigned long long* xj = a.x + (static_cast<size_t>(2 * j + (st & 1)) * a.ns + sl) *
                                       (R * kFH) + kFH * wave + lane;
    unsigned long long  xv[W];
    const bool          next = diag && j + kNext >= i;
    // polls the values until all are there
    auto poll = [&]() {
      bool in = false;
      for(uint32_t polls = 0; !in && !dead;) {
#pragma unroll
        for(int q = 0; q < W; ++q)
          xv[q] = __hip_atomic_load(xj + 8 * kFH * q, __ATOMIC_RELAXED,
                                    __HIP_MEMORY_SCOPE_AGENT);
        in = all_there(xv);
        if(!in) dead = ++polls > a.polls;
      }
    };
    if(wave < R) {
      if(next) {
        __builtin_amdgcn_s_setprio(3);
        poll();
      } else {
        const int* flag = a.flags + j * a.ns + sl;
        uint32_t   polls = 0;
        while(!dead && !__hip_atomic_load(flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) {
          dead = ++polls > a.polls;
          __builtin_amdgcn_s_sleep(8);
        }
        asm volatile("" : : : "memory");  // the values are read after the flag
#pragma unroll
        for(int q = 0; q < W; ++q)
          xv[q] = __hip_atomic_load(xj + 8 * kFH * q, __ATOMIC_RELAXED,
                                    __HIP_MEMORY_SCOPE_WORKGROUP);
      }
    }
    if(st + 1 < mine) {
      const int cn = half_row(st + 1);
      load_block<TRANS>(a.T, a.ldt, r0, nr, cn, min(kFH, a.d1 - cn), tn);
    }
    double* x = xs[st & 1];
    if(wave < R) {
      auto put = [&]() {
#pragma unroll
        for(int q = 0; q < W; ++q)
          x[(wave + 8 * q) * kFLd + lane] =
              -__longlong_as_double(static_cast<long long>(xv[q]));
      };
      put();
      // what was read after a flag is checked only now, out of the loads' way (N =
      // 16384, 64 right-hand sides 2.73 ms checked before T's loads, 2.71 so)
      if(!next && !all_there(xv)) {
        poll();
        put();
      }
      if(dead) {
        if(a.err && lane == 0)
          __hip_atomic_store(a.err, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
#pragma unroll
        for(int q = 0; q < W; ++q) xv[q] = 0x7ff8000000000000ull;
        put();
      }
    }
    __syncthreads();  // this buffer is written again two barriers on
    // a half's sum is formed by itself: N / 64 roundings at the magnitude of
    // the whole instead of N
    acc += block_product<WIDE>(tv, x);
  }
  if(!diag) {
    // (a row that a block on the diagonal takes from here was read before that
    // block's x appeared)
#pragma unroll
    for(int e = 0; e < E; ++e)
      if(P::row(e) < nr && ac < nc) {
        const double v = b[e] + acc[e];
        const int    q = r0 - a.d1 + P::row(e);
        Bc[P::row(e)]  = v;
        if(swap && q < a.next_rows) a.next[q + static_cast<size_t>(c0 + ac) * a.next_rows] = v;
      }
    return;
  }
  for(int h = 0; h < 2; ++h) {
    // the half's right-hand sides into LDS, in the order of their positions
    const int half = BACK ? 1 - h : h, left = w - kFH * half;
    double*   x    = xs[0];
    __syncthreads();  // the last products have read xs
    if((wave >> 2) == half)
#pragma unroll
      for(int e = 0; e < E; ++e) x[ac * kFLd + 16 * (wave & 3) + P::row(e)] = b[e] + acc[e];
    __syncthreads();
    // 4 right-hand sides a wave, lane (m, g): rows m, 16 + m, ... in solving
    // order of the g-th
    if(wave < R / 4) {
      const int     m = lane & 15, c = 4 * wave + (lane >> 4);
      const double* p = tri + h * kTri + 2 * m;
      double        v[4];
      double*       xc = x + c * kFLd;
#pragma unroll
      for(int s = 0; s < 4; ++s) {
        const int q = 16 * s + m;
        v[s]        = xc[BACK ? kFH - 1 - q : q] * (UNIT ? 1.0 : scale[kFH * h + q]);
      }
      tri_columns<0>(v, p);
      tri_columns<1>(v, p);
      tri_columns<2>(v, p);
      tri_columns<3>(v, p);
      const bool fine = fabs(v[0]) <= kHuge && fabs(v[1]) <= kHuge && fabs(v[2]) <= kHuge &&
                        fabs(v[3]) <= kHuge;
      // which path a right-hand side takes does not depend on the others
      const unsigned long long bad = __ballot(rare || !fine);
      if(bad) {
        double u[4];
        solve_half<TRANS, BACK>(a.T + r + static_cast<size_t>(r) * a.ldt, a.ldt, kFH * half,
                                left, xc, u);
        // past the block's rows nothing, whatever infinite values made of their
        // zeros: the rows further on multiply them by zeros of T
        if((bad >> (lane & 48)) & 0xffff)
#pragma unroll
          for(int s = 0; s < 4; ++s)
            v[s] = (BACK ? kFH - 1 - (16 * s + m) : 16 * s + m) < left ? u[s] : 0.0;
      }
      unsigned long long* xi =
          a.x + (static_cast<size_t>(2 * i + h) * a.ns + sl) * (R * kFH) + c * kFH;
#pragma unroll
      for(int s = 0; s < 4; ++s) {
        const int q = BACK ? kFH - 1 - (16 * s + m) : 16 * s + m;
        __hip_atomic_store(
            xi + q,
            v[s] == v[s] ? static_cast<unsigned long long>(__double_as_longlong(v[s]))
                         : 0x7ff8000000000000ull,
            __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
#pragma unroll
      for(int s = 0; s < 4; ++s) {
        const int q = BACK ? kFH - 1 - (16 * s + m) : 16 * s + m;
        xc[q]       = -v[s];
        if(q < left && c < nc) a.B[r + kFH * half + q + static_cast<size_t>(c0 + c) * a.ldb] = v[s];
      }
      wait_vm<0>();  // the values have reached the device's memory
    }
    __syncthreads();
    if(h == 0 && second) acc += block_product<WIDE>(tn, x);
  }
  if(t == 0)
    __hip_atomic_store(a.flags + i * a.ns + sl, 1, __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_AGENT);
}

// A panel's interchanges and where its rows of B are kept (FlowArgs).
struct FlowSwap {
  const int*    perm      = nullptr;
  const double* top       = nullptr;
  double*       next      = nullptr;
  int           next_rows = 0;
};

// The solves of one call on a stream, for at most as many right-hand sides as
// getrs_enqueue takes at once.
struct Flow {
  hipStream_t        s;
  const double*      T;
  int                ldt;
  double*            B;
  int                ldb, nrhs, rows;  // rows: of T
  const FlowScratch& w;

  bool wide() const {
    return static_cast<long>((rows + kFB - 1) / kFB) * ((nrhs + 3) / 4) > kNarrowGrid;
  }
  bool split() const { return nrhs >= kSplitRhs; }
  int  group() const { return wide() ? Product<true>::kR : Product<false>::kR; }
  int slices() const { return (nrhs + group() - 1) / group(); }
  // blocks whose x fit the exchange buffer
  int blocks() const {
    const size_t b = kFlowX / x_panel(1);
    return b < static_cast<size_t>(kFlowBlocks) ? static_cast<int>(b) : kFlowBlocks;
  }
  size_t x_panel(int bpp) const {
    return static_cast<size_t>(bpp) * slices() * group() * kFB;
  }

  // np panels' (of bpp blocks) x marked as not there yet, and the first `rows`
  // rows of B kept in top (if not null)
  hipError_t prepare(int np, int bpp, double* top = nullptr, int top_rows = 0) {
    if(np * bpp > blocks()) return hipErrorInvalidValue;
    const int n = static_cast<int>(x_panel(bpp)) * np;
    hipLaunchKernelGGL(fill_kernel, dim3(n < 256 * 1024 ? (n + 255) / 256 : 1024),
                       dim3(256), 0, s, w.x, n, w.flags, np * bpp * slices(), w.raised, B,
                       ldb, nrhs, top, top_rows);
    return hipGetLastError();
  }

  template <bool WIDE>
  void launch(bool trans, bool back, dim3 g, dim3 b, const FlowArgs& a) {
    if(trans && back)
      hipLaunchKernelGGL((flow_kernel<true, true, WIDE>), g, b, 0, s, a);
    else if(trans)
      hipLaunchKernelGGL((flow_kernel<true, false, WIDE>), g, b, 0, s, a);
    else if(back)
      hipLaunchKernelGGL((flow_kernel<false, true, WIDE>), g, b, 0, s, a);
    else
      hipLaunchKernelGGL((flow_kernel<false, false, WIDE>), g, b, 0, s, a);
  }

  // op(T) on rows [d0, d1) solved, then applied to rows [o0, o1); block: the
  // index of the first of these blocks among the prepared ones.
  hipError_t solve(bool trans, bool back, int d0, int d1, int o0, int o1,
                   int block, const FlowSwap& sw = FlowSwap()) {
    if(!split()) return flow(trans, back, d0, d1, o0, o1, block, sw);
    const int n = (d1 - d0 + kSplitRows - 1) / kSplitRows;
    for(int k = 0; k < n; ++k) {
      const int q  = back ? n - 1 - k : k;
      const int s0 = d0 + q * kSplitRows;
      const int s1 = s0 + kSplitRows < d1 ? s0 + kSplitRows : d1;
      hipError_t e =
          flow(trans, back, s0, s1, s0, s0, block + q * (kSplitRows / kFB), FlowSwap());
      // the rows of the diagonal range still to be solved, then the others
      if(e == hipSuccess) e = back ? update(trans, s0, s1, d0, s0) : update(trans, s0, s1, s1, d1);
      if(e == hipSuccess) e = update(trans, s0, s1, o0, o1);
      if(e != hipSuccess) return e;
    }
    return hipSuccess;
  }

  // rows [o0, o1) -= op(T) x for the solved rows [s0, s1)
  hipError_t update(bool trans, int s0, int s1, int o0, int o1) {
    if(o1 <= o0) return hipSuccess;
    if(trans)
      return launch_tn_sub(s, s1 - s0, o1 - o0, nrhs,
                           T + s0 + static_cast<size_t>(o0) * ldt, ldt, B + s0, ldb,
                           B + o0, ldb, w.work, w.work_doubles);
    return launch_nn_sub(s, s1 - s0, o1 - o0, nrhs,
                         T + o0 + static_cast<size_t>(s0) * ldt, ldt, B + s0, ldb,
                         B + o0, ldb);
  }

  hipError_t flow(bool trans, bool back, int d0, int d1, int o0, int o1, int block,
                  const FlowSwap& sw) {
    FlowArgs a;
    a.perm      = sw.perm;
    a.top       = sw.top;
    a.next      = sw.next;
    a.next_rows = sw.next_rows;
    a.T     = T;
    a.ldt   = ldt;
    a.x     = w.x + x_panel(block);
    a.flags = w.flags + block * slices();
    a.err   = w.err;
    a.polls = w.polls;
    a.B     = B;
    a.ldb   = ldb;
    a.nrhs  = nrhs;
    a.ns    = slices();
    a.d0    = d0;
    a.d1    = d1;
    a.o0    = o0;
    a.o1    = o1;
    a.nd    = (d1 - d0 + kFB - 1) / kFB;
    a.nt    = a.nd + (o1 - o0 + kFB - 1) / kFB;
    a.xcd_bits      = a.nt >> kXcdBits ? kXcdBits : 0;
    const long grid = ((a.nt + (1L << a.xcd_bits) - 1) >> a.xcd_bits << a.xcd_bits) * a.ns;
    if(block + a.nd > blocks() || grid > 0x7fffffffL) return hipErrorInvalidValue;
    const dim3 g(static_cast<unsigned>(grid)), b(512);
    if(wide())
      launch<true>(trans, back, g, b, a);
    else
      launch<false>(trans, back, g, b, a);
    return hipGetLastError();
  }

  // U x = b over rows [0, n): chunks from the bottom
  hipError_t upper(int n) {
    const int c = blocks() * kFB;
    for(int d0 = (n - 1) / c * c; d0 >= 0; d0 -= c) {
      const int  d1 = d0 + c < n ? d0 + c : n;
      hipError_t e  = prepare(1, (d1 - d0 + kFB - 1) / kFB);
      if(e == hipSuccess) e = solve(false, true, d0, d1, 0, d0, 0);
      if(e != hipSuccess) return e;
    }
    return hipSuccess;
  }

  // U^T x = b over rows [0, n)
  hipError_t upper_trans(int n) {
    const int c = blocks() * kFB;
    for(int d0 = 0; d0 < n; d0 += c) {
      const int  d1 = d0 + c < n ? d0 + c : n;
      hipError_t e  = prepare(1, (d1 - d0 + kFB - 1) / kFB);
      if(e == hipSuccess) e = solve(true, false, d0, d1, d1, n, 0);
      if(e != hipSuccess) return e;
    }
    return hipSuccess;
  }
};

}  // namespace

hipError_t launch_trsv(hipStream_t s, int n, const double* A, int lda, double* x,
                       const FlowScratch& w) {
  if(n <= 0) return hipSuccess;
  return Flow{s, A, lda, x, n, 1, n, w}.upper(n);
}

#define HCHK(expr)                  \
  do {                              \
    const hipError_t e_ = (expr);   \
    if(e_ != hipSuccess) return e_; \
  } while(0)

// At most as many right-hand sides as getrs_enqueue takes at once.
static hipError_t getrs_slices(hipStream_t s, const double* A, int N, int nb,
                               int lda, const int* ipiv, int trans, int nrhs,
                               double* B, int ldb, const FlowScratch& w) {
  if(N <= 0) return hipSuccess;
  if(nb > N) nb = N;  // one panel: any wider one is the same
  if(nb < 1 || nb > kMaxNB) return hipErrorInvalidValue;
  Flow f{s, A, lda, B, ldb, nrhs, N, w};
  const int np  = (N + nb - 1) / nb;
  const int bpp = (nb + kFB - 1) / kFB;
  const int pc  = f.blocks() / bpp;  // panels prepared at once
  // Few right-hand sides: a panel's interchanges are applied by the launch that
  // solves with it, its rows kept in one half of the work buffer while the
  // first rows below go to the other half for the next panel.  A launch of
  // their own took 4.6 us a panel (N = 5000, NB = 128, one right-hand side 0.74
  // ms with it, 0.69 without; N = 1000, NB = 64, five 0.226, 0.200).
  const size_t half  = static_cast<size_t>(nb) * nrhs;
  const bool   fused = !f.split() && 2 * half <= w.work_doubles;
  // panels [p0, p0 + pc): their exchange buffers, and the interchanges composed
  auto prepare = [&](int p0) -> hipError_t {
    const int p1 = p0 + pc < np ? p0 + pc : np;
    HCHK(f.prepare(p1 - p0, bpp, fused && !trans && p0 == 0 ? w.work : nullptr,
                   nb));
    return launch_pipid_panels(s, p1 - p0, nb, N - p0 * nb, ipiv + p0 * nb,
                               p0 * nb, w.perm);
  };
  if(!trans) {
    // L solve with the panel-by-panel interchanges, as b is carried through
    // the factorisation (HPL_pdgesv), then U x = y (HPL_pdtrsv)
    for(int p = 0; p < np; ++p) {
      const int j = p * nb, jb = (N - j) < nb ? (N - j) : nb, pi = p % pc;
      if(pi == 0) HCHK(prepare(p));
      FlowSwap sw;
      if(fused) {
        const int left = N - j - jb;
        sw.perm      = w.perm + pi * 2 * nb;
        sw.top       = w.work + (p & 1) * half;
        sw.next      = w.work + (1 - (p & 1)) * half;
        sw.next_rows = left < nb ? left : nb;
      } else {
        HCHK(launch_swap_inplace(s, jb, nrhs, B + j, ldb, w.perm + pi * 2 * nb));
      }
      HCHK(f.solve(false, false, j, j + jb, j + jb, N, pi * bpp, sw));
    }
    return f.upper(N);
  }
  // A = P0^T L0 P1^T L1 ... U  =>  A^T z = g  is solved as
  // w = U^{-T} g, then for panels from the last: z_p -= L21^T z_below,
  // z_p = L11^{-T} z_p, z = P_p^T z.
  HCHK(f.upper_trans(N));
  for(int p = np - 1; p >= 0; --p) {
    const int j = p * nb, jb = (N - j) < nb ? (N - j) : nb, e = j + jb, pi = p % pc;
    if(p == np - 1 || pi == pc - 1) HCHK(prepare(p - pi));
    // z_p -= L21^T z_below reduces over all N - e rows below the panel for a
    // jb x nrhs result: split over K, the partials in the work buffer, while
    // they fit
    if(e < N)
      HCHK(launch_tn_sub(s, N - e, jb, nrhs, A + e + static_cast<size_t>(j) * lda,
                         lda, B + e, ldb, B + j, ldb, w.work, w.work_doubles));
    HCHK(f.solve(true, true, j, e, e, e, pi * bpp));
    HCHK(launch_swap_inverse(s, jb, nrhs, B + j, ldb, w.perm + pi * 2 * nb));
  }
  return hipSuccess;
}

hipError_t getrs_enqueue(hipStream_t s, const double* A, int N, int nb, int lda,
                         const int* ipiv, int trans, int nrhs, double* B,
                         int ldb, const FlowScratch& w) {
  // the right-hand sides whose blocks fit the exchange buffer, for a matrix of
  // up to 8 blocks
  const int rows = N < kMaxNB ? (N + kFB - 1) / kFB * kFB : kMaxNB;
  const int cols = rows > 0 ? static_cast<int>(kFlowX / rows) / 16 * 16 : kFlowCols;
  for(int c = 0; c < nrhs; c += cols)
    HCHK(getrs_slices(s, A, N, nb, lda, ipiv, trans, nrhs - c < cols ? nrhs - c : cols,
                      B + static_cast<size_t>(c) * ldb, ldb, w));
  return hipSuccess;
}
#undef HCHK

}  // namespace hplx
