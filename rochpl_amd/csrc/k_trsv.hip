// Products of the solves: the GEMVs of the mixed-precision solves (rocblas_dgemv
// at src/pgesv/HPL_pdtrsv_device.cpp:195-332), and the products with many
// right-hand sides of the FP64 solves and the adjoint.
#include <type_traits>
#include "gemm_tile.hpp"
#include "mxp.hpp"

namespace hplx {
namespace {

typedef double ud4 __attribute__((ext_vector_type(4)));

template <typename V, typename MT>
__device__ inline V to_v(MT x) {
  if constexpr(sizeof(MT) == 2)
    return static_cast<V>(__half2float(x));
  else
    return static_cast<V>(x);
}

// y[0:m] -= U[0:m, 0:kb] * xs[0:kb] in the vectors' type V (FP64, or FP32 in
// the mixed-precision correction solves), U of element type MT (double, or
// the FP32 / FP16 factors of the mixed forms).  Workgroup = 64 rows; wave w
// takes a quarter of the columns, 32 of their loads in flight at a time, since
// the kernel waits for memory (on average over a solve of N = 16384, kb = 512 in
// FP32 18.5 us with 4 in flight, 7.8 now; 32768, 1024 in FP16 34.2, 13.5), with
// the sums in the order of the columns; partial sums meet in LDS.
// xback (optional): workgroup 0 also copies xs[0:kb] there.
template <typename MT, typename V>
__global__ __launch_bounds__(256) void gemv_sub_kernel(
    int m, int kb, const MT* __restrict__ U, int ldu,
    const V* __restrict__ xs, V* __restrict__ y,
    V* __restrict__ xback) {
  __shared__ V sxs[kMaxNB];
  __shared__ V part[4][64];
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  for(int i = t; i < kb; i += blockDim.x) sxs[i] = xs[i];
  __syncthreads();
  if(xback && blockIdx.x == 0)
    for(int i = t; i < kb; i += blockDim.x) xback[i] = sxs[i];
  const int row = blockIdx.x * 64 + lane;
  const int ck  = (kb + 3) / 4;
  const int c0  = wave * ck;
  const int c1  = min(kb, c0 + ck);
  V         acc = 0;
  if(row < m) {
    const MT* u = U + row + static_cast<size_t>(c0) * ldu;
    int       c = c0;
    auto      run = [&](auto width) {
      constexpr int W = decltype(width)::value;
      for(; c + W <= c1; c += W) {
        MT v[W];
#pragma unroll
        for(int j = 0; j < W; ++j) v[j] = u[static_cast<size_t>(j) * ldu];
#pragma unroll
        for(int j = 0; j < W; ++j) acc = fma(to_v<V>(v[j]), sxs[c + j], acc);
        u += W * static_cast<size_t>(ldu);
      }
    };
    run(std::integral_constant<int, 32>());
    run(std::integral_constant<int, 4>());
    for(; c < c1; ++c) {
      acc = fma(to_v<V>(u[0]), sxs[c], acc);
      u += ldu;
    }
  }
  part[wave][lane] = acc;
  __syncthreads();
  if(wave == 0 && row < m)
    y[row] -= (part[0][lane] + part[1][lane]) + (part[2][lane] + part[3][lane]);
}

// y[0:k] = Inv * x[0:k] for a k x k matrix of type V (FP64 or FP32;
// column-major, leading dimension k), k <= kMaxNB.  Workgroup = 64 rows with
// 16 waves, each wave a sixteenth of the columns in chunks of 32 whose loads
// are all in flight at once (the matrix is small: the kernel is latency
// bound).
template <typename V>
__global__ __launch_bounds__(1024) void inv_gemv_kernel(
    int k, const V* __restrict__ Inv, const V* __restrict__ x,
    V* __restrict__ y) {
  __shared__ V sx[kMaxNB];
  __shared__ V part[16][64];
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  for(int i = t; i < k; i += blockDim.x) sx[i] = x[i];
  __syncthreads();
  const int row = blockIdx.x * 64 + lane;
  const int ck  = (k + 15) / 16;
  const int c0  = wave * ck;
  const int c1  = min(k, c0 + ck);
  V         acc = 0;
  if(row < k) {
    for(int cc = c0; cc < c1; cc += 32) {
      const V* p = Inv + row + static_cast<size_t>(cc) * k;
      V             v[32];
#pragma unroll
      for(int j = 0; j < 32; ++j)
        v[j] = cc + j < c1 ? p[static_cast<size_t>(j) * k] : V(0);
#pragma unroll
      for(int j = 0; j < 32; ++j)
        if(cc + j < c1) acc = fma(v[j], sx[cc + j], acc);
    }
  }
  part[wave][lane] = acc;
  __syncthreads();
  if(wave == 0 && row < k) {
    V sum = 0;
#pragma unroll
    for(int w = 0; w < 16; ++w) sum += part[w][lane];
    y[row] = sum;
  }
}

// C (m x n) -= A^T B for the transposed solves, A (K x m) and B (K x n)
// column-major: one 64 x 64 tile of the result per workgroup over k in [s * kc,
// min(K, (s + 1) * kc)).  DIRECT (one split): C is updated in place; otherwise
// split s writes its partial tile to P + s * m * n (column-major, leading
// dimension m) for tn_reduce_kernel.  Two forms with the same order of
// operations: tn_tile_kernel for aligned operands (gemm_tile.hpp), tn_kernel for
// any (N = 16384, NB = 512: 64 right-hand sides alike, 22 us a panel; 256 6.22
// against 6.43 ms for the whole solve).
template <bool DIRECT>
__global__ __launch_bounds__(256) void tn_tile_kernel(
    int K, int m, int n, int kc, const double* __restrict__ A, int lda,
    const double* __restrict__ B, int ldb, double* __restrict__ out, int ldo,
    int tiles_m, int tiles_n) {
  __shared__ gemm::TileShared<double, 64, 64> sh;
  const int tiles = tiles_m * tiles_n, split = blockIdx.x / tiles;
  const int k0 = split * kc;
  gemm::gemm_tile<double, !DIRECT, DIRECT, false, 64, 64, true, false>(
      threadIdx.x, blockIdx.x - split * tiles, true, m, n, min(kc, K - k0), A + k0, lda,
      B + k0, ldb, DIRECT ? out : out + static_cast<size_t>(split) * m * n,
      DIRECT ? ldo : m, tiles_m, tiles_n, sh);
}

template <bool DIRECT>
__global__ __launch_bounds__(256) void tn_kernel(
    int K, int m, int n, int kc, const double* __restrict__ A, int lda,
    const double* __restrict__ B, int ldb, double* __restrict__ out, int ldo,
    int tiles_m, int tiles_n) {
  __shared__ double sa[32][65];
  __shared__ double sb[32][65];
  const int tiles = tiles_m * tiles_n, split = blockIdx.x / tiles;
  const int tile = blockIdx.x - split * tiles;
  const int m0 = (tile % tiles_m) * 64, n0 = (tile / tiles_m) * 64;
  const int k0 = split * kc, k1 = min(K, k0 + kc);
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int wm0 = (wave & 1) * 32, wn0 = (wave >> 1) * 32;
  const int l16 = lane & 15, lk = lane >> 4;
  double ra[8], rb[8];
  // element r of a thread's share: k row e % 32, column e / 32 of the 32 x 64
  // step
  auto load = [&](int k) {
#pragma unroll
    for(int r = 0; r < 8; ++r) {
      const int e = t + 256 * r;
      const int kk = k + (e & 31), c = e >> 5;
      ra[r] = kk < k1 && m0 + c < m ? A[kk + static_cast<size_t>(m0 + c) * lda] : 0.0;
      rb[r] = kk < k1 && n0 + c < n ? B[kk + static_cast<size_t>(n0 + c) * ldb] : 0.0;
    }
  };
  ud4 acc[2][2];
#pragma unroll
  for(int i = 0; i < 2; ++i)
#pragma unroll
    for(int j = 0; j < 2; ++j) acc[i][j] = ud4{0.0, 0.0, 0.0, 0.0};
  if(k0 < k1) load(k0);
  for(int k = k0; k < k1; k += 32) {
#pragma unroll
    for(int r = 0; r < 8; ++r) {
      const int e = t + 256 * r;
      sa[e & 31][e >> 5] = ra[r];
      sb[e & 31][e >> 5] = rb[r];
    }
    __syncthreads();
    if(k + 32 < k1) load(k + 32);
#pragma unroll
    for(int ks = 0; ks < 8; ++ks) {
      double fa[2], fb[2];
#pragma unroll
      for(int i = 0; i < 2; ++i) fa[i] = sa[ks * 4 + lk][wm0 + i * 16 + l16];
#pragma unroll
      for(int j = 0; j < 2; ++j) fb[j] = sb[ks * 4 + lk][wn0 + j * 16 + l16];
#pragma unroll
      for(int i = 0; i < 2; ++i)
#pragma unroll
        for(int j = 0; j < 2; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(fb[j], fa[i],
                                                           acc[i][j], 0, 0, 0);
    }
    __syncthreads();
  }
  // acc[i][j][r]: row wm0 + 16 i + l16, column wn0 + 16 j + 4 r + lk
  double* po = DIRECT ? out : out + static_cast<size_t>(split) * m * n;
#pragma unroll
  for(int i = 0; i < 2; ++i) {
    const int row = m0 + wm0 + i * 16 + l16;
    if(row >= m) continue;
#pragma unroll
    for(int j = 0; j < 2; ++j)
#pragma unroll
      for(int r = 0; r < 4; ++r) {
        const int col = n0 + wn0 + j * 16 + 4 * r + lk;
        if(col >= n) continue;
        if(DIRECT)
          po[row + static_cast<size_t>(col) * ldo] -= acc[i][j][r];
        else
          po[row + static_cast<size_t>(col) * m] = acc[i][j][r];
      }
  }
}

// C[i, j] -= sum over the splits of P, in split order (the result does not
// depend on how the splits were scheduled).
__global__ __launch_bounds__(256) void tn_reduce_kernel(
    int m, int n, int splits, const double* __restrict__ P,
    double* __restrict__ C, int ldc) {
  const long e = static_cast<long>(blockIdx.x) * 256 + threadIdx.x;
  if(e >= static_cast<long>(m) * n) return;
  const int i = static_cast<int>(e % m), j = static_cast<int>(e / m);
  double sum = 0.0;
  for(int sp = 0; sp < splits; ++sp) sum += P[static_cast<size_t>(sp) * m * n + e];
  C[i + static_cast<size_t>(j) * ldc] -= sum;
}

template <typename MT, typename V>
hipError_t gemv_sub_t(hipStream_t s, int m, int k, const MT* M, int ldm,
                      const V* x, V* y, V* xback) {
  if(m <= 0 || k <= 0) return hipSuccess;
  if(k > kMaxNB) return hipErrorInvalidValue;
  hipLaunchKernelGGL((gemv_sub_kernel<MT, V>), dim3((m + 63) / 64), dim3(256), 0,
                     s, m, k, M, ldm, x, y, xback);
  return hipGetLastError();
}

}  // namespace

hipError_t launch_gemv_sub(hipStream_t s, int m, int k, const float* M,
                           int ldm, const double* x, double* y,
                           double* xback) {
  return gemv_sub_t(s, m, k, M, ldm, x, y, xback);
}

hipError_t launch_gemv_sub(hipStream_t s, int m, int k, const float* M,
                           int ldm, const float* x, float* y, float* xback) {
  return gemv_sub_t(s, m, k, M, ldm, x, y, xback);
}

hipError_t launch_gemv_sub(hipStream_t s, int m, int k, const __half* M,
                           int ldm, const float* x, float* y, float* xback) {
  return gemv_sub_t(s, m, k, M, ldm, x, y, xback);
}

hipError_t launch_gemv_sub(hipStream_t s, int m, int k, const __half* M,
                           int ldm, const double* x, double* y,
                           double* xback) {
  return gemv_sub_t(s, m, k, M, ldm, x, y, xback);
}

template <typename V>
hipError_t inv_gemv_t(hipStream_t s, int k, const V* Inv, const V* x, V* y) {
  if(k <= 0) return hipSuccess;
  if(k > kMaxNB) return hipErrorInvalidValue;
  hipLaunchKernelGGL(inv_gemv_kernel<V>, dim3((k + 63) / 64), dim3(1024), 0, s,
                     k, Inv, x, y);
  return hipGetLastError();
}

hipError_t launch_inv_gemv(hipStream_t s, int k, const double* Inv,
                           const double* x, double* y) {
  return inv_gemv_t(s, k, Inv, x, y);
}

hipError_t launch_inv_gemv(hipStream_t s, int k, const float* Inv,
                           const float* x, float* y) {
  return inv_gemv_t(s, k, Inv, x, y);
}

hipError_t launch_tn_sub(hipStream_t s, int K, int m, int n, const double* A,
                         int lda, const double* B, int ldb, double* C, int ldc,
                         double* work, size_t work_doubles) {
  if(K <= 0 || m <= 0 || n <= 0) return hipSuccess;
  const size_t mn = static_cast<size_t>(m) * n;
  const int tiles_m = (m + 63) / 64, tiles_n = (n + 63) / 64;
  const long tiles = static_cast<long>(tiles_m) * tiles_n;
  // split K when the tiles alone leave the GPU short of work: about 256 k
  // per split, at most 64 splits and what the work buffer holds
  long splits = tiles >= 256 ? 1 : (K + 255) / 256;
  splits = splits < 64 ? splits : 64;
  const long cap = work ? static_cast<long>(work_doubles / mn) : 0;
  splits = splits < cap ? splits : (cap < 1 ? 1 : cap);
  const int kc = static_cast<int>(((K + splits - 1) / splits + 31) / 32 * 32);
  splits = (K + kc - 1) / kc;
  if(tiles * splits > 0x7fffffffL) return hipErrorInvalidValue;
  const dim3 grid(static_cast<unsigned>(tiles * splits));
  const auto al16 = [](const double* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; };
  const bool pairs = al16(A) && lda % 2 == 0 && al16(B) && ldb % 2 == 0;
  if(splits == 1) {
    if(pairs)
      hipLaunchKernelGGL(tn_tile_kernel<true>, grid, dim3(256), 0, s, K, m, n, kc, A, lda, B,
                         ldb, C, ldc, tiles_m, tiles_n);
    else
      hipLaunchKernelGGL(tn_kernel<true>, grid, dim3(256), 0, s, K, m, n, kc, A, lda, B, ldb,
                         C, ldc, tiles_m, tiles_n);
    return hipGetLastError();
  }
  if(pairs)
    hipLaunchKernelGGL(tn_tile_kernel<false>, grid, dim3(256), 0, s, K, m, n, kc, A, lda, B,
                       ldb, work, m, tiles_m, tiles_n);
  else
    hipLaunchKernelGGL(tn_kernel<false>, grid, dim3(256), 0, s, K, m, n, kc, A, lda, B, ldb,
                       work, m, tiles_m, tiles_n);
  hipLaunchKernelGGL(tn_reduce_kernel,
                     dim3(static_cast<unsigned>((mn + 255) / 256)), dim3(256),
                     0, s, m, n, static_cast<int>(splits), work, C, ldc);
  return hipGetLastError();
}

hipError_t launch_nn_sub(hipStream_t s, int K, int m, int n, const double* A,
                         int lda, const double* B, int ldb, double* C,
                         int ldc) {
  if(K <= 0) return hipSuccess;
  return launch_dgemm(s, m, n, K, -1.0, A, lda, B, ldb, 1.0, C, ldc, false);
}

hipError_t launch_outer_neg(hipStream_t s, int K, int m, int n,
                            const double* A, int lda, const double* B, int ldb,
                            double* C, int ldc) {
  if(m <= 0 || n <= 0) return hipSuccess;
  if(K <= 0) return hipErrorInvalidValue;
  return launch_dgemm(s, m, n, K, -1.0, A, lda, B, ldb, 0.0, C, ldc, false, 0, false, true);
}

}  // namespace hplx
