// Blocked Cholesky: diagonal blocks of 128 in one workgroup's registers, panels
// and trailing updates by rocBLAS.
//
// It takes the place of rocsolver_dpotrf, whose result is not repeatable while
// other queues' work shares the device: beside products and copies on six
// other streams, about one factor in a thousand of orders 70 to 128 differed
// from the same call's result alone, by up to 5e10, and the 70 to 80 occupied
// orbitals of (H2O)14 to (H2O)16 took another factor in 3% of the iterations
// of a batch.  Orders up to 64 were never seen to differ.  This one gives the
// bits that the library's gives alone up to order 127, and takes 46 us at
// order 80 and 343 at 320 where that takes 89 and 709.
#include "cholesky.hpp"

namespace vqc {
namespace {

// A block's rows and columns are dealt cyclically: thread (tr, tc) of a
// kRows x kCols grid holds elements (tr + kRows x, tc + kCols y) of the upper
// triangle.  Step k: the half wave that holds row k divides it by the root of
// its diagonal and hands it round through LDS; every thread then subtracts its
// part of the outer product.  Rows alternate between two LDS buffers, so a
// step has one barrier.  The order of operations is that of the unblocked
// right-looking algorithm, each update one fused multiply-add.  Bound by the
// chain of steps (root, quotient, LDS, barrier): 0.5 us each.
constexpr int kRows = 16, kCols = 32, kThreads = kRows * kCols;
constexpr int kEdge = 128, kX = kEdge / kRows, kY = kEdge / kCols;

template <bool LOWER>
__global__ __launch_bounds__(kThreads) void cholesky_block_kernel(double* __restrict__ A, int n, int lda, int offset,
                                                                  rocblas_int* __restrict__ info) {
  __shared__ double row[2][kEdge];
  __shared__ int bad[2];
  // A block before this one failed: nothing of this one is written.
  if (offset > 0 && info[0] != 0) return;
  const int tid = threadIdx.x, tr = tid / kCols, tc = tid % kCols;
  const auto at = [&](int r, int c) {
    return LOWER ? c + static_cast<std::size_t>(r) * lda : r + static_cast<std::size_t>(c) * lda;
  };
  double a[kX][kY];
#pragma unroll
  for (int x = 0; x < kX; ++x)
#pragma unroll
    for (int y = 0; y < kY; ++y) {
      const int r = tr + kRows * x, c = tc + kCols * y;
      a[x][y] = r <= c && c < n ? A[at(r, c)] : 0.0;
    }
  int failed = 0;
#pragma unroll
  for (int x = 0; x < kX; ++x) {  // rows 16 x .. 16 x + 15: register indices stay constants
    for (int q = 0; q < kRows; ++q) {
      const int k = x * kRows + q;
      if (k >= n || failed) break;
      if (tr == q) {
        // The diagonal element sits in this half wave.
        const int yd = x * kRows / kCols;
        const double d = __shfl(a[x][yd], (tid & 32) + k % kCols);
        const double u = sqrt(d);
#pragma unroll
        for (int y = 0; y < kY; ++y) {
          const int c = tc + kCols * y;
          if (c == k) a[x][y] = u;
          else if (c > k) a[x][y] /= u;
          row[k & 1][c] = c > k ? a[x][y] : 0.0;
        }
        if (tc == 0) bad[k & 1] = !(d > 0.0);
      }
      __syncthreads();
      if (bad[k & 1]) {
        failed = k + 1;
        break;
      }
      double uc[kY];
#pragma unroll
      for (int y = 0; y < kY; ++y) uc[y] = row[k & 1][tc + kCols * y];
#pragma unroll
      for (int z = x; z < kX; ++z) {
        const double ur = row[k & 1][tr + kRows * z];  // zero up to row k
#pragma unroll
        for (int y = 0; y < kY; ++y)
          if (kCols * y + kCols > kRows * z) a[z][y] = fma(-ur, uc[y], a[z][y]);
      }
    }
  }
#pragma unroll
  for (int x = 0; x < kX; ++x)
#pragma unroll
    for (int y = 0; y < kY; ++y) {
      const int r = tr + kRows * x, c = tc + kCols * y;
      if (r <= c && c < n) A[at(r, c)] = a[x][y];
    }
  if (tid == 0) {
    if (failed) info[0] = offset + failed;
    else if (offset == 0) info[0] = 0;
  }
}

}  // namespace

void cholesky_factor(rocblas_handle blas, rocblas_fill fill, int n, double* A, int lda, rocblas_int* info, hipStream_t s) {
  if (n < 1 || lda < n) throw std::invalid_argument("Cholesky shape");
  if (fill != rocblas_fill_upper && fill != rocblas_fill_lower) throw std::invalid_argument("Cholesky triangle");
  const bool lower = fill == rocblas_fill_lower;
  const double one = 1.0, minus = -1.0;
  for (int k = 0; k < n; k += kEdge) {
    const int nb = std::min(kEdge, n - k), rest = n - k - nb;
    double* diag = A + k + static_cast<std::size_t>(k) * lda;
    hipLaunchKernelGGL(lower ? cholesky_block_kernel<true> : cholesky_block_kernel<false>, dim3(1), dim3(kThreads), 0, s, diag,
                       nb, lda, k, info);
    VQC_LAUNCH("cholesky_block_kernel");
    if (!rest) break;
    double* trail = diag + nb + static_cast<std::size_t>(nb) * lda;
    if (lower) {
      double* panel = diag + nb;
      VQC_BLAS(rocblas_dtrsm(blas, rocblas_side_right, fill, rocblas_operation_transpose, rocblas_diagonal_non_unit, rest, nb,
                             &one, diag, lda, panel, lda));
      VQC_BLAS(rocblas_dsyrk(blas, fill, rocblas_operation_none, rest, nb, &minus, panel, lda, &one, trail, lda));
    } else {
      double* panel = diag + static_cast<std::size_t>(nb) * lda;
      VQC_BLAS(rocblas_dtrsm(blas, rocblas_side_left, fill, rocblas_operation_transpose, rocblas_diagonal_non_unit, nb, rest,
                             &one, diag, lda, panel, lda));
      VQC_BLAS(rocblas_dsyrk(blas, fill, rocblas_operation_transpose, rest, nb, &minus, panel, lda, &one, trail, lda));
    }
  }
}

}  // namespace vqc
