// Cholesky factorisation of a symmetric positive definite matrix (FP64).
#pragma once

#include "common.hpp"

namespace vqc {

// In place: A (n x n, column-major, leading dimension lda) -> its factor in
// the `fill` triangle, A = U^T U (upper) or L L^T (lower); the other triangle
// is neither read nor written.  info[0] (device) is 0, or k when the leading
// minor of order k is not positive; the factor is then incomplete.
void cholesky_factor(rocblas_handle blas, rocblas_fill fill, int n, double* A, int lda, rocblas_int* info, hipStream_t s);

}  // namespace vqc
