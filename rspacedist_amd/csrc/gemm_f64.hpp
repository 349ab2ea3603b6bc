// gemm_f64.hpp — FP64 matrix-core products of libkukan_hip.so (gemm_f64.hip).  Each call says
// whether it took the product; where it did not (sizes, alignment), rocBLAS is the better one.
#pragma once
#include <hip/hip_runtime.h>

namespace kukan {

// C(M1 x M2) = alpha A^T B + beta C, A (K x M1), B (K x M2), column-major.  tri (M1 = M2 only):
// 1 / 2 computes the tiles that hold the triangle on and below / above the diagonal, other
// entries of C are left as they are.
bool gemm_f64_tn(int M1, int M2, long K, double alpha, const double *A, long lda, const double *B,
                 long ldb, double beta, double *C, long ldc, int tri, hipStream_t s);
// Y(R x M2) = alpha X(R x K) C(K x M2) + beta Y, C upper triangular (its entries below the
// diagonal are not read), Y not aliasing X
bool gemm_f64_nn_upper(long R, int K, int M2, double alpha, const double *X, long ldx, const double *C, long ldc,
                       double beta, double *Y, long ldy, hipStream_t s);
// X <- X C in place, C (M x M) upper triangular: column tiles from the last to the first, each
// reading only columns that no earlier launch has replaced
bool apply_upper_ok(long R, int M, const double *X, long ldx);
void gemm_f64_apply_upper(long R, int M, double *X, long ldx, const double *C, long ldc, hipStream_t s);

}  // namespace kukan
