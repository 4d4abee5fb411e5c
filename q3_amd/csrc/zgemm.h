// Complex GEMM on MFMA (zgemm.hip, zgemm64.hip, zgemm32.hip).
#pragma once
#include <hip/hip_runtime.h>

#include <cstddef>

namespace q3x {

// Element types of A, B, the MFMA/accumulation type, and C.  D = complex128, F = complex64.
enum class GemmTypes { D_D_D_D, F_D_F_F, F_F_F_D, D_D_F_D };

// C (m x n) = alpha * op(A) * B + beta * C ; opa = 0: A is m x k ; opa = 1: A is k x m, op = A^H.
// Leading dimensions in complex elements.  work (may be null) enables split-K for skinny shapes.
hipError_t zgemm(GemmTypes types, int opa, int m, int n, int k, double alpha, const void* A, long lda,
                 const void* B, long ldb, double beta, void* C, long ldc, void* work, size_t work_bytes,
                 hipStream_t st);

// The FP64 products (zgemm64.hip) of 16-byte aligned matrices: m, n > 0.  tile: 10 r + c for a
// workgroup tile of 32 r rows by 16 c complex columns (44, 42, 25, 24, 23, 22, 21, 12) or 0 for the
// built-in choice; split: K chunks, <= 0 for the built-in choice.
bool zgemm64_has_tile(int tile);
bool zgemm64_aligned(const void* A, const void* B, const void* C, const void* work);
hipError_t zgemm64(int tile, int split, int opa, int m, int n, int k, double alpha, const void* A, long lda, const void* B,
                   long ldb, double beta, void* C, long ldc, void* work, size_t work_bytes, hipStream_t st);

// The FP32 products (zgemm32.hip): A^H B with F_D_F_F, A B with F_F_F_D, both with D_D_F_D, of matrices
// aligned to their elements (zgemm32_takes); tiles 45, 44, 42, 25, 24, 22, 21, 12.
bool zgemm32_has_tile(int tile);
bool zgemm32_takes(GemmTypes types, int opa, const void* A, const void* B, const void* C, const void* work);
hipError_t zgemm32(int tile, int split, GemmTypes types, int opa, int m, int n, int k, double alpha, const void* A,
                   long lda, const void* B, long ldb, double beta, void* C, long ldc, void* work, size_t work_bytes,
                   hipStream_t st);

}  // namespace q3x
