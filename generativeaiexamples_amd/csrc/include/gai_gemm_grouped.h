// bf16 products of rows sorted by expert, C[offs[e] .. offs[e+1]) = A[..] . B[e]^T, on the 256x256 kernel (gemm_impl.h).
#pragma once
#include <hip/hip_runtime.h>

// A [M, K], B [E, N, K], offs [E + 1] on the device; swiglu: B's rows interleaved [gate16 | up16], C [M, N / 2]. False (nothing
// launched) where the shape does not fit: N % 16 (32 with swiglu), K % 64, K >= 128, either operand below 2 GiB.
bool gai_gemm_grouped(const void* A, const void* B, void* C, const int* offs, int E, int M, int N, int K, int swiglu,
                      hipStream_t st);
