// bf16 GEMM for up to 64 rows and K <= 4096 in one launch (gemm_slim.hip).
#pragma once
#include <hip/hip_runtime.h>

// 16-column fragments per workgroup this kernel takes for the shape; 0: the split-K kernels are expected to be faster, or
// the shape does not fit (glu: the epilogue pairs [gate16 | up16] columns)
int gai_gemm_slim_nf(int M, int N, int K, bool glu);
// C = epilogue(A . W^T) (epi / out_f32 as gai_gemm_splitk; psw: W in MFMA fragment order)
void gai_gemm_slim(const void* A, const void* W, void* C, const void* bias, const void* R, int M, int N, int K, int ldc,
                   int epi, int out_f32, int nf, int psw, hipStream_t st);
// out = LayerNorm(A . W^T + bias + R) with K in gai_gemm_slim_ks slices (0: not for this shape); ws: slices x M x N floats
int gai_gemm_slim_ks(int M, int N, int K);
// slices, longer ones first, of a product whose K is deeper than that (0: not for this shape)
int gai_gemm_slim_few_ks(int M, int N, int K);
void gai_gemm_slim_partials(const void* A, const void* W, int M, int N, int K, int ks, float* ws, int psw, hipStream_t st);
void gai_gemm_slim_layernorm(const void* A, const void* W, const void* bias, const void* R, const void* g, const void* b,
                             void* out, int M, int N, int K, float eps, float* ws, int psw, hipStream_t st);
