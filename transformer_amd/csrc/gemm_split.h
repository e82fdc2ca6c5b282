// float32 products of many rows (gemm_split.hip), which gemm_simple.hip hands over.
#pragma once
#include <hip/hip_runtime.h>

// Which of its forms takes a product (k above 32), 0: none, few rows are better taken elsewhere. vec: rows on 16 bytes and whole pieces of 4.
extern "C" int ta_gemm_split_form(int M, int N, int K, int lda, int ldw, int batch, bool vec);
void ta_gemm_split(hipStream_t stream, int form, const float* A, int lda, long long sa, const float* W, int ldw, long long sw,
                   const float* bias, float* C, int ldc, long long sc, int M, int N, int K, int batch, bool vec);
