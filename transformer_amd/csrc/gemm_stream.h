// float32 products of up to 8 rows (gemm_stream.hip), which gemm_simple.hip hands over where they pay.
#pragma once
#include <hip/hip_runtime.h>

extern "C" int ta_gemm_stream_pays(int M, int N, int K, int glu);
extern "C" int ta_gemm_stream(hipStream_t stream, const float* A, int lda, const float* W, int ldw, const float* bias, float* C,
                              int ldc, int M, int N, int K, int glu, int add, const float* norm_w, float eps);
