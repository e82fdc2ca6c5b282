// float32 products of many rows (gemm_split.hip), which gemm_simple.hip hands over.
#pragma once
#include <hip/hip_runtime.h>

#define SPLIT_BLOCKS_K 512         // up to this k few rows are gemm_blocks', whatever their number

// Rows of a workgroup of gemm_blocks, 0 where few rows are gemm_walk's or gemm_few_rows'. Over the segments of a longer k the waves have enough to do (us by few
// rows, by blocks): 2,048 x 768 at 16 rows 7.1 and 7.3, at 4 rows of k = 1,280 6.8 and 6.6, of 1,500 7.2 and 7.4. From 33 rows on tiles of 64 rows would take more than
// 64 KB of LDS, and tiles of 32 read W twice: 2,048 x 516 at 64 rows 10.7 and 6.7, x 768 11.0 and 9.0; 4,096 x 516 (512 workgroups) 11.1 and 8.9, x 768 11.0 and 13.2.
static inline int few_blocks_rows(int M, int N, int K, int batch) {
  const long long groups = (long long)((N + 15) / 16) * ((M + 31) / 32) * batch;
  if (M <= 8) return K <= 1280 ? 8 : 0;
  if (M <= 32) return K <= SPLIT_BLOCKS_K || (K <= 640 && groups <= 512) ? (M <= 16 ? 16 : 32) : 0;
  return K <= SPLIT_BLOCKS_K ? 64 : K <= 768 && groups <= (K <= 576 ? 512 : 384) ? 32 : 0;
}
// Waves of a workgroup of gemm_few_rows (more than 8 float32 rows): eight where the workgroups leave every CU one at the most and k is long, or would leave half of four
// waves without a segment in the last round: 2,048 x 1,028 at 32 / 64 rows 14.0 / 16.9 us by four and 10.3 / 11.9 by eight, x 1,500 14.8 / 20.4 and 14.8 / 16.5, but 3,072 x 2,048 at
// 9 / 16 rows, from memory, 10.2 / 11.6 and 10.6 / 12.0.
static inline int few_rows_waves(int M, int N, int K, int batch) {
  const int rest = (K + 255) / 256 % 4;
  return K > 1024 && (K >= 4096 || rest == 1 || rest == 2) && (long long)((N + 15) / 16) * ((M + 63) / 64) * batch <= 256 ? 8 : 4;
}

// Which of its forms takes a product (k above 32), 0: none, few rows are better taken elsewhere. vec: rows on 16 bytes and whole pieces of 4.
extern "C" int ta_gemm_split_form(int M, int N, int K, int lda, int ldw, int batch, bool vec);
void ta_gemm_split(hipStream_t stream, int form, const float* A, int lda, long long sa, const float* W, int ldw, long long sw,
                   const float* bias, float* C, int ldc, long long sc, int M, int N, int K, int batch, bool vec);
