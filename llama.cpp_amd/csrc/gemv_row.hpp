// One activation row against a matrix of few rows (gemv_row.hip).
#pragma once
#include "common.hpp"

namespace mi355 {

// Up to 8192 rows, or 32768 of 4096 elements and more.  us, k_gemv_q / this, the matrices from memory: 512 x 14336 Q4_K 5.5 / 3.3, Q6_K 6.9 / 5.6, Q8_0 5.0 / 3.6; 4096 x 1024 3.7 / 3.0,
// 3.5 / 3.2, 3.1 / 2.7; 4096 x 4096 4.2 / 3.7, 5.6 / 4.7, 5.7 / 5.1; 4096 x 14336 10.8 / 8.6, 12.1 / 11.4, 13.5 / 12.3; 8192 x 4096 6.7 / 5.3, 8.1 / 7.2, 8.5 / 7.7; 28672 x 4096 13.4 / 12.4,
// 19.6 / 16.8, 23.0 / 21.1.  Beyond, many short rows: two or four of them per wave share the activation's copy, 16384 x 1024 5.5 / 5.8, 6.6 / 6.7, 5.7 / 6.2; 65536 x 2048 18.5 / 21.9, 22.1 /
// 23.7, 23.0 / 21.2; 128256 x 4096 49.2 / 50.0, 71.7 / 71.9, 93.3 / 89.3.
inline bool gemv_row_serves(int64_t N, int64_t K) { return K <= 32768 && (N <= 8192 || (N <= 32768 && K >= 4096)); }
int launch_gemv_row(hipStream_t s, int type, const void *W, const int8_t *aq, const act_ds *ads, float *dst, const float *residual, int64_t N, int64_t K);

}  // namespace mi355
