// The products that gemm_deep.hip takes over from the weight-streaming, the tiled and the library's product, inside their entry points.
#pragma once
#include <hip/hip_runtime.h>

// The tile of M rows against a bf16 weight [N, K] (gated: the packed pair), 0: not served
extern "C" int mv_gemm_deep_shape(int M, int N, int K, int gated);
extern "C" int mv_gemm_deep_fold_parts(int N);
extern "C" int mv_gemm_deep(const void* A, long lda, const void* W, const void* bias, void* C, long ldc, int c_dtype, int M, int N, int K,
                            int gated, const float* partial, int P, float eps, float limit, float slope, int square_relu, int shape,
                            hipStream_t stream);
extern "C" int mv_gemm_deep_fold(const void* A, long lda, const void* W, const void* bias, float* resid, long ldr, const void* norm_weight,
                                 int norm_weight_dtype, int unit_offset, void* weighted, long ldw, float* partial, int P, int M, int N, int K,
                                 int shape, hipStream_t stream);

// ... and the gated pairs that gemm_pair.hip takes over from the tiled product: the tile, 0: not served
extern "C" int mv_gemm_pair_shape(int M, int N, int K, int units);
extern "C" int mv_gemm_pair_reaches(long lda, int N, int K);
extern "C" int mv_gemm_pair(const void* A, long lda, const void* W, const void* bias, void* C, long ldc, int M, int N, int K, float limit, float slope,
                            int tile, hipStream_t stream);
