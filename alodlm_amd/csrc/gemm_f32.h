// The float matrix-core GEMM (gemm_f32.hip) as the dispatch calls it.
#pragma once

#include "common.h"

bool gemm_f32_eligible(const void* A, int64_t lda, int a_kmajor, const void* B, int64_t ldb,
                       int b_kmajor, int64_t M, int64_t N, int64_t K);
int64_t gemm_f32_splits(int64_t M, int64_t N, int64_t K);
// Returns the number of K splits launched; more than one leaves their sums in
// `workspace` ([splits][M][N]) for the caller to reduce into C.
int64_t gemm_f32_launch(const float* A, int64_t lda, int a_kmajor, const float* B, int64_t ldb,
                        int b_kmajor, float* C, int64_t ldc, const float* R, int64_t ldr,
                        int64_t M, int64_t N, int64_t K, float alpha, int epi, float* workspace,
                        hipStream_t st);
