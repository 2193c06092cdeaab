// The few-row GEMM (gemm_skinny.hip) as the dispatch calls it.
#pragma once

#include "common.h"

constexpr int64_t SKINNY_M = ALODLM_FEW_ROWS;  // rows up to which it is taken

bool gemm_skinny_eligible(const void* A, int64_t lda, int a_kmajor, const void* B, int64_t ldb,
                          int b_kmajor, int64_t M, int64_t N, int64_t K, int epi, int dtype);
void gemm_skinny_launch(const void* A, int64_t lda, const void* B, int64_t ldb, void* C,
                        int64_t ldc, const void* R, int64_t ldr, int64_t M, int64_t N, int64_t K,
                        float alpha, int epi, int dtype, hipStream_t st);
