// The 128x128-tile bf16 GEMM (gemm_mid.hip) as the dispatch calls it.
#pragma once

#include "common.h"

bool gemm_mid_eligible(const void* A, int64_t lda, int a_kmajor, const void* B, int64_t ldb,
                       int b_kmajor, int64_t M, int64_t N, int64_t K);
// Tile rows of a product (tiles have 128 columns).
int gemm_mid_rows(int a_kmajor, int64_t M, int epi);
// Returns the number of K splits launched; more than one leaves their sums in
// `workspace` ([splits][M][N]) for the caller to reduce into C.
int64_t gemm_mid_launch(const bf16_t* A, int64_t lda, int a_kmajor, const bf16_t* B, int64_t ldb,
                        int b_kmajor, void* C, int64_t ldc, const bf16_t* R, int64_t ldr,
                        int64_t M, int64_t N, int64_t K, float alpha, int epi, int64_t splits,
                        float* workspace, hipStream_t st);
