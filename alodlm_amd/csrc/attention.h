// The attention forward as the layer calls launch it.
#pragma once

#include <stdint.h>

// alodlm_attention_fwd; with `chain` (bf16, head_dim 128) never on the kernel
// whose waves share a query's keys, so that a row's sums run in one order over
// its keys whatever the number of rows.
int attention_fwd(const void* q, const void* k, const void* v, int64_t ldv, const int64_t* bounds,
                  const int32_t* row_segment, const int32_t* tiles, int64_t n_tiles, void* o,
                  float* lse, int64_t rows, int64_t nq, int64_t nkv, int64_t dh,
                  int64_t block_size, int dtype, bool chain, void* stream);
