// GQA attention under the dual-stream training mask (alodlm/batch.py:23-31).
//
// Segment s occupies dual-stream rows [base, base + 2L): the clean stream
// [base, base + L) is causal; a noisy row in block b (of size B) sees the
// clean keys of earlier blocks [base, base + b*B) and, causally, the noisy
// rows of its own block.  The kernels enumerate exactly those key ranges, so
// no masked pair and no cross-segment pair is ever visited.
//
// bf16 with head_dim 64 or 128 runs attention_mfma.hip / attention_fa128.hip
// (few queries: attention_few.hip),
// float with head_dim 128 attention_f32.hip.
// Reference kernels (any dtype, any head_dim): one wavefront per (query row,
// head) in the forward and dQ passes and one per (key row, kv head) in the
// dK/dV pass; the wavefront spreads head_dim over its lanes.
#include <initializer_list>

#include "attention.h"
#include "attention_rows.h"

template <typename T>
__global__ void __launch_bounds__(256)
attn_fwd_ref_kernel(const T* __restrict__ q, const T* __restrict__ k, const T* __restrict__ v,
                    int64_t ldv, const int64_t* __restrict__ bounds,
                    const int32_t* __restrict__ row_segment, T* __restrict__ o,
                    float* __restrict__ lse, int64_t rows, int64_t nq, int64_t nkv, int64_t dh,
                    int64_t B, float scale) {
  const int64_t item = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (item < rows * nq)
    attn_fwd_row<T>(q, k, v, ldv, bounds, row_segment, o, lse, rows, nq, nkv, dh, B, scale,
                    item / nq, item % nq);
}

// delta[h, r] = sum_e dO[r, h, e] * O[r, h, e]
template <typename T>
__global__ void __launch_bounds__(256)
attn_delta_kernel(const T* __restrict__ o, const T* __restrict__ dout, float* __restrict__ delta,
                  int64_t rows, int64_t nq, int64_t dh) {
  const int lane = threadIdx.x & 63;
  const int64_t item = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (item >= rows * nq) return;
  const int64_t r = item / nq, h = item % nq;
  float s = 0.f;
  for (int64_t e = lane; e < dh; e += 64)
    s += Elem<T>::load(o, (r * nq + h) * dh + e) * Elem<T>::load(dout, (r * nq + h) * dh + e);
  s = wave_sum(s);
  if (lane == 0) delta[h * rows + r] = s;
}

template <typename T>
__global__ void __launch_bounds__(256)
attn_dq_ref_kernel(const T* __restrict__ q, const T* __restrict__ k, const T* __restrict__ v,
                   int64_t ldv, const float* __restrict__ lse, const float* __restrict__ delta,
                   const T* __restrict__ dout, const int64_t* __restrict__ bounds,
                   const int32_t* __restrict__ row_segment, T* __restrict__ dq, int64_t rows,
                   int64_t nq, int64_t nkv, int64_t dh, int64_t B, float scale) {
  const int64_t item = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (item < rows * nq)
    attn_dq_row<T>(q, k, v, ldv, lse, delta, dout, bounds, row_segment, dq, rows, nq, nkv, dh, B,
                   scale, item / nq, item % nq);
}

template <typename T>
__global__ void __launch_bounds__(256)
attn_dkdv_ref_kernel(const T* __restrict__ q, const T* __restrict__ k, const T* __restrict__ v,
                     int64_t ldv, const float* __restrict__ lse, const float* __restrict__ delta,
                     const T* __restrict__ dout, const int64_t* __restrict__ bounds,
                     const int32_t* __restrict__ row_segment, T* __restrict__ dk,
                     T* __restrict__ dv, int64_t lddv, int64_t rows, int64_t nq, int64_t nkv,
                     int64_t dh, int64_t B, float scale) {
  const int64_t item = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (item < rows * nkv)
    attn_dkdv_row<T>(q, k, v, ldv, lse, delta, dout, bounds, row_segment, dk, dv, lddv, rows, nq,
                     nkv, dh, B, scale, item / nkv, item % nkv);
}

static int check_attn(int64_t rows, int64_t nq, int64_t nkv, int64_t dh, int64_t B) {
  ALODLM_CHECK_ARG(rows >= 0 && nq > 0 && nkv > 0 && nq % nkv == 0, "attention: bad head counts");
  ALODLM_CHECK_ARG(dh > 0 && dh <= 64 * ATT_MAX_PER_LANE, "attention: head_dim must be <= 256");
  ALODLM_CHECK_ARG(B >= 1, "attention: block_size must be positive");
  return ALODLM_OK;
}

int fa_fwd_launch(const bf16_t* q, const bf16_t* k, const bf16_t* v, int64_t ldv,
                  const int64_t* bounds, const int32_t* tiles, int64_t n_tiles, bf16_t* o,
                  float* lse, int64_t N, int nq, int nkv, int dh, int B, float scale,
                  hipStream_t st);
int fa_bwd_launch(const bf16_t* q, const bf16_t* k, const bf16_t* v, int64_t ldv,
                  const float* lse, const float* delta, const bf16_t* dout,
                  const int64_t* bounds, const int32_t* tiles, int64_t n_tiles, bf16_t* dq,
                  bf16_t* dk, bf16_t* dv, int64_t lddv, int64_t N, int nq, int nkv, int dh,
                  int B, float scale, hipStream_t st);

int fa128_fwd_launch(const bf16_t* q, const bf16_t* k, const bf16_t* v, int64_t ldv,
                     const int64_t* bounds, const int32_t* tiles, int64_t n_tiles, bf16_t* o,
                     float* lse, int64_t N, int nq, int nkv, int B, float scale, hipStream_t st);
int fa128_bwd_launch(const bf16_t* q, const bf16_t* k, const bf16_t* v, int64_t ldv,
                     const float* lse, const bf16_t* o, float* delta, const bf16_t* dout,
                     const int64_t* bounds, const int32_t* tiles, int64_t n_tiles, bf16_t* dq,
                     bf16_t* dk, bf16_t* dv, int64_t lddv, int64_t N, int nq, int nkv, int B,
                     float scale, const int64_t* ds_base, int64_t ds_blocks, hipStream_t st);

void fa128_few_launch(const bf16_t* q, const bf16_t* k, const bf16_t* v, int64_t ldv,
                      const int64_t* bounds, const int32_t* tiles, int64_t n_tiles, bf16_t* o,
                      float* lse, int64_t N, int nq, int nkv, int B, float scale, hipStream_t st);
bool attn_f32_eligible(int64_t rows, int64_t nq, int64_t nkv, int64_t dh, int64_t ldv);
void attn_f32_fwd_launch(const float* q, const float* k, const float* v, int64_t ldv,
                         const int64_t* bounds, const int32_t* row_segment, float* o, float* lse,
                         int64_t rows, int64_t nq, int64_t nkv, int64_t B, float scale,
                         hipStream_t st);
void attn_f32_bwd_launch(const float* q, const float* k, const float* v, int64_t ldv,
                         const float* lse, const float* delta, const float* dout,
                         const int64_t* bounds, const int32_t* row_segment, float* dq, float* dk,
                         float* dv, int64_t lddv, int64_t rows, int64_t nq, int64_t nkv, int64_t B,
                         float scale, hipStream_t st);

// The float matrix-core kernels take head_dim 128 and 16-byte aligned rows.
static bool use_f32(int dtype, int64_t rows, int64_t nq, int64_t nkv, int64_t dh, int64_t ldv,
                    std::initializer_list<const void*> ptrs) {
  if (dtype != ALODLM_F32 || !attn_f32_eligible(rows, nq, nkv, dh, ldv)) return false;
  for (const void* p : ptrs)
    if (reinterpret_cast<uintptr_t>(p) % 16) return false;
  return true;
}

// The MFMA kernels take bf16, head_dim 64 or 128, 16-byte aligned rows and a
// tile table; everything else runs the reference kernels above.
static bool use_mfma(int dtype, int64_t dh, const int32_t* tiles, int64_t ldv,
                     std::initializer_list<const void*> ptrs) {
  if (dtype != ALODLM_BF16 || tiles == nullptr || (dh != 64 && dh != 128) || ldv % 8) return false;
  for (const void* p : ptrs)
    if (reinterpret_cast<uintptr_t>(p) % 16) return false;
  return true;
}

// 128-row workgroups below which the forward takes 32-row ones whose waves
// share the keys (attention_few.hip).
constexpr int64_t FEW_WORKGROUPS = 256;

int attention_fwd(const void* q, const void* k, const void* v, int64_t ldv, const int64_t* bounds,
                  const int32_t* row_segment, const int32_t* tiles, int64_t n_tiles, void* o,
                  float* lse, int64_t rows, int64_t nq, int64_t nkv, int64_t dh,
                  int64_t block_size, int dtype, bool chain, void* stream) {
  int rc = check_attn(rows, nq, nkv, dh, block_size);
  if (rc) return rc;
  if (rows == 0) return ALODLM_OK;
  const float scale = 1.0f / sqrtf((float)dh);
  if (use_mfma(dtype, dh, tiles, ldv, {q, k, v, o})) {
    if (n_tiles == 0) return ALODLM_OK;
    ALODLM_CHECK_ARG(n_tiles <= 65535, "attention: too many 128-row tiles (%lld)", (long long)n_tiles);
    if (dh == 128 && !chain && n_tiles * nq < FEW_WORKGROUPS && 4 * n_tiles <= 65535) {
      fa128_few_launch((const bf16_t*)q, (const bf16_t*)k, (const bf16_t*)v, ldv, bounds, tiles,
                       n_tiles, (bf16_t*)o, lse, rows, (int)nq, (int)nkv, (int)block_size, scale,
                       as_stream(stream));
      ALODLM_CHECK_LAUNCH("attention_fwd_few");
      return ALODLM_OK;
    }
    if (dh == 128)
      return fa128_fwd_launch((const bf16_t*)q, (const bf16_t*)k, (const bf16_t*)v, ldv, bounds,
                              tiles, n_tiles, (bf16_t*)o, lse, rows, (int)nq, (int)nkv,
                              (int)block_size, scale, as_stream(stream));
    return fa_fwd_launch((const bf16_t*)q, (const bf16_t*)k, (const bf16_t*)v, ldv, bounds, tiles,
                         n_tiles, (bf16_t*)o, lse, rows, (int)nq, (int)nkv, (int)dh,
                         (int)block_size, scale, as_stream(stream));
  }
  if (use_f32(dtype, rows, nq, nkv, dh, ldv, {q, k, v, o})) {
    attn_f32_fwd_launch((const float*)q, (const float*)k, (const float*)v, ldv, bounds,
                        row_segment, (float*)o, lse, rows, nq, nkv, block_size, scale,
                        as_stream(stream));
    ALODLM_CHECK_LAUNCH("attention_fwd_f32");
    return ALODLM_OK;
  }
  ALODLM_DISPATCH(dtype, T, {
    attn_fwd_ref_kernel<T><<<ceil_div_u(rows * nq, 4), 256, 0, as_stream(stream)>>>(
        (const T*)q, (const T*)k, (const T*)v, ldv, bounds, row_segment, (T*)o, lse, rows, nq,
        nkv, dh, block_size, scale);
  });
  ALODLM_CHECK_LAUNCH("attention_fwd");
  return ALODLM_OK;
}

extern "C" int alodlm_attention_fwd(const void* q, const void* k, const void* v, int64_t ldv,
                                    const int64_t* bounds, const int32_t* row_segment,
                                    const int32_t* tiles, int64_t n_tiles, void* o, float* lse,
                                    int64_t rows, int64_t nq, int64_t nkv, int64_t dh,
                                    int64_t block_size, int dtype, void* stream) {
  return attention_fwd(q, k, v, ldv, bounds, row_segment, tiles, n_tiles, o, lse, rows, nq, nkv, dh,
                       block_size, dtype, false, stream);
}

extern "C" int alodlm_attention_fwd_chain(const void* q, const void* k, const void* v, int64_t ldv,
                                          const int64_t* bounds, const int32_t* row_segment,
                                          const int32_t* tiles, int64_t n_tiles, void* o,
                                          float* lse, int64_t rows, int64_t nq, int64_t nkv,
                                          int64_t dh, int64_t block_size, int dtype,
                                          void* stream) {
  return attention_fwd(q, k, v, ldv, bounds, row_segment, tiles, n_tiles, o, lse, rows, nq, nkv, dh,
                       block_size, dtype, true, stream);
}

int64_t fa128_bwd_workspace(int64_t N, int nq, int nkv, int64_t n_tiles, int64_t ds_blocks);

// 32x32 dS blocks per query head that the mask allows in a pack (the stored-dS
// backward's buffer): per segment of L tokens, T (T + 1) with T = ceil(L / 32);
// 0 unless block_size is 32.  base_out (S + 1 entries, may be NULL) receives
// each segment's first block and the total.  Host only.
extern "C" int64_t alodlm_attention_ds_blocks(const int64_t* token_offsets, int64_t segments,
                                              int64_t block_size, int64_t* base_out) {
  if (token_offsets == nullptr || segments < 0) return 0;
  int64_t total = 0;
  for (int64_t s = 0; s < segments; ++s) {
    if (base_out) base_out[s] = total;
    const int64_t L = token_offsets[s + 1] - token_offsets[s];
    const int64_t T = (L + 31) / 32;
    total += T * (T + 1);
  }
  if (base_out) base_out[segments] = total;
  return block_size == 32 ? total : 0;
}

extern "C" int64_t alodlm_attention_bwd_workspace(int64_t rows, int64_t nq, int64_t nkv,
                                                  int64_t dh, int64_t n_tiles, int64_t ds_blocks) {
  // delta [nq][rows]; the head_dim-128 kernels may also keep dK/dV partials
  // and the stored dS blocks
  if (dh == 128 && nq > 0 && nkv > 0)
    return fa128_bwd_workspace(rows, (int)nq, (int)nkv, n_tiles, ds_blocks);
  return rows * nq;
}

extern "C" int alodlm_attention_bwd(const void* q, const void* k, const void* v, int64_t ldv,
                                    const void* o, const float* lse, const void* dout,
                                    const int64_t* bounds, const int32_t* row_segment,
                                    const int32_t* tiles, int64_t n_tiles, void* dq, void* dk,
                                    void* dv, int64_t lddv, float* workspace,
                                    const int64_t* ds_base, int64_t ds_blocks, int64_t rows,
                                    int64_t nq, int64_t nkv, int64_t dh, int64_t block_size,
                                    int dtype, void* stream) {
  int rc = check_attn(rows, nq, nkv, dh, block_size);
  if (rc) return rc;
  if (rows == 0) return ALODLM_OK;
  const float scale = 1.0f / sqrtf((float)dh);
  hipStream_t st = as_stream(stream);
  float* delta = workspace;
  const bool mfma = use_mfma(dtype, dh, tiles, ldv, {q, k, v, o, dout, dq, dk, dv}) && lddv % 8 == 0;
  if (mfma && dh == 128) {
    // the head_dim-128 kernels compute delta themselves
    if (n_tiles == 0) return ALODLM_OK;
    ALODLM_CHECK_ARG(n_tiles <= 65535, "attention: too many 128-row tiles (%lld)", (long long)n_tiles);
    return fa128_bwd_launch((const bf16_t*)q, (const bf16_t*)k, (const bf16_t*)v, ldv, lse,
                            (const bf16_t*)o, delta, (const bf16_t*)dout, bounds, tiles, n_tiles,
                            (bf16_t*)dq, (bf16_t*)dk, (bf16_t*)dv, lddv, rows, (int)nq, (int)nkv,
                            (int)block_size, scale, ds_base, ds_blocks, st);
  }
  ALODLM_DISPATCH(dtype, T, {
    attn_delta_kernel<T><<<ceil_div_u(rows * nq, 4), 256, 0, st>>>((const T*)o, (const T*)dout,
                                                                   delta, rows, nq, dh);
  });
  ALODLM_CHECK_LAUNCH("attention_delta");
  if (mfma) {  // head_dim 64
    if (n_tiles == 0) return ALODLM_OK;
    ALODLM_CHECK_ARG(n_tiles <= 65535, "attention: too many 128-row tiles (%lld)", (long long)n_tiles);
    return fa_bwd_launch((const bf16_t*)q, (const bf16_t*)k, (const bf16_t*)v, ldv, lse, delta,
                         (const bf16_t*)dout, bounds, tiles, n_tiles, (bf16_t*)dq, (bf16_t*)dk,
                         (bf16_t*)dv, lddv, rows, (int)nq, (int)nkv, (int)dh, (int)block_size,
                         scale, st);
  }
  if (use_f32(dtype, rows, nq, nkv, dh, ldv, {q, k, v, dout, dq, dk, dv}) && lddv % 4 == 0) {
    attn_f32_bwd_launch((const float*)q, (const float*)k, (const float*)v, ldv, lse, delta,
                        (const float*)dout, bounds, row_segment, (float*)dq, (float*)dk,
                        (float*)dv, lddv, rows, nq, nkv, block_size, scale, st);
    ALODLM_CHECK_LAUNCH("attention_bwd_f32");
    return ALODLM_OK;
  }
  ALODLM_DISPATCH(dtype, T, {
    attn_dq_ref_kernel<T><<<ceil_div_u(rows * nq, 4), 256, 0, st>>>(
        (const T*)q, (const T*)k, (const T*)v, ldv, lse, delta, (const T*)dout, bounds,
        row_segment, (T*)dq, rows, nq, nkv, dh, block_size, scale);
    attn_dkdv_ref_kernel<T><<<ceil_div_u(rows * nkv, 4), 256, 0, st>>>(
        (const T*)q, (const T*)k, (const T*)v, ldv, lse, delta, (const T*)dout, bounds,
        row_segment, (T*)dk, (T*)dv, lddv, rows, nq, nkv, dh, block_size, scale);
  });
  ALODLM_CHECK_LAUNCH("attention_bwd");
  return ALODLM_OK;
}
