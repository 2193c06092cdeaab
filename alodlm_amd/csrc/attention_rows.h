// Attention of one row by one wavefront, which spreads head_dim over its lanes
// and walks the rows that the mask allows, one at a time: any dtype, any
// head_dim up to 256.  The reference kernels of attention.hip, and what the
// float matrix-core kernels fall back to.
#pragma once

#include "attention_common.h"

#define ATT_MAX_PER_LANE 4  // head_dim <= 256

// Output and log-sum-exp of query row r, head h.
template <typename T>
__device__ void attn_fwd_row(const T* __restrict__ q, const T* __restrict__ k,
                             const T* __restrict__ v, int64_t ldv,
                             const int64_t* __restrict__ bounds,
                             const int32_t* __restrict__ row_segment, T* __restrict__ o,
                             float* __restrict__ lse, int64_t rows, int64_t nq, int64_t nkv,
                             int64_t dh, int64_t B, float scale, int64_t r, int64_t h) {
  const int lane = threadIdx.x & 63;
  const int64_t hk = h / (nq / nkv);
  const int per = (int)((dh + 63) / 64);
  float qv[ATT_MAX_PER_LANE], acc[ATT_MAX_PER_LANE];
  for (int t = 0; t < per; ++t) {
    const int64_t e = lane + 64 * t;
    qv[t] = e < dh ? Elem<T>::load(q, (r * nq + h) * dh + e) : 0.f;
    acc[t] = 0.f;
  }
  const SegRow sr = seg_row(bounds, row_segment, r);
  int64_t ra[2][2];
  query_key_ranges(sr, B, ra[0][0], ra[0][1], ra[1][0], ra[1][1]);
  float m = -INFINITY, l = 0.f;
  for (int rg = 0; rg < 2; ++rg) {
    for (int64_t kr = ra[rg][0]; kr < ra[rg][1]; ++kr) {
      float s = 0.f;
      for (int t = 0; t < per; ++t) {
        const int64_t e = lane + 64 * t;
        if (e < dh) s += qv[t] * Elem<T>::load(k, (kr * nkv + hk) * dh + e);
      }
      s = wave_sum(s) * scale;
      const float mn = fmaxf(m, s);
      const float corr = expf(m - mn), p = expf(s - mn);
      l = l * corr + p;
      for (int t = 0; t < per; ++t) {
        const int64_t e = lane + 64 * t;
        const float vv = e < dh ? Elem<T>::load(v, kr * ldv + hk * dh + e) : 0.f;
        acc[t] = acc[t] * corr + p * vv;
      }
      m = mn;
    }
  }
  const float inv = 1.0f / l;
  for (int t = 0; t < per; ++t) {
    const int64_t e = lane + 64 * t;
    if (e < dh) Elem<T>::store(o, (r * nq + h) * dh + e, acc[t] * inv);
  }
  if (lane == 0) lse[h * rows + r] = m + logf(l);
}

// dQ of query row r, head h.
template <typename T>
__device__ void attn_dq_row(const T* __restrict__ q, const T* __restrict__ k,
                            const T* __restrict__ v, int64_t ldv,
                            const float* __restrict__ lse, const float* __restrict__ delta,
                            const T* __restrict__ dout, const int64_t* __restrict__ bounds,
                            const int32_t* __restrict__ row_segment, T* __restrict__ dq,
                            int64_t rows, int64_t nq, int64_t nkv, int64_t dh, int64_t B,
                            float scale, int64_t r, int64_t h) {
  const int lane = threadIdx.x & 63;
  const int64_t hk = h / (nq / nkv);
  const int per = (int)((dh + 63) / 64);
  float qv[ATT_MAX_PER_LANE], dov[ATT_MAX_PER_LANE], acc[ATT_MAX_PER_LANE];
  for (int t = 0; t < per; ++t) {
    const int64_t e = lane + 64 * t;
    qv[t] = e < dh ? Elem<T>::load(q, (r * nq + h) * dh + e) : 0.f;
    dov[t] = e < dh ? Elem<T>::load(dout, (r * nq + h) * dh + e) : 0.f;
    acc[t] = 0.f;
  }
  const float L_ = lse[h * rows + r], D = delta[h * rows + r];
  const SegRow sr = seg_row(bounds, row_segment, r);
  int64_t ra[2][2];
  query_key_ranges(sr, B, ra[0][0], ra[0][1], ra[1][0], ra[1][1]);
  for (int rg = 0; rg < 2; ++rg) {
    for (int64_t kr = ra[rg][0]; kr < ra[rg][1]; ++kr) {
      float s = 0.f, dp = 0.f;
      for (int t = 0; t < per; ++t) {
        const int64_t e = lane + 64 * t;
        if (e < dh) {
          s += qv[t] * Elem<T>::load(k, (kr * nkv + hk) * dh + e);
          dp += dov[t] * Elem<T>::load(v, kr * ldv + hk * dh + e);
        }
      }
      s = wave_sum(s) * scale;
      dp = wave_sum(dp);
      const float p = expf(s - L_);
      const float ds = p * (dp - D) * scale;
      for (int t = 0; t < per; ++t) {
        const int64_t e = lane + 64 * t;
        if (e < dh) acc[t] += ds * Elem<T>::load(k, (kr * nkv + hk) * dh + e);
      }
    }
  }
  for (int t = 0; t < per; ++t) {
    const int64_t e = lane + 64 * t;
    if (e < dh) Elem<T>::store(dq, (r * nq + h) * dh + e, acc[t]);
  }
}

// dK and dV of key row r, key/value head hk.
template <typename T>
__device__ void attn_dkdv_row(const T* __restrict__ q, const T* __restrict__ k,
                              const T* __restrict__ v, int64_t ldv,
                              const float* __restrict__ lse, const float* __restrict__ delta,
                              const T* __restrict__ dout, const int64_t* __restrict__ bounds,
                              const int32_t* __restrict__ row_segment, T* __restrict__ dk,
                              T* __restrict__ dv, int64_t lddv, int64_t rows, int64_t nq,
                              int64_t nkv, int64_t dh, int64_t B, float scale, int64_t r,
                              int64_t hk) {
  const int lane = threadIdx.x & 63;
  const int64_t group = nq / nkv;
  const int per = (int)((dh + 63) / 64);
  float kv[ATT_MAX_PER_LANE], vv[ATT_MAX_PER_LANE], dka[ATT_MAX_PER_LANE], dva[ATT_MAX_PER_LANE];
  for (int t = 0; t < per; ++t) {
    const int64_t e = lane + 64 * t;
    kv[t] = e < dh ? Elem<T>::load(k, (r * nkv + hk) * dh + e) : 0.f;
    vv[t] = e < dh ? Elem<T>::load(v, r * ldv + hk * dh + e) : 0.f;
    dka[t] = dva[t] = 0.f;
  }
  const SegRow sr = seg_row(bounds, row_segment, r);
  int64_t ra[2][2];
  key_query_ranges(sr, B, ra[0][0], ra[0][1], ra[1][0], ra[1][1]);
  for (int64_t h = hk * group; h < (hk + 1) * group; ++h) {
    for (int rg = 0; rg < 2; ++rg) {
      for (int64_t qr = ra[rg][0]; qr < ra[rg][1]; ++qr) {
        float s = 0.f, dp = 0.f;
        for (int t = 0; t < per; ++t) {
          const int64_t e = lane + 64 * t;
          if (e < dh) {
            s += kv[t] * Elem<T>::load(q, (qr * nq + h) * dh + e);
            dp += vv[t] * Elem<T>::load(dout, (qr * nq + h) * dh + e);
          }
        }
        s = wave_sum(s) * scale;
        dp = wave_sum(dp);
        const float p = expf(s - lse[h * rows + qr]);
        const float ds = p * (dp - delta[h * rows + qr]) * scale;
        for (int t = 0; t < per; ++t) {
          const int64_t e = lane + 64 * t;
          if (e < dh) {
            dva[t] += p * Elem<T>::load(dout, (qr * nq + h) * dh + e);
            dka[t] += ds * Elem<T>::load(q, (qr * nq + h) * dh + e);
          }
        }
      }
    }
  }
  for (int t = 0; t < per; ++t) {
    const int64_t e = lane + 64 * t;
    if (e < dh) {
      Elem<T>::store(dk, (r * nkv + hk) * dh + e, dka[t]);
      Elem<T>::store(dv, r * lddv + hk * dh + e, dva[t]);
    }
  }
}
