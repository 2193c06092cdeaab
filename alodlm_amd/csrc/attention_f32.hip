// float32 attention for head_dim 128 on the matrix cores (forward, dQ, dK/dV)
// under the dual-stream training mask or a decoding window's.
//
// Bound: v_mfma_f32_32x32x2_f32, 64 cycles per 32x32x2 block: 8192 cycles per
// 32 queries x 32 keys in the forward, 12288 in dQ, 16384 in dK/dV.  The
// operands of a block are two 16 KB tiles read in that time, so they come from
// L1/L2 straight into registers: no LDS staging, and no layout change between
// the products, because a float MFMA takes one k per lane half and the sums'
// layout can be fed back as an operand:
//  * lane = (col, half); scores are formed as S^T = K Q^T (dK/dV: S = Q K^T),
//    so a lane holds one query (key) and, in element 4 a + e, key (query)
//    8 a + 4 half + e of the tile;
//  * the next product contracts over exactly that index: step (a, e) takes
//    element 4 a + e as one operand and, for the other, 16 bytes of the row
//    8 a + 4 half + e at columns 4 col .. 4 col + 3 - one column for each of
//    four accumulators, which therefore hold columns 4 i + d (i the block row).
// A workgroup owns one 32-row tile of one head; its four waves take the tile's
// key (query) tiles in turn and add up in LDS in wave order, so that a short
// pack (the 700 rows of one 350-token segment: 352 tiles) still fills the chip.
// A tile of rows with an infinity or NaN among the rows it multiplies is done
// again row by row (attention_rows.h), so that no row depends on rows that the
// mask hides from it; the check is VALU work beside the matrix instructions.
// At that shape (16 / 8 heads): forward 603 us, dQ 635, dK/dV 1269 with one
// wave per row and no matrix instruction.
#include <limits.h>

#include "attention_rows.h"

namespace {

constexpr int HD = 128, NB = HD / 32, NK = HD / 8, AW = 4;

__device__ __forceinline__ f32x16_t mfma2(float a, float b, f32x16_t c) {
  return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ float4 load4f(const float* p) { return *reinterpret_cast<const float4*>(p); }

// Row `row`'s 4 columns at 8 b + 4 half of every 8-column block b.
__device__ __forceinline__ void row_frags(const float* p, int half, float4 (&f)[NK]) {
#pragma unroll
  for (int b = 0; b < NK; ++b) f[b] = load4f(p + 8 * b + 4 * half);
}

// acc += rows(p) . f^T over the head dimension: p is this lane's row.
__device__ __forceinline__ f32x16_t dot_rows(const float* p, int half, const float4 (&f)[NK]) {
  f32x16_t s = zero16();
#pragma unroll
  for (int b = 0; b < NK; ++b) {
    const float4 r = load4f(p + 8 * b + 4 * half);
    s = mfma2(r.x, f[b].x, s);
    s = mfma2(r.y, f[b].y, s);
    s = mfma2(r.z, f[b].z, s);
    s = mfma2(r.w, f[b].w, s);
  }
  return s;
}

// acc[d] += sum over the tile's rows t of p[row0 + t][4 col + d] * w[t]
// (rows past `last` re-read it: their weights are zero).  z becomes NaN where a
// row holds an infinity or NaN: the product gives it a part in the sums of
// lanes whose weight for it is zero because the mask hides it.
__device__ __forceinline__ void add_rows(f32x16_t (&acc)[NB], const float* p, int64_t ld, int row0,
                                         int last, int col, int half, const f32x16_t& w, float& z) {
#pragma unroll
  for (int t = 0; t < 16; ++t) {
    int r = row0 + 8 * (t >> 2) + 4 * half + (t & 3);
    r = r < last ? r : last;
    const float4 x = load4f(p + r * ld + 4 * col);
    acc[0] = mfma2(x.x, w[t], acc[0]);
    acc[1] = mfma2(x.y, w[t], acc[1]);
    acc[2] = mfma2(x.z, w[t], acc[2]);
    acc[3] = mfma2(x.w, w[t], acc[3]);
    z = fmaf(x.w, 0.f, fmaf(x.z, 0.f, fmaf(x.y, 0.f, fmaf(x.x, 0.f, z))));
  }
}

// Whether some wave of the workgroup met such a row.
__device__ __forceinline__ bool any_wave(int* flags, int wave, int lane, float z) {
  const bool mine = __any(z != 0.f);
  if (lane == 0) flags[wave] = mine;
  __syncthreads();
  bool some = false;
#pragma unroll
  for (int v = 0; v < AW; ++v) some |= flags[v] != 0;
  return some;
}

// This lane's intervals and their union over the wave (the tile's ranges).
struct Ranges {
  int lo[2], hi[2];    // this lane's
  int tlo[2], thi[2];  // the tile's (wave-uniform)
};
__device__ __forceinline__ void make_union(Ranges& g) {
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const bool some = g.lo[i] < g.hi[i];
    int lo = some ? g.lo[i] : INT_MAX, hi = some ? g.hi[i] : INT_MIN;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
      const int l2 = __shfl_xor(lo, off, 64), h2 = __shfl_xor(hi, off, 64);
      lo = lo < l2 ? lo : l2;
      hi = hi > h2 ? hi : h2;
    }
    g.tlo[i] = __builtin_amdgcn_readfirstlane(lo);
    g.thi[i] = __builtin_amdgcn_readfirstlane(hi);
  }
}
__device__ __forceinline__ Ranges ranges_of(const int64_t* bounds, const int32_t* row_segment,
                                            int row, bool valid, int64_t B, bool of_query) {
  Ranges g = {{0, 0}, {0, 0}, {0, 0}, {0, 0}};
  if (valid) {
    const SegRow s = seg_row(bounds, row_segment, row);
    int64_t a0, a1, b0, b1;
    if (of_query) query_key_ranges(s, B, a0, a1, b0, b1);
    else key_query_ranges(s, B, a0, a1, b0, b1);
    g.lo[0] = (int)a0; g.hi[0] = (int)a1; g.lo[1] = (int)b0; g.hi[1] = (int)b1;
  }
  make_union(g);
  return g;
}

// Sum over the waves of this workgroup, in wave order, of acc (each wave's
// weighted by w[its index] per lane); wave v then stores its quarter of the
// rows' columns: float4 at row `out`, scaled.
__device__ __forceinline__ void combine(float4* lds, const f32x16_t (&acc)[NB], const float* w,
                                        int wave, int lane, float scale, float* out, bool store) {
  const int half = lane >> 5;
#pragma unroll
  for (int t = 0; t < 16; ++t)
    lds[(wave * 16 + t) * 64 + lane] = make_float4(acc[0][t], acc[1][t], acc[2][t], acc[3][t]);
  __syncthreads();
#pragma unroll
  for (int e = 0; e < 4; ++e) {  // element 4 wave + e: columns 4 (8 wave + 4 half + e) + 0..3
    float4 s = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
    for (int v = 0; v < AW; ++v) {
      const float4 x = lds[(v * 16 + 4 * wave + e) * 64 + lane];
      const float c = w ? w[v] : 1.f;
      s.x += c * x.x; s.y += c * x.y; s.z += c * x.z; s.w += c * x.w;
    }
    if (store)
      *reinterpret_cast<float4*>(out + 4 * (8 * wave + 4 * half + e)) =
          make_float4(s.x * scale, s.y * scale, s.z * scale, s.w * scale);
  }
}

}  // namespace

__global__ void __launch_bounds__(64 * AW, 1)
attn_fwd_f32_kernel(const float* __restrict__ q, const float* __restrict__ k,
                    const float* __restrict__ v, int64_t ldv, const int64_t* __restrict__ bounds,
                    const int32_t* __restrict__ row_segment, float* __restrict__ o,
                    float* __restrict__ lse, int rows, int nq, int nkv, int64_t B, float scale) {
  __shared__ float4 lds[AW * 16 * 64];
  __shared__ float ml[2][AW][32];
  __shared__ int flags[AW];
  const int lane = threadIdx.x & 63, half = lane >> 5, col = lane & 31;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int h = blockIdx.x, hk = h / (nq / nkv);
  const int row = blockIdx.y * 32 + col;
  const bool valid = row < rows;
  const int64_t ldq = (int64_t)nq * HD, ldk = (int64_t)nkv * HD;
  const Ranges g = ranges_of(bounds, row_segment, row, valid, B, true);
  float4 qf[NK];
  row_frags(q + (int64_t)(valid ? row : rows - 1) * ldq + h * HD, half, qf);
  const float* kh = k + hk * HD;
  const float* vh = v + hk * HD;
  f32x16_t acc[NB] = {zero16(), zero16(), zero16(), zero16()};
  float m = -INFINITY, l = 0.f;
  float z = 0.f;
  int turn = 0;
#pragma unroll 1
  for (int rg = 0; rg < 2; ++rg)
#pragma unroll 1
    for (int k0 = g.tlo[rg]; k0 < g.thi[rg]; k0 += 32, ++turn) {
      if (turn % AW != wave) continue;
      const int last = g.thi[rg] - 1;
      const int kr = k0 + col < last ? k0 + col : last;
      f32x16_t s = dot_rows(kh + kr * ldk, half, qf);
      float mx = -INFINITY;
#pragma unroll
      for (int t = 0; t < 16; ++t) {
        const int key = k0 + 8 * (t >> 2) + 4 * half + (t & 3);
        s[t] = key >= g.lo[rg] && key < g.hi[rg] ? s[t] * scale : -INFINITY;
        mx = fmaxf(mx, s[t]);
      }
      mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
      const float mn = fmaxf(m, mx), use = mn == -INFINITY ? 0.f : mn;
      const float corr = expf(m - use);  // 0 when m was -inf
      float sum = 0.f;
#pragma unroll
      for (int t = 0; t < 16; ++t) {
        s[t] = expf(s[t] - use);
        sum += s[t];
      }
      l = l * corr + (sum + __shfl_xor(sum, 32, 64));
      m = mn;
#pragma unroll
      for (int i = 0; i < NB; ++i)
#pragma unroll
        for (int t = 0; t < 16; ++t) acc[i][t] *= corr;
      add_rows(acc, vh, ldv, k0, last, col, half, s, z);
    }
  if (half == 0) { ml[0][wave][col] = m; ml[1][wave][col] = l; }
  if (any_wave(flags, wave, lane, z)) {  // the rows one by one, which reads allowed keys only
    for (int r = blockIdx.y * 32 + wave; r < rows && r < (int)(blockIdx.y + 1) * 32; r += AW)
      attn_fwd_row<float>(q, k, v, ldv, bounds, row_segment, o, lse, rows, nq, nkv, HD, B, scale, r,
                          h);
    return;
  }
  float M = -INFINITY, L = 0.f, w[AW];
#pragma unroll
  for (int i = 0; i < AW; ++i) M = fmaxf(M, ml[0][i][col]);
#pragma unroll
  for (int i = 0; i < AW; ++i) {
    w[i] = ml[0][i][col] == -INFINITY ? 0.f : expf(ml[0][i][col] - M);
    L += ml[1][i][col] * w[i];
  }
  combine(lds, acc, w, wave, lane, 1.0f / L, o + row * ldq + h * HD, valid);
  if (valid && threadIdx.x < 32) lse[(int64_t)h * rows + row] = M + logf(L);
}

__global__ void __launch_bounds__(64 * AW, 1)
attn_dq_f32_kernel(const float* __restrict__ q, const float* __restrict__ k,
                   const float* __restrict__ v, int64_t ldv, const float* __restrict__ lse,
                   const float* __restrict__ delta, const float* __restrict__ dout,
                   const int64_t* __restrict__ bounds, const int32_t* __restrict__ row_segment,
                   float* __restrict__ dq, int rows, int nq, int nkv, int64_t B, float scale) {
  __shared__ float4 lds[AW * 16 * 64];
  __shared__ int flags[AW];
  const int lane = threadIdx.x & 63, half = lane >> 5, col = lane & 31;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int h = blockIdx.x, hk = h / (nq / nkv);
  const int row = blockIdx.y * 32 + col;
  const bool valid = row < rows;
  const int64_t ldq = (int64_t)nq * HD, ldk = (int64_t)nkv * HD;
  const Ranges g = ranges_of(bounds, row_segment, row, valid, B, true);
  const int rr = valid ? row : rows - 1;
  float4 qf[NK], df[NK];
  row_frags(q + rr * ldq + h * HD, half, qf);
  row_frags(dout + rr * ldq + h * HD, half, df);
  const float ls = lse[(int64_t)h * rows + rr], de = delta[(int64_t)h * rows + rr];
  const float* kh = k + hk * HD;
  const float* vh = v + hk * HD;
  f32x16_t acc[NB] = {zero16(), zero16(), zero16(), zero16()};
  float z = 0.f;
  int turn = 0;
#pragma unroll 1
  for (int rg = 0; rg < 2; ++rg)
#pragma unroll 1
    for (int k0 = g.tlo[rg]; k0 < g.thi[rg]; k0 += 32, ++turn) {
      if (turn % AW != wave) continue;
      const int last = g.thi[rg] - 1;
      const int kr = k0 + col < last ? k0 + col : last;
      f32x16_t s = dot_rows(kh + kr * ldk, half, qf);
      const f32x16_t dp = dot_rows(vh + kr * ldv, half, df);
#pragma unroll
      for (int t = 0; t < 16; ++t) {
        const int key = k0 + 8 * (t >> 2) + 4 * half + (t & 3);
        s[t] = key >= g.lo[rg] && key < g.hi[rg]
                   ? expf(s[t] * scale - ls) * (dp[t] - de) * scale : 0.f;
      }
      add_rows(acc, kh, ldk, k0, last, col, half, s, z);
    }
  if (any_wave(flags, wave, lane, z)) {
    for (int r = blockIdx.y * 32 + wave; r < rows && r < (int)(blockIdx.y + 1) * 32; r += AW)
      attn_dq_row<float>(q, k, v, ldv, lse, delta, dout, bounds, row_segment, dq, rows, nq, nkv, HD,
                         B, scale, r, h);
    return;
  }
  combine(lds, acc, nullptr, wave, lane, 1.f, dq + row * ldq + h * HD, valid);
}

__global__ void __launch_bounds__(64 * AW, 1)
attn_dkdv_f32_kernel(const float* __restrict__ q, const float* __restrict__ k,
                     const float* __restrict__ v, int64_t ldv, const float* __restrict__ lse,
                     const float* __restrict__ delta, const float* __restrict__ dout,
                     const int64_t* __restrict__ bounds, const int32_t* __restrict__ row_segment,
                     float* __restrict__ dk, float* __restrict__ dv, int64_t lddv, int rows,
                     int nq, int nkv, int64_t B, float scale) {
  __shared__ float4 lds[AW * 16 * 64];
  __shared__ int flags[AW];
  const int lane = threadIdx.x & 63, half = lane >> 5, col = lane & 31;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int hk = blockIdx.x, group = nq / nkv;
  const int row = blockIdx.y * 32 + col;
  const bool valid = row < rows;
  const int64_t ldq = (int64_t)nq * HD, ldk = (int64_t)nkv * HD;
  const Ranges g = ranges_of(bounds, row_segment, row, valid, B, false);
  const int rr = valid ? row : rows - 1;
  float4 kf[NK], vf[NK];
  row_frags(k + rr * ldk + hk * HD, half, kf);
  row_frags(v + rr * ldv + hk * HD, half, vf);
  f32x16_t dka[NB] = {zero16(), zero16(), zero16(), zero16()};
  f32x16_t dva[NB] = {zero16(), zero16(), zero16(), zero16()};
  float z = 0.f;
  int turn = 0;
#pragma unroll 1
  for (int h = hk * group; h < (hk + 1) * group; ++h) {
    const float* qh = q + h * HD;
    const float* dh = dout + h * HD;
#pragma unroll 1
    for (int rg = 0; rg < 2; ++rg)
#pragma unroll 1
      for (int q0 = g.tlo[rg]; q0 < g.thi[rg]; q0 += 32, ++turn) {
        if (turn % AW != wave) continue;
        const int last = g.thi[rg] - 1;
        const int qr = q0 + col < last ? q0 + col : last;
        f32x16_t p = dot_rows(qh + qr * ldq, half, kf);
        f32x16_t ds = dot_rows(dh + qr * ldq, half, vf);
#pragma unroll
        for (int t = 0; t < 16; ++t) {
          const int qi = q0 + 8 * (t >> 2) + 4 * half + (t & 3);
          const int64_t at = (int64_t)h * rows + (qi < last ? qi : last);
          const bool in = qi >= g.lo[rg] && qi < g.hi[rg];
          p[t] = in ? expf(p[t] * scale - lse[at]) : 0.f;
          ds[t] = in ? p[t] * (ds[t] - delta[at]) * scale : 0.f;
        }
        add_rows(dva, dh, ldq, q0, last, col, half, p, z);
        add_rows(dka, qh, ldq, q0, last, col, half, ds, z);
      }
  }
  if (any_wave(flags, wave, lane, z)) {
    for (int r = blockIdx.y * 32 + wave; r < rows && r < (int)(blockIdx.y + 1) * 32; r += AW)
      attn_dkdv_row<float>(q, k, v, ldv, lse, delta, dout, bounds, row_segment, dk, dv, lddv, rows,
                           nq, nkv, HD, B, scale, r, hk);
    return;
  }
  combine(lds, dka, nullptr, wave, lane, 1.f, dk + row * ldk + hk * HD, valid);
  __syncthreads();
  combine(lds, dva, nullptr, wave, lane, 1.f, dv + row * lddv + hk * HD, valid);
}

// float, head_dim 128, 16-byte aligned rows; row indices (a window's keys may
// start before row 0) as 32-bit.
bool attn_f32_eligible(int64_t rows, int64_t nq, int64_t nkv, int64_t dh, int64_t ldv) {
  return dh == HD && ldv % 4 == 0 && rows < (1 << 21) && nq <= 65535 && nkv <= 65535;
}

void attn_f32_fwd_launch(const float* q, const float* k, const float* v, int64_t ldv,
                         const int64_t* bounds, const int32_t* row_segment, float* o, float* lse,
                         int64_t rows, int64_t nq, int64_t nkv, int64_t B, float scale,
                         hipStream_t st) {
  const dim3 grid((unsigned)nq, ceil_div_u(rows, 32));
  attn_fwd_f32_kernel<<<grid, 64 * AW, 0, st>>>(q, k, v, ldv, bounds, row_segment, o, lse,
                                                (int)rows, (int)nq, (int)nkv, B, scale);
}

void attn_f32_bwd_launch(const float* q, const float* k, const float* v, int64_t ldv,
                         const float* lse, const float* delta, const float* dout,
                         const int64_t* bounds, const int32_t* row_segment, float* dq, float* dk,
                         float* dv, int64_t lddv, int64_t rows, int64_t nq, int64_t nkv, int64_t B,
                         float scale, hipStream_t st) {
  const dim3 gq((unsigned)nq, ceil_div_u(rows, 32)), gk((unsigned)nkv, ceil_div_u(rows, 32));
  attn_dq_f32_kernel<<<gq, 64 * AW, 0, st>>>(q, k, v, ldv, lse, delta, dout, bounds, row_segment,
                                             dq, (int)rows, (int)nq, (int)nkv, B, scale);
  attn_dkdv_f32_kernel<<<gk, 64 * AW, 0, st>>>(q, k, v, ldv, lse, delta, dout, bounds, row_segment,
                                               dk, dv, lddv, (int)rows, (int)nq, (int)nkv, B,
                                               scale);
}
