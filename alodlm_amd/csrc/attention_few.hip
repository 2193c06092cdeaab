// bf16 attention forward for head_dim 128 where the query tiles are too few to
// fill the chip (a decoder window of 16 to 64 rows after thousands of cached
// keys, a prompt's prefill, one short conversation).
//
// The 128-row kernel (attention_fa128.hip) walks all keys of a tile in one
// workgroup: 27 rows after 3100 keys took 68 us on 32 workgroups, a chain of
// 49 key tiles.  Here a workgroup owns 32 query rows of one head and its eight
// waves take the 32-key tiles in turn, so the chain is an eighth as long (and
// 777 rows make 400 workgroups instead of 112).  Bound: the latency of a key
// tile's loads, hidden by loading the next tile's keys during this one's
// softmax; there is no barrier before the waves meet, so operands come from
// global memory straight into registers:
//  * S^T = K Q^T: 16 bytes of key row `lane % 32` per MFMA 32x32x16 (lane half
//    = 8 of the 16 k), Q fragments held in registers; a lane then holds one
//    query and the keys 8 a + 4 half + e;
//  * O^T = V^T P^T: P's registers are the operand as they are (elements 8 s ..
//    8 s + 7 of step s are keys 16 s + 4 half + {0..3, 8..11}); for V^T a lane
//    loads columns 4 col .. 4 col + 3 of those eight rows and regroups them, so
//    block d of the output holds columns 4 i + d (i the block row).
// A decoder layer call of 27 rows after 3100 at the 8B shapes 196 -> 173 us, of
// 16 after 300 at the 1.7B shapes 96 -> 92 us, a 777-row prefill 185 -> 181 us.
// The waves' sums are scaled to the common maximum and added in LDS in wave
// order.
#include <limits.h>

#include "attention_common.h"

namespace {

constexpr int HD = 128, NB = 4, FW = 8;  // waves

__device__ __forceinline__ f32x16_t mfma16(bf16x8_t a, bf16x8_t b, f32x16_t c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

// Column d (0..3) of the 4-column pieces of eight rows as one operand.
__device__ __forceinline__ bf16x8_t column8(const uint2 (&r)[8], int d) {
  uint32_t w[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const uint32_t a = d < 2 ? r[2 * i].x : r[2 * i].y, b = d < 2 ? r[2 * i + 1].x : r[2 * i + 1].y;
    w[i] = (d & 1) ? (a >> 16) | (b & 0xffff0000u) : (a & 0xffffu) | (b << 16);
  }
  return __builtin_bit_cast(bf16x8_t, make_uint4(w[0], w[1], w[2], w[3]));
}

}  // namespace

__global__ void __launch_bounds__(64 * FW, 1)
fa128_few_kernel(const bf16_t* __restrict__ q, const bf16_t* __restrict__ k,
                 const bf16_t* __restrict__ v, int64_t ldv, const int64_t* __restrict__ bounds,
                 const int32_t* __restrict__ tiles, bf16_t* __restrict__ o,
                 float* __restrict__ lse, int64_t N, int nq, int nkv, int B, float scale) {
  __shared__ float4 sums[FW / 2][16][64];
  __shared__ float ml[2][FW][32];
  const int lane = threadIdx.x & 63, half = lane >> 5, col = lane & 31;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int h = blockIdx.x, hk = h / (nq / nkv);
  // 32 rows of a 128-row tile of the list
  const int seg = tiles[2 * (blockIdx.y >> 2)], tile = tiles[2 * (blockIdx.y >> 2) + 1];
  const int64_t base = bounds[seg];
  const int L = (int)((bounds[seg + 1] - base) / 2);
  const int end = tile < L ? L : 2 * L;
  const int q0 = tile + 32 * (int)(blockIdx.y & 3);
  const int q1 = (q0 + 32 < end ? q0 + 32 : end);
  if (q0 >= q1) return;  // the whole workgroup
  const int qi = q0 + col;
  const bool valid = qi < q1;
  const int64_t ldq = (int64_t)nq * HD, ldk = (int64_t)nkv * HD;
  const float c = scale * FA_LOG2E;

  const bf16_t* qr = q + (base + (valid ? qi : q1 - 1)) * ldq + h * HD + 8 * half;
  bf16x8_t qf[HD / 16];
#pragma unroll
  for (int kk = 0; kk < HD / 16; ++kk) qf[kk] = load_frag(qr + 16 * kk);
  const Interval2 mine = keys_of_query(qi, valid, L, B);
  const Interval2 R = key_ranges(q0, q1, L, B);
  const int n0 = R.hi0 > R.lo0 ? (R.hi0 - R.lo0 + 31) / 32 : 0;
  const int n1 = R.hi1 > R.lo1 ? (R.hi1 - R.lo1 + 31) / 32 : 0;
  const bf16_t* kh = k + base * ldk + hk * HD + 8 * half;
  const bf16_t* vh = v + base * ldv + hk * HD + 4 * col;
  // key tile t of the two ranges: first key, last key of the range
  auto first = [&](int t) { return t < n0 ? R.lo0 + 32 * t : R.lo1 + 32 * (t - n0); };
  auto last = [&](int t) { return (t < n0 ? R.hi0 : R.hi1) - 1; };
  bf16x8_t kf[HD / 16];
  auto load_keys = [&](int t) {
    const int key = first(t) + col, end_key = last(t);
    const bf16_t* p = kh + (int64_t)(key < end_key ? key : end_key) * ldk;
#pragma unroll
    for (int kk = 0; kk < HD / 16; ++kk) kf[kk] = load_frag(p + 16 * kk);
  };

  f32x16_t acc[NB] = {zero16(), zero16(), zero16(), zero16()};
  float m = -INFINITY, l = 0.f;  // running maximum (log2 units) and sum
  if (wave < n0 + n1) load_keys(wave);
#pragma unroll 1
  for (int t = wave; t < n0 + n1; t += FW) {
    const int k0 = first(t), end_key = last(t);
    const int lo = t < n0 ? mine.lo0 : mine.lo1, hi = t < n0 ? mine.hi0 : mine.hi1;
    uint2 vr[2][8];  // value rows 16 s + 4 half + {0..3, 8..11}, columns 4 col ..
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int key = k0 + 16 * s + 4 * half + (j < 4 ? j : j + 4);
        vr[s][j] = *reinterpret_cast<const uint2*>(vh + (int64_t)(key < end_key ? key : end_key) * ldv);
      }
    f32x16_t sc = zero16();
#pragma unroll
    for (int kk = 0; kk < HD / 16; ++kk) sc = mfma16(kf[kk], qf[kk], sc);
    if (t + FW < n0 + n1) load_keys(t + FW);
    float mx = -INFINITY;
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      const int key = k0 + 8 * (e >> 2) + 4 * half + (e & 3);
      sc[e] = key >= lo && key < hi ? sc[e] * c : -INFINITY;
      mx = fmaxf(mx, sc[e]);
    }
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
    const float mn = fmaxf(m, mx), use = mn == -INFINITY ? 0.f : mn;
    const float corr = fast_exp2(m - use);  // 0 when m was -inf
    float sum = 0.f;
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      sc[e] = fast_exp2(sc[e] - use);
      sum += sc[e];
    }
    l = l * corr + (sum + __shfl_xor(sum, 32, 64));
    m = mn;
#pragma unroll
    for (int d = 0; d < NB; ++d)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[d][e] *= corr;
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      const bf16x8_t p = pack8(sc, 8 * s);
#pragma unroll
      for (int d = 0; d < NB; ++d) acc[d] = mfma16(column8(vr[s], d), p, acc[d]);
    }
  }

  // the common maximum and this wave's weight
  if (half == 0) { ml[0][wave][col] = m; ml[1][wave][col] = l; }
  __syncthreads();
  float M = -INFINITY, sum = 0.f;
#pragma unroll
  for (int w = 0; w < FW; ++w) M = fmaxf(M, ml[0][w][col]);
#pragma unroll
  for (int w = 0; w < FW; ++w) sum += ml[1][w][col] * (ml[0][w][col] == -INFINITY ? 0.f : fast_exp2(ml[0][w][col] - M));
  const float mine_w = m == -INFINITY ? 0.f : fast_exp2(m - M);
  auto put = [&](int slot) {
#pragma unroll
    for (int e = 0; e < 16; ++e)
      sums[slot][e][lane] = make_float4(acc[0][e] * mine_w, acc[1][e] * mine_w,
                                        acc[2][e] * mine_w, acc[3][e] * mine_w);
  };
  if (wave < FW / 2) put(wave);
  __syncthreads();
  float4 part[2];  // elements 2 wave, 2 wave + 1 of the first four waves
#pragma unroll
  for (int e = 0; e < 2; ++e) {
    float4 s = sums[0][2 * wave + e][lane];
#pragma unroll
    for (int w = 1; w < FW / 2; ++w) {
      const float4 x = sums[w][2 * wave + e][lane];
      s.x += x.x; s.y += x.y; s.z += x.z; s.w += x.w;
    }
    part[e] = s;
  }
  __syncthreads();
  if (wave >= FW / 2) put(wave - FW / 2);
  __syncthreads();
  const float inv = 1.0f / sum;
#pragma unroll
  for (int e = 0; e < 2; ++e) {
    float4 s = part[e];
#pragma unroll
    for (int w = 0; w < FW / 2; ++w) {
      const float4 x = sums[w][2 * wave + e][lane];
      s.x += x.x; s.y += x.y; s.z += x.z; s.w += x.w;
    }
    // element t = 4 a + b: block row 8 a + 4 half + b
    const int t = 2 * wave + e, i = 8 * (t >> 2) + 4 * half + (t & 3);
    if (valid)
      *reinterpret_cast<uint2*>(o + (base + qi) * ldq + h * HD + 4 * i) =
          make_uint2(pack2(s.x * inv, s.y * inv), pack2(s.z * inv, s.w * inv));
  }
  if (valid && threadIdx.x < 32)
    lse[(int64_t)h * N + base + qi] = M * FA_LN2 + logf(sum);
}

void fa128_few_launch(const bf16_t* q, const bf16_t* k, const bf16_t* v, int64_t ldv,
                      const int64_t* bounds, const int32_t* tiles, int64_t n_tiles, bf16_t* o,
                      float* lse, int64_t N, int nq, int nkv, int B, float scale, hipStream_t st) {
  fa128_few_kernel<<<dim3((unsigned)nq, (unsigned)(4 * n_tiles)), 64 * FW, 0, st>>>(
      q, k, v, ldv, bounds, tiles, o, lse, N, nq, nkv, B, scale);
}
