// Products of a few rows with a weight matrix (the decoder's windows):
//   C[m, n] = alpha * sum_k A[m, k] W[n, k],  M <= SKINNY_M, both k-contiguous,
// bf16 or float, plain or added to a residual.
//
// Bound: the weights, read once.  A 128x128 tile kernel leaves such a product
// on N / 128 workgroups, each a serial walk over K.  Here a workgroup owns 16
// (or 32) weight rows and its 8 waves split K between them, so that N / 16
// workgroups keep 8 waves of loads in flight and no wave walks more than K / 8;
// fragments go from global memory straight to the MFMA (a weight element is
// used by one wave only, so LDS staging would only add latency), each wave's
// sums meet in LDS once and are added in wave order.  The rows of A are re-read
// per workgroup from L2.  16 rows, bf16, against the tile kernels: 4096 x 2048
// 6.3 us (29.6), 2048 x 2048 5.8 (38.4), 12288 x 2048 14.4 (37.3), 2048 x 6144
// 12.9 (103.6); 27 rows, 24576 x 4096 59 us (77), 3.4 TB/s of weights.  More
// loads in flight per wave do not raise that: a CU's vector memory path takes
// about 30 KB/us of these 64-byte row pieces (weights and A together).
//
// Fragment: lane l holds 16 bytes of row l % 16 at 16-byte chunk l / 16, i.e.
// 64 bytes of each of 16 rows per instruction; two neighbouring fragments are
// one 128-byte line per row.  For float the four k of a lane's chunk feed four
// 16x16x4 MFMAs (both operands permute k alike, which only reorders the sum).
#include "common.h"
#include "gemm_skinny.h"

typedef __attribute__((__vector_size__(8 * sizeof(short)))) short bf16x8_t;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float f32x4_t;

namespace {

constexpr int WAVES = 8;

template <typename T> struct SkinnyType;
template <> struct SkinnyType<bf16_t> {
  static constexpr int VEC = 8, KS = 32;  // elements per lane, k per fragment
  static __device__ __forceinline__ f32x4_t mma(uint4 w, uint4 x, f32x4_t acc) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, w),
                                                   __builtin_bit_cast(bf16x8_t, x), acc, 0, 0, 0);
  }
};
template <> struct SkinnyType<float> {
  static constexpr int VEC = 4, KS = 16;
  static __device__ __forceinline__ f32x4_t mma(uint4 w, uint4 x, f32x4_t acc) {
    acc = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(w.x), __uint_as_float(x.x), acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(w.y), __uint_as_float(x.y), acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(w.z), __uint_as_float(x.z), acc, 0, 0, 0);
    return __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(w.w), __uint_as_float(x.w), acc, 0, 0, 0);
  }
};

// One 16-byte chunk of a bf16 row of x, normalised: w * cast(x * r), as the RMSNorm
// kernels round.
__device__ __forceinline__ uint4 normed(uint4 x, uint4 w, float r) {
  const uint32_t xv[4] = {x.x, x.y, x.z, x.w}, wv[4] = {w.x, w.y, w.z, w.w};
  uint32_t o[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const uint32_t t = pack_bf16x2(bf16_to_float((bf16_t)(xv[e] & 0xffffu)) * r,
                                   bf16_to_float((bf16_t)(xv[e] >> 16)) * r);
    o[e] = pack_bf16x2(bf16_to_float((bf16_t)(wv[e] & 0xffffu)) * bf16_to_float((bf16_t)(t & 0xffffu)),
                       bf16_to_float((bf16_t)(wv[e] >> 16)) * bf16_to_float((bf16_t)(t >> 16)));
  }
  return make_uint4(o[0], o[1], o[2], o[3]);
}
// What the product does beside A W^T (bf16): SKINNY_NORM takes A through an
// RMSNorm (weight nw, eps) first, SKINNY_GLU has W's first half of rows as gate and its
// second half as up projection and stores silu(gate) * up (N / 2 columns).
constexpr int SKINNY_NORM = 1, SKINNY_GLU = 2;

// MT: 16-row blocks of A; NT: 16-row blocks of W per workgroup; U: fragment
// pairs per operand block and register set (two sets: one loading, one used).
template <typename T, int MT, int NT, int U, int EPI, int FUSE = 0>
__global__ void __launch_bounds__(64 * WAVES)
gemm_skinny_kernel(const T* __restrict__ A, int64_t lda, const T* __restrict__ W, int64_t ldw,
                   T* C, int64_t ldc, const T* R, int64_t ldr, int M, int N, int K, float alpha,
                   const T* __restrict__ nw, float eps) {
  typedef SkinnyType<T> S;
  constexpr int STEP = 2 * S::KS;  // k per fragment pair
  constexpr int COLS = 16 * NT, ROWS = 16 * MT;
  constexpr bool NORM = FUSE & SKINNY_NORM, GLU = FUSE & SKINNY_GLU;
  static_assert(!GLU || NT == 2, "one gate block and one up block");
  __shared__ __attribute__((aligned(16))) float red[WAVES][ROWS][COLS];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int i = lane & 15, kl = S::VEC * (lane >> 4);
  const int n0 = blockIdx.x * (GLU ? 16 : COLS);
  const int cols = GLU ? N / 2 : N;  // of the output
  // Operands as buffers based at the workgroup's rows: one 32-bit lane offset
  // per block, and a chunk past K reads at an offset the range check turns
  // into zeros, so the loop has no branch around a load.
  constexpr uint32_t ES = sizeof(T), OUT = 0xffffff00u;
  const int64_t nrows = GLU ? N - n0 : N - n0 < COLS ? N - n0 : COLS;
  const __amdgpu_buffer_rsrc_t wr = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<T*>(W) + (int64_t)n0 * ldw, 0, (int)(((nrows - 1) * ldw + K) * ES), 0x00020000);
  const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<T*>(A), 0, (int)(((M - 1) * lda + K) * ES), 0x00020000);
  uint32_t wo[NT], xo[MT];
#pragma unroll
  for (int b = 0; b < NT; ++b) {  // rows past the edge re-read the last one (never stored)
    const int64_t r = GLU ? (int64_t)b * cols + (n0 + i < cols ? i : cols - 1 - n0)
                          : 16 * b + i < nrows ? 16 * b + i : nrows - 1;
    wo[b] = (uint32_t)((r * ldw + kl) * ES);
  }
#pragma unroll
  for (int a = 0; a < MT; ++a) {
    const int m = 16 * a + i;
    xo[a] = (uint32_t)(((int64_t)(m < M ? m : M - 1) * lda + kl) * ES);
  }
  f32x4_t acc[MT][NT];
#pragma unroll
  for (int a = 0; a < MT; ++a)
#pragma unroll
    for (int b = 0; b < NT; ++b) acc[a][b] = f32x4_t{0.f, 0.f, 0.f, 0.f};

  // 1 / rms of the rows (every workgroup for itself: 16 rows of 2048 are 64 KB
  // from L2, less than a launch of its own costs)
  float rs[MT];
  __amdgpu_buffer_rsrc_t nr;
  if constexpr (NORM) {
    __shared__ float inv_rms[ROWS];
    nr = __builtin_amdgcn_make_buffer_rsrc(const_cast<T*>(nw), 0, (int)(K * ES), 0x00020000);
    for (int m = wave; m < M; m += WAVES) {
      float s = 0.f;
      for (int c = lane * 8; c < K; c += 512) {  // the RMSNorm kernels' order: the same bits
        float v[8];
        Vec8<T>::load(A + (int64_t)m * lda + c, v);
#pragma unroll
        for (int e = 0; e < 8; ++e) s = fmaf(v[e], v[e], s);
      }
      s = wave_sum(s);
      if (lane == 0) inv_rms[m] = 1.0f / sqrtf(s / (float)K + eps);
    }
    __syncthreads();
#pragma unroll
    for (int a = 0; a < MT; ++a) rs[a] = inv_rms[16 * a + i < M ? 16 * a + i : M - 1];
  }

  uint4 w[2][U][2][NT], x[2][U][2][MT], nv[NORM ? 2 : 1][U][2];
  auto fetch = [&](const int set, const int k) {
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int kk = k + u * WAVES * STEP + h * S::KS;
        const bool in = kk + kl + S::VEC <= K;
#pragma unroll
        for (int b = 0; b < NT; ++b)
          w[set][u][h][b] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(
              wr, in ? wo[b] + kk * ES : OUT, 0, 0));
        if constexpr (NORM)
          nv[set][u][h] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(
              nr, in ? (kk + kl) * ES : OUT, 0, 0));
#pragma unroll
        for (int a = 0; a < MT; ++a)
          x[set][u][h][a] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(
              xr, in ? xo[a] + kk * ES : OUT, 0, 0));
      }
  };
  auto product = [&](const int set) {
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int a = 0; a < MT; ++a) {
          uint4 xa = x[set][u][h][a];
          if constexpr (NORM) xa = normed(xa, nv[set][u][h], rs[a]);
#pragma unroll
          for (int b = 0; b < NT; ++b) acc[a][b] = S::mma(w[set][u][h][b], xa, acc[a][b]);
        }
  };
  constexpr int SPAN = U * WAVES * STEP;
  const int k0 = wave * STEP;
  if (k0 < K) fetch(0, k0);
  for (int k = k0; k < K; k += 2 * SPAN) {
    if (k + SPAN < K) fetch(1, k + SPAN);
    product(0);
    if (k + SPAN < K) {
      if (k + 2 * SPAN < K) fetch(0, k + 2 * SPAN);
      product(1);
    }
  }

  // lane: row lane % 16, columns 4 (lane / 16) .. +3 of each 16x16 block
#pragma unroll
  for (int a = 0; a < MT; ++a)
#pragma unroll
    for (int b = 0; b < NT; ++b)
      *reinterpret_cast<f32x4_t*>(&red[wave][16 * a + i][16 * b + 4 * (lane >> 4)]) = acc[a][b];
  __syncthreads();
  constexpr int OUTS = GLU ? 16 : COLS;
  for (int t = threadIdx.x; t < ROWS * OUTS; t += 64 * WAVES) {
    const int m = t / OUTS, c = t % OUTS, n = n0 + c;
    if (m >= M || n >= cols) continue;
    float v = 0.f;
#pragma unroll
    for (int s = 0; s < WAVES; ++s) v += red[s][m][c];
    v *= alpha;
    if constexpr (GLU) {
      float up = 0.f;
#pragma unroll
      for (int s = 0; s < WAVES; ++s) up += red[s][m][16 + c];
      const float g = Elem<T>::round(v);
      v = Elem<T>::round(g / (1.0f + expf(-g))) * Elem<T>::round(alpha * up);
    }
    if (EPI == ALODLM_EPI_RESIDUAL) v = Elem<T>::load(R, m * ldr + n) + Elem<T>::round(v);
    Elem<T>::store(C, m * ldc + n, v);
  }
}

template <typename T, int MT, int NT, int U>
void launch(const T* A, int64_t lda, const T* W, int64_t ldw, T* C, int64_t ldc, const T* R,
            int64_t ldr, int M, int N, int K, float alpha, int epi, hipStream_t st) {
  const unsigned grid = ceil_div_u(N, 16 * NT);
  if (epi == ALODLM_EPI_STORE)
    gemm_skinny_kernel<T, MT, NT, U, ALODLM_EPI_STORE><<<grid, 64 * WAVES, 0, st>>>(
        A, lda, W, ldw, C, ldc, R, ldr, M, N, K, alpha, nullptr, 0.f);
  else
    gemm_skinny_kernel<T, MT, NT, U, ALODLM_EPI_RESIDUAL><<<grid, 64 * WAVES, 0, st>>>(
        A, lda, W, ldw, C, ldc, R, ldr, M, N, K, alpha, nullptr, 0.f);
}

template <typename T, int NT>
void launch_rows(const T* A, int64_t lda, const T* W, int64_t ldw, T* C, int64_t ldc, const T* R,
                 int64_t ldr, int M, int N, int K, float alpha, int epi, hipStream_t st) {
  if (M <= 16) launch<T, 1, NT, 2>(A, lda, W, ldw, C, ldc, R, ldr, M, N, K, alpha, epi, st);
  else if (M <= 32) launch<T, 2, NT, 2>(A, lda, W, ldw, C, ldc, R, ldr, M, N, K, alpha, epi, st);
  else if (M <= 48) launch<T, 3, NT, 1>(A, lda, W, ldw, C, ldc, R, ldr, M, N, K, alpha, epi, st);
  else launch<T, 4, NT, 1>(A, lda, W, ldw, C, ldc, R, ldr, M, N, K, alpha, epi, st);
}

template <typename T>
void launch_typed(const void* A, int64_t lda, const void* W, int64_t ldw, void* C, int64_t ldc,
                  const void* R, int64_t ldr, int64_t M, int64_t N, int64_t K, float alpha,
                  int epi, hipStream_t st) {
  // A workgroup reads its 16 NT weight rows and all of A: 32 weight rows halve
  // the re-reads of A, but also the workgroups.  They win where 16 would give
  // more than one workgroup per CU and A is more than one block (27 rows, 6144
  // x 4096: 20.4 us against 24.0; 24576 x 4096: 59 against 69; but 4096 x
  // 12288: 54 against 38) or more than three per CU (48 x 24576 x 4096: 70
  // against 97; one block of 16 rows, 12288 x 2048: 15.4 against 14.4).
  if ((N > 16 * 256 && M > 16) || N > 16 * 3 * 256)
    launch_rows<T, 2>((const T*)A, lda, (const T*)W, ldw, (T*)C, ldc, (const T*)R, ldr, (int)M,
                      (int)N, (int)K, alpha, epi, st);
  else
    launch_rows<T, 1>((const T*)A, lda, (const T*)W, ldw, (T*)C, ldc, (const T*)R, ldr, (int)M,
                      (int)N, (int)K, alpha, epi, st);
}

// 16 rows after 300 cached ones at the 1.7B shapes, a whole decoder layer call:
// 92 us with the norms, the products, SwiGLU and the value copy in launches of
// their own, 66 us with both norms and SwiGLU in the products and the values
// copied by the rotary kernel.  float rows lose (154 us to 169): their norm
// re-reads twice the bytes.
void launch_fused(const bf16_t* A, int64_t lda, const bf16_t* nw, float eps, const bf16_t* W,
                  int64_t ldw, bf16_t* C, int64_t ldc, int M, int N, int K, bool glu,
                  hipStream_t st) {
  if (glu)
    gemm_skinny_kernel<bf16_t, 1, 2, 2, ALODLM_EPI_STORE, SKINNY_NORM | SKINNY_GLU>
        <<<ceil_div_u(N / 2, 16), 64 * WAVES, 0, st>>>(A, lda, W, ldw, C, ldc, nullptr, 0, M, N, K,
                                                       1.f, nw, eps);
  else
    gemm_skinny_kernel<bf16_t, 1, 1, 2, ALODLM_EPI_STORE, SKINNY_NORM>
        <<<ceil_div_u(N, 16), 64 * WAVES, 0, st>>>(A, lda, W, ldw, C, ldc, nullptr, 0, M, N, K, 1.f,
                                                   nw, eps);
}

}  // namespace

bool gemm_skinny_eligible(const void* A, int64_t lda, int a_kmajor, const void* B, int64_t ldb,
                          int b_kmajor, int64_t M, int64_t N, int64_t K, int epi, int dtype) {
  if (!a_kmajor || !b_kmajor || M < 1 || M > SKINNY_M) return false;
  if (epi != ALODLM_EPI_STORE && epi != ALODLM_EPI_RESIDUAL) return false;
  const int64_t vec = dtype == ALODLM_BF16 ? 8 : 4;  // whole 16-byte chunks
  if (K < vec || K % vec || K > lda || K > ldb || lda % vec || ldb % vec) return false;
  // 32-bit offsets from a workgroup's first row
  const int64_t es = dtype == ALODLM_BF16 ? 2 : 4;
  if (N > (1 << 30) || 32 * ldb * es > (1 << 30) || SKINNY_M * lda * es > (1 << 30)) return false;
  return ((reinterpret_cast<uintptr_t>(A) | reinterpret_cast<uintptr_t>(B)) & 15) == 0;
}

void gemm_skinny_launch(const void* A, int64_t lda, const void* B, int64_t ldb, void* C,
                        int64_t ldc, const void* R, int64_t ldr, int64_t M, int64_t N, int64_t K,
                        float alpha, int epi, int dtype, hipStream_t st) {
  if (dtype == ALODLM_BF16)
    launch_typed<bf16_t>(A, lda, B, ldb, C, ldc, R, ldr, M, N, K, alpha, epi, st);
  else
    launch_typed<float>(A, lda, B, ldb, C, ldc, R, ldr, M, N, K, alpha, epi, st);
}

// C = rmsnorm(x) W^T, or with `swiglu` silu(gate) * up of its two halves, for
// at most 16 bf16 rows; returns ALODLM_EINVAL for anything wider or unaligned.
extern "C" int alodlm_norm_product(const void* x, int64_t ldx, const void* norm_weight, float eps,
                                   const void* W, int64_t ldw, void* C, int64_t ldc, int64_t M,
                                   int64_t N, int64_t K, int swiglu, int dtype, void* stream) {
  ALODLM_CHECK_ARG(dtype == ALODLM_BF16, "norm_product: bf16 only");
  ALODLM_CHECK_ARG(M >= 0 && M <= 16, "norm_product: at most 16 rows");
  if (M == 0 || N == 0) return ALODLM_OK;
  ALODLM_CHECK_ARG(gemm_skinny_eligible(x, ldx, 1, W, ldw, 1, M, N, K, ALODLM_EPI_STORE, dtype) &&
                       reinterpret_cast<uintptr_t>(norm_weight) % 16 == 0 &&
                       N * ldw * 2 < (1LL << 31),
                   "norm_product: rows must be 16-byte aligned and the weight below 2 GiB");
  ALODLM_CHECK_ARG(!swiglu || N % 2 == 0, "norm_product: gate and up rows must pair");
  launch_fused((const bf16_t*)x, ldx, (const bf16_t*)norm_weight, eps, (const bf16_t*)W, ldw,
               (bf16_t*)C, ldc, (int)M, (int)N, (int)K, swiglu, as_stream(stream));
  ALODLM_CHECK_LAUNCH("norm_product");
  return ALODLM_OK;
}
