// Products of a few rows with a weight matrix (the decoder's windows):
//   C[m, n] = alpha * sum_k A[m, k] W[n, k],  M <= SKINNY_M, both k-contiguous,
// bf16 or float, plain or added to a residual.
//
// Bound: the weights, read once.  A 128x128 tile kernel leaves such a product
// on N / 128 workgroups, each a serial walk over K.  Here a workgroup owns 16
// (or 64) weight rows and its 8 waves split K between them, so that N / 16
// workgroups keep 8 waves of loads in flight and no wave walks more than K / 8;
// each wave's sums meet in LDS once and are added in wave order.  The rows of A
// are re-read per workgroup from L2.
//
// Each wave brings its own 128-byte row pieces into its own LDS ring by direct
// loads (no barrier: a wave waits for its loads only) and reads its fragments
// there.  Loading fragments straight into registers makes every 16 lanes of a
// load touch 16 lines, which a CU's address path serves at about 30 KB/us; 8
// consecutive lanes per line reach 58.  16 rows, bf16, direct to registers and
// now: 4096 x 2048 6.3 and 5.9 us, 2048 x 2048 5.8 and 4.8, 2048 x 6144 12.8 and
// 7.6, 12288 x 2048 14.3 and 12.1; float 2048 x 6144 24.3 and 17.5, 48 rows of
// 4096 x 12288 101 and 65.
//
// Fragment: lane l holds 16 bytes of row l % 16 at 16-byte chunk l / 16.  For
// float the four k of a lane's chunk feed four 16x16x4 MFMAs (both operands
// permute k alike, which only reorders the sum).
#include "common.h"
#include "gemm_skinny.h"
#include "lds_dma.h"

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

// MT: 16-row blocks of A; NT: 16-row blocks of W per workgroup; H: fragments
// (64 bytes of a row) per stage; S: stages of a wave's ring.
template <typename T, int MT, int NT, int H, int S, int EPI, int FUSE = 0>
__global__ void __launch_bounds__(64 * WAVES, 2)
gemm_skinny_kernel(const T* __restrict__ A, int64_t lda, const T* __restrict__ W, int64_t ldw,
                   T* C, int64_t ldc, const T* R, int64_t ldr, int M, int N, int K, float alpha,
                   const T* __restrict__ nw, float eps) {
  typedef SkinnyType<T> F;
  constexpr int STEP = 2 * F::KS;  // k a wave takes at a time: 128 bytes of a row
  constexpr int COLS = 16 * NT, ROWS = 16 * MT;
  constexpr bool NORM = FUSE & SKINNY_NORM, GLU = FUSE & SKINNY_GLU;
  static_assert(!GLU || NT == 2, "one gate block and one up block");
  constexpr uint32_t ES = sizeof(T), OUT = 0xffffff00u;
  // a stage: W's blocks, A's blocks, the norm weight
  constexpr uint32_t BLOCK = 1024 * H, STAGE = (NT + MT) * BLOCK + (NORM ? 256 : 0);
  constexpr uint32_t REGION = S * STAGE;  // of a wave
  constexpr int PER = (NT + MT) * H + (NORM ? 1 : 0);  // loads per stage
  static_assert(REGION >= ROWS * COLS * 4, "the sums reuse the ring");
  __shared__ __attribute__((aligned(1024))) char lds[WAVES * REGION];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int i = lane & 15, q = lane >> 4;
  const int n0 = blockIdx.x * (GLU ? 16 : COLS);
  const int cols = GLU ? N / 2 : N;  // of the output
  // Operands as buffers based at the workgroup's rows, with 32-bit lane
  // offsets; a chunk past K reads at an offset the range check turns into zeros.
  const int64_t nrows = GLU ? N - n0 : N - n0 < COLS ? N - n0 : COLS;
  const v4i_t wr = buffer_of(W + (int64_t)n0 * ldw, ((nrows - 1) * ldw + K) * ES);
  const v4i_t xr = buffer_of(A, ((M - 1) * lda + K) * ES);
  const v4i_t nr = buffer_of(NORM ? nw : A, K * ES);
  // Load j of a block: row j 16/H + lane / 4H, chunk lane % 4H of its 64 H bytes,
  // stored at slot `lane`; chunks of a row are permuted by the row so that the
  // 16 rows a fragment read touches fall into different banks.
  auto swizzle = [](int r) { return H == 2 ? (r >> 1) & 7 : (r >> 1) & 3; };
  uint32_t wo[NT][H], xo[MT][H];
  int kc[H];
#pragma unroll
  for (int j = 0; j < H; ++j) {
    const int r = j * (16 / H) + lane / (4 * H), c = (lane % (4 * H)) ^ swizzle(r);
    kc[j] = c * F::VEC;
#pragma unroll
    for (int b = 0; b < NT; ++b) {  // rows past the edge re-read the last one (never stored)
      const int64_t row = GLU ? (int64_t)b * cols + (n0 + r < cols ? r : cols - 1 - n0)
                              : 16 * b + r < nrows ? 16 * b + r : nrows - 1;
      wo[b][j] = (uint32_t)((row * ldw + kc[j]) * ES);
    }
#pragma unroll
    for (int a = 0; a < MT; ++a) {
      const int m = 16 * a + r;
      xo[a][j] = (uint32_t)(((int64_t)(m < M ? m : M - 1) * lda + kc[j]) * ES);
    }
  }
  const uint32_t ring = lds_addr(lds) + (uint32_t)wave * REGION;
  int k = wave * STEP;  // of the next stage to load
  const int stages = k < K ? ((K - k - 1) / (WAVES * STEP) + 1) * (2 / H) : 0;
  int half = 0;
  auto load = [&](int slot) {
    const uint32_t at = ring + (uint32_t)slot * STAGE;
    const int kk = k + half * F::KS;
#pragma unroll
    for (int j = 0; j < H; ++j) {
      const bool in = kk + kc[j] + F::VEC <= K;
#pragma unroll
      for (int b = 0; b < NT; ++b)
        dma16_buf(wr, in ? wo[b][j] + kk * ES : OUT, at + b * BLOCK + j * 1024);
#pragma unroll
      for (int a = 0; a < MT; ++a)
        dma16_buf(xr, in ? xo[a][j] + kk * ES : OUT, at + (NT + a) * BLOCK + j * 1024);
    }
    if constexpr (NORM) {  // 4 bytes a lane, the stage's k in the first 16 H lanes
      const int kn = kk + 2 * lane;
      dma4_buf(nr, lane < 16 * H && kn + 2 <= K ? kn * ES : OUT, at + (NT + MT) * BLOCK);
    }
    if (H == 2 || half) k += WAVES * STEP;
    if (H == 1) half ^= 1;
  };
#pragma unroll
  for (int s = 0; s < S - 1; ++s) load(s);

  // 1 / rms of the rows (every workgroup for itself: 16 rows of 2048 are 64 KB
  // from L2, less than a launch of its own costs), under the first loads
  float rs[MT];
  if constexpr (NORM) {
    __shared__ float inv_rms[ROWS];
    for (int m = wave; m < M; m += WAVES) {
      float sum = 0.f;
      for (int c = lane * 8; c < K; c += 512) {  // the RMSNorm kernels' order: the same bits
        float v[8];
        Vec8<T>::load(A + (int64_t)m * lda + c, v);
#pragma unroll
        for (int e = 0; e < 8; ++e) sum = fmaf(v[e], v[e], sum);
      }
      sum = wave_sum(sum);
      if (lane == 0) inv_rms[m] = 1.0f / sqrtf(sum / (float)K + eps);
    }
    __syncthreads();
#pragma unroll
    for (int a = 0; a < MT; ++a) rs[a] = inv_rms[16 * a + i < M ? 16 * a + i : M - 1];
  }

  f32x4_t acc[MT][NT];
#pragma unroll
  for (int a = 0; a < MT; ++a)
#pragma unroll
    for (int b = 0; b < NT; ++b) acc[a][b] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  char* own = lds + wave * REGION;
  int cur = 0;
  for (int t = 0; t < stages; ++t) {
    // stage t has landed once at most the S - 2 newer ones are in flight; the
    // slot filled next was read in the step before
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_waitcnt vmcnt(%0)" ::"n"((S - 2) * PER) : "memory");
    load(cur == 0 ? S - 1 : cur - 1);
    const char* st = own + cur * STAGE;
    cur = cur + 1 < S ? cur + 1 : 0;
#pragma unroll
    for (int h = 0; h < H; ++h) {
      const uint32_t at = i * 64 * H + (((4 * h + q) ^ swizzle(i)) << 4);
      uint4 w[NT];
#pragma unroll
      for (int b = 0; b < NT; ++b) w[b] = *reinterpret_cast<const uint4*>(st + b * BLOCK + at);
#pragma unroll
      for (int a = 0; a < MT; ++a) {
        uint4 xa = *reinterpret_cast<const uint4*>(st + (NT + a) * BLOCK + at);
        if constexpr (NORM)
          xa = normed(xa, *reinterpret_cast<const uint4*>(st + (NT + MT) * BLOCK + (4 * h + q) * 16),
                      rs[a]);
#pragma unroll
        for (int b = 0; b < NT; ++b) acc[a][b] = F::mma(w[b], xa, acc[a][b]);
      }
    }
  }

  // the ring is free once its last loads have landed; its bytes hold the sums.
  // lane: row lane % 16, columns 4 (lane / 16) .. +3 of each 16x16 block
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_waitcnt vmcnt(0)" ::: "memory");
#pragma unroll
  for (int a = 0; a < MT; ++a)
#pragma unroll
    for (int b = 0; b < NT; ++b)
      *reinterpret_cast<f32x4_t*>(own + ((16 * a + i) * COLS + 16 * b + 4 * q) * 4) = acc[a][b];
  __syncthreads();
  auto part = [&](int s, int m, int c) {
    return *reinterpret_cast<const float*>(lds + s * REGION + (m * COLS + c) * 4);
  };
  constexpr int OUTS = GLU ? 16 : COLS;
  for (int t = threadIdx.x; t < ROWS * OUTS; t += 64 * WAVES) {
    const int m = t / OUTS, c = t % OUTS, n = n0 + c;
    if (m >= M || n >= cols) continue;
    float v = 0.f;
#pragma unroll
    for (int s = 0; s < WAVES; ++s) v += part(s, m, c);
    v *= alpha;
    if constexpr (GLU) {
      float up = 0.f;
#pragma unroll
      for (int s = 0; s < WAVES; ++s) up += part(s, m, 16 + c);
      const float g = Elem<T>::round(v);
      v = Elem<T>::round(g / (1.0f + expf(-g))) * Elem<T>::round(alpha * up);
    }
    if (EPI == ALODLM_EPI_RESIDUAL) v = Elem<T>::load(R, m * ldr + n) + Elem<T>::round(v);
    Elem<T>::store(C, m * ldc + n, v);
  }
}

template <typename T, int MT, int NT, int H, int S>
void launch(const T* A, int64_t lda, const T* W, int64_t ldw, T* C, int64_t ldc, const T* R,
            int64_t ldr, int M, int N, int K, float alpha, int epi, hipStream_t st) {
  const unsigned grid = ceil_div_u(N, 16 * NT);
  if (epi == ALODLM_EPI_STORE)
    gemm_skinny_kernel<T, MT, NT, H, S, ALODLM_EPI_STORE><<<grid, 64 * WAVES, 0, st>>>(
        A, lda, W, ldw, C, ldc, R, ldr, M, N, K, alpha, nullptr, 0.f);
  else
    gemm_skinny_kernel<T, MT, NT, H, S, ALODLM_EPI_RESIDUAL><<<grid, 64 * WAVES, 0, st>>>(
        A, lda, W, ldw, C, ldc, R, ldr, M, N, K, alpha, nullptr, 0.f);
}

// Weight rows per workgroup and ring depth.  128-byte pieces (H = 2) throughout:
// with 64-byte ones the loads touch twice the lines (16 rows, 2048 x 6144: 9.7
// us against 7.5; 48 float rows, 4096 x 12288: 92 against 65).  Outputs of at
// most one 16-row workgroup per CU take the deepest ring; wider ones two
// workgroups per CU (16 rows, 24576 x 4096: 40 us against 44; 6144 x 4096: 12.8
// against 14.1).  One block of rows against 64-row workgroups re-reads A less
// and starts fewer rings, which pays for short rows (below 8 KB), in one round
// of such workgroups or in many (12288 x 2048: 12.1 us against 16.8; float 21.1
// against 25.4; 151936 x 2048: 129 against 142; but 24576 x 4096, one and a half
// rounds: 45 against 40).  Two blocks and more want 16 weight rows everywhere (27
// rows, 24576 x 4096: 51 us against 57).  Timed over eight copies of the weight in
// turn: the smaller shapes' copies stay in the 256 MB last-level cache.
template <typename T>
void launch_typed(const T* A, int64_t lda, const T* W, int64_t ldw, T* C, int64_t ldc, const T* R,
                  int64_t ldr, int M, int N, int K, float alpha, int epi, hipStream_t st) {
  const bool wide = N > 16 * 256;
  const bool rows64 = N >= 64 * 192 && (N <= 64 * 256 || N >= 64 * 1024 || K * (int)sizeof(T) < 8192);
  if (M > 48) launch<T, 4, 1, 2, 2>(A, lda, W, ldw, C, ldc, R, ldr, M, N, K, alpha, epi, st);
  else if (M > 32) launch<T, 3, 1, 2, 2>(A, lda, W, ldw, C, ldc, R, ldr, M, N, K, alpha, epi, st);
  else if (M > 16) launch<T, 2, 1, 2, 3>(A, lda, W, ldw, C, ldc, R, ldr, M, N, K, alpha, epi, st);
  else if (rows64) launch<T, 1, 4, 2, 2>(A, lda, W, ldw, C, ldc, R, ldr, M, N, K, alpha, epi, st);
  else if (wide) launch<T, 1, 1, 2, 2>(A, lda, W, ldw, C, ldc, R, ldr, M, N, K, alpha, epi, st);
  else launch<T, 1, 1, 2, 4>(A, lda, W, ldw, C, ldc, R, ldr, M, N, K, alpha, epi, st);
}

// 16 rows after 300 cached ones at the 1.7B shapes, a whole decoder layer call:
// 92 us with the norms, the products, SwiGLU and the value copy in launches of
// their own, 66 us with both norms and SwiGLU in the products and the values
// copied by the rotary kernel (57 with the LDS rings).  float rows lose (154 us
// to 169): their norm re-reads twice the bytes.  With SwiGLU a ring of 64-byte
// pieces leaves room for two workgroups per CU, which hide each other's norm.
void launch_fused(const bf16_t* A, int64_t lda, const bf16_t* nw, float eps, const bf16_t* W,
                  int64_t ldw, bf16_t* C, int64_t ldc, int M, int N, int K, bool glu,
                  hipStream_t st) {
  if (glu)
    gemm_skinny_kernel<bf16_t, 1, 2, 1, 3, ALODLM_EPI_STORE, SKINNY_NORM | SKINNY_GLU>
        <<<ceil_div_u(N / 2, 16), 64 * WAVES, 0, st>>>(A, lda, W, ldw, C, ldc, nullptr, 0, M, N, K,
                                                       1.f, nw, eps);
  else
    gemm_skinny_kernel<bf16_t, 1, 1, 2, 4, ALODLM_EPI_STORE, SKINNY_NORM>
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
  if (N > (1 << 30) || 64 * ldb * es > (1 << 30) || SKINNY_M * lda * es > (1 << 30)) return false;
  return ((reinterpret_cast<uintptr_t>(A) | reinterpret_cast<uintptr_t>(B)) & 15) == 0;
}

void gemm_skinny_launch(const void* A, int64_t lda, const void* B, int64_t ldb, void* C,
                        int64_t ldc, const void* R, int64_t ldr, int64_t M, int64_t N, int64_t K,
                        float alpha, int epi, int dtype, hipStream_t st) {
  if (dtype == ALODLM_BF16)
    launch_typed((const bf16_t*)A, lda, (const bf16_t*)B, ldb, (bf16_t*)C, ldc, (const bf16_t*)R,
                 ldr, (int)M, (int)N, (int)K, alpha, epi, st);
  else
    launch_typed((const float*)A, lda, (const float*)B, ldb, (float*)C, ldc, (const float*)R, ldr,
                 (int)M, (int)N, (int)K, alpha, epi, st);
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
