// float GEMM on the matrix cores:  C[m, n] = alpha * sum_k A(m, k) B(n, k),
// operands k-contiguous or m/n-contiguous in any combination, float sums.
//
// Bound: v_mfma_f32_32x32x2_f32 (157 TFLOP/s dense; an FMA kernel without
// packed float instructions has half of that and spends its issue slots on
// LDS reads: 17 TFLOP/s measured).  128x128 tiles, 4 waves of 64x64 (2 x 2
// blocks of 32x32), 16-deep k stages double-buffered in LDS with the next
// stage's global loads in registers during the 32 MFMAs (2048 cycles) of the
// current one, so neither LDS nor memory is near its limit.
//
// LDS: a k-contiguous operand as [128 rows][16 k] of pitch 20 floats, read 4 k
// at a time (ds_read_b128, free of bank conflicts: 20 i mod 64 are 16 distinct
// quads); an m/n-contiguous one as [16 k][128] of pitch 136, read one k at a
// time (the two lane halves 4 rows apart fall 32 banks apart).  The MFMA's
// k index is permuted alike for both operands: half h of the lanes takes k =
// 8 b + 4 h + j in step j of block b, which only reorders the sum.
// B's rows are the MFMA's first operand, so a lane owns 4 consecutive columns.
#include "common.h"
#include "gemm_f32.h"

typedef __attribute__((__vector_size__(16 * sizeof(float)))) float f32x16_t;

namespace {

constexpr int BM = 128, BK = 16;
constexpr int PK = BK + 4, PN = BM + 8;          // LDS pitches (floats)
constexpr int OPF = BM * PK > BK * PN ? BM * PK : BK * PN;

// One operand's stage: two float4 per thread.
template <bool KMAJ> struct Stage {
  float4 v[2];
  __device__ __forceinline__ void load(const float* __restrict__ P, int64_t ld, int64_t r0,
                                       int64_t rows, int64_t k0, int64_t kend) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int c = threadIdx.x + 256 * i;
      const int64_t r = r0 + (KMAJ ? c >> 2 : (c & 31) * 4), k = k0 + (KMAJ ? (c & 3) * 4 : c >> 5);
      // rows (KMAJ: k) come in whole groups of 4
      v[i] = r < rows && k < kend ? *reinterpret_cast<const float4*>(KMAJ ? P + r * ld + k : P + k * ld + r)
                                  : make_float4(0.f, 0.f, 0.f, 0.f);
    }
  }
  __device__ __forceinline__ void store(float* lds) const {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int c = threadIdx.x + 256 * i;
      *reinterpret_cast<float4*>(KMAJ ? lds + (c >> 2) * PK + (c & 3) * 4
                                      : lds + (c >> 5) * PN + (c & 31) * 4) = v[i];
    }
  }
  // the four k of block b for row `row`, this lane half
  static __device__ __forceinline__ float4 frag(const float* lds, int row, int b, int half) {
    if constexpr (KMAJ) return *reinterpret_cast<const float4*>(lds + row * PK + 8 * b + 4 * half);
    const float* p = lds + (8 * b + 4 * half) * PN + row;
    return make_float4(p[0], p[PN], p[2 * PN], p[3 * PN]);
  }
};

template <bool AK, bool BKM, int EPI>
__global__ void __launch_bounds__(256, 2)
gemm_f32_kernel(const float* __restrict__ A, int64_t lda, const float* __restrict__ B, int64_t ldb,
                float* C, int64_t ldc, const float* R, int64_t ldr, int64_t M, int64_t N,
                int64_t K, float alpha, int64_t k_per_split, float* __restrict__ partial) {
  __shared__ __attribute__((aligned(16))) float lds[2][2][OPF];
  const int64_t tiles_m = (M + BM - 1) / BM;
  // tile rows fastest: neighbouring workgroups share B's rows
  const int64_t m0 = (blockIdx.x % tiles_m) * BM, n0 = (blockIdx.x / tiles_m) * BM;
  const int64_t kbeg = (int64_t)blockIdx.y * k_per_split;
  const int64_t kend = kbeg + k_per_split < K ? kbeg + k_per_split : K;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int half = lane >> 5, col = lane & 31, wm = (wave >> 1) * 64, wn = (wave & 1) * 64;

  f32x16_t acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;

  Stage<AK> sa;
  Stage<BKM> sb;
  if (kbeg < kend) {
    sa.load(A, lda, m0, M, kbeg, kend);
    sb.load(B, ldb, n0, N, kbeg, kend);
    sa.store(lds[0][0]);
    sb.store(lds[0][1]);
  }
  __syncthreads();
  int buf = 0;
  for (int64_t k0 = kbeg; k0 < kend; k0 += BK) {
    const bool more = k0 + BK < kend;
    if (more) {
      sa.load(A, lda, m0, M, k0 + BK, kend);
      sb.load(B, ldb, n0, N, k0 + BK, kend);
    }
    const float *la = lds[buf][0], *lb = lds[buf][1];
#pragma unroll
    for (int b = 0; b < BK / 8; ++b) {
      float4 fa[2], fb[2];
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        fa[i] = Stage<AK>::frag(la, wm + 32 * i + col, b, half);
        fb[i] = Stage<BKM>::frag(lb, wn + 32 * i + col, b, half);
      }
#pragma unroll
      for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int j = 0; j < 2; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32((&fb[j].x)[s], (&fa[i].x)[s],
                                                             acc[i][j], 0, 0, 0);
    }
    if (more) {
      sa.store(lds[buf ^ 1][0]);
      sb.store(lds[buf ^ 1][1]);
    }
    __syncthreads();
    buf ^= 1;
  }

  // lane: row lane % 32, columns 8 q + 4 half .. +3 of each 32x32 block
  float* P = partial ? partial + (int64_t)blockIdx.y * M * N : nullptr;
  const int64_t ldo = P ? N : ldc;
  float* out = P ? P : C;
  const bool vec = ldo % 4 == 0 && reinterpret_cast<uintptr_t>(out) % 16 == 0 &&
                   (EPI != ALODLM_EPI_RESIDUAL || P ||
                    (ldr % 4 == 0 && reinterpret_cast<uintptr_t>(R) % 16 == 0));
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int64_t m = m0 + wm + 32 * i + col, n = n0 + wn + 32 * j + 8 * q + 4 * half;
        if (m >= M) continue;
        float v[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = alpha * acc[i][j][4 * q + e];
        float* dst = out + m * ldo + n;
        if (vec && n + 4 <= N) {
          if (!P && EPI != ALODLM_EPI_STORE) {
            const float4 r = *reinterpret_cast<const float4*>(
                EPI == ALODLM_EPI_RESIDUAL ? R + m * ldr + n : (const float*)dst);
            v[0] += r.x; v[1] += r.y; v[2] += r.z; v[3] += r.w;
          }
          *reinterpret_cast<float4*>(dst) = make_float4(v[0], v[1], v[2], v[3]);
          continue;
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          if (n + e >= N) continue;
          if (!P && EPI == ALODLM_EPI_RESIDUAL) v[e] += R[m * ldr + n + e];
          if (!P && EPI == ALODLM_EPI_ACCUM) v[e] += dst[e];
          dst[e] = v[e];
        }
      }
}

template <bool AK, bool BKM>
void launch(const float* A, int64_t lda, const float* B, int64_t ldb, float* C, int64_t ldc,
            const float* R, int64_t ldr, int64_t M, int64_t N, int64_t K, float alpha, int epi,
            int64_t kps, int64_t nsplit, float* part, hipStream_t st) {
  const dim3 grid((unsigned)(((M + BM - 1) / BM) * ((N + BM - 1) / BM)), (unsigned)nsplit);
  if (epi == ALODLM_EPI_RESIDUAL)
    gemm_f32_kernel<AK, BKM, ALODLM_EPI_RESIDUAL><<<grid, 256, 0, st>>>(
        A, lda, B, ldb, C, ldc, R, ldr, M, N, K, alpha, kps, part);
  else if (epi == ALODLM_EPI_ACCUM)
    gemm_f32_kernel<AK, BKM, ALODLM_EPI_ACCUM><<<grid, 256, 0, st>>>(
        A, lda, B, ldb, C, ldc, R, ldr, M, N, K, alpha, kps, part);
  else
    gemm_f32_kernel<AK, BKM, ALODLM_EPI_STORE><<<grid, 256, 0, st>>>(
        A, lda, B, ldb, C, ldc, R, ldr, M, N, K, alpha, kps, part);
}

}  // namespace

bool gemm_f32_eligible(const void* A, int64_t lda, int a_kmajor, const void* B, int64_t ldb,
                       int b_kmajor, int64_t M, int64_t N, int64_t K) {
  if (K < 1 || lda % 4 || ldb % 4) return false;
  if (((reinterpret_cast<uintptr_t>(A) | reinterpret_cast<uintptr_t>(B)) & 15) != 0) return false;
  if ((a_kmajor || b_kmajor) && K % 4) return false;
  return (a_kmajor || M % 4 == 0) && (b_kmajor || N % 4 == 0);
}

// The fewest splits of K (powers of two, each keeping 128 of K) whose rounds of
// 256 workgroups cost the least per unit of work; a product of two rounds and
// more runs unsplit.
int64_t gemm_f32_splits(int64_t M, int64_t N, int64_t K) {
  const int64_t tiles = ((M + BM - 1) / BM) * ((N + BM - 1) / BM), cus = 256;
  if (tiles >= 2 * cus) return 1;
  auto cost = [&](int64_t s) { return (double)((tiles * s + cus - 1) / cus) / (double)s; };
  int64_t best = 1;
  for (int64_t s = 2; s <= 32 && K / s >= 128; s *= 2)
    if (cost(s) < 0.9 * cost(best)) best = s;
  return best;
}

int64_t gemm_f32_launch(const float* A, int64_t lda, int a_kmajor, const float* B, int64_t ldb,
                        int b_kmajor, float* C, int64_t ldc, const float* R, int64_t ldr,
                        int64_t M, int64_t N, int64_t K, float alpha, int epi, float* workspace,
                        hipStream_t st) {
  const int64_t splits = workspace ? gemm_f32_splits(M, N, K) : 1;
  const int64_t kps = ((K + splits - 1) / splits + BK - 1) / BK * BK;
  const int64_t nsplit = (K + kps - 1) / kps;
  float* part = nsplit > 1 ? workspace : nullptr;
  if (a_kmajor && b_kmajor) launch<true, true>(A, lda, B, ldb, C, ldc, R, ldr, M, N, K, alpha, epi, kps, nsplit, part, st);
  else if (a_kmajor) launch<true, false>(A, lda, B, ldb, C, ldc, R, ldr, M, N, K, alpha, epi, kps, nsplit, part, st);
  else if (b_kmajor) launch<false, true>(A, lda, B, ldb, C, ldc, R, ldr, M, N, K, alpha, epi, kps, nsplit, part, st);
  else launch<false, false>(A, lda, B, ldb, C, ldc, R, ldr, M, N, K, alpha, epi, kps, nsplit, part, st);
  return nsplit;
}
