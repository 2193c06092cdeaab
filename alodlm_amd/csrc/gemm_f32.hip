// float GEMM on the matrix cores:  C[m, n] = alpha * sum_k A(m, k) B(n, k),
// operands k-contiguous or m/n-contiguous in any combination, float sums.
//
// Bound: v_mfma_f32_32x32x2_f32 (157 TFLOP/s dense; an FMA kernel without
// packed float instructions has half of that and spends its issue slots on
// LDS reads: 17 TFLOP/s measured).  128x128 tiles (16-deep k stages) or 64x64
// ones (32-deep), 4 waves of 2 x 2 or one 32x32 block each, double-buffered in
// LDS with the next stage's global loads in registers during the current
// stage's MFMAs (2048 or 1024 cycles), so neither LDS nor memory is near its
// limit: 0.79 of the matrix rate (120 TFLOP/s) is reached on 4096 x 4096 x
// 4096, 0.74 by the small tile.  A few hundred rows make few 128x128 tiles; the
// small tile and K splits even the rounds out (plan, below): 700 rows, 12288 x
// 2048 353 us (424 on the large tile), 4096 x 2048 120 us (133).
//
// LDS: a k-contiguous operand as rows of pitch 20 (36) floats, read 4 k at a
// time (ds_read_b128, free of bank conflicts: multiples of 20 (36) mod 64 are 16
// distinct quads); an m/n-contiguous one as k rows of pitch 136 (72), read one
// k at a time (the two lane halves 4 rows apart fall 32 banks apart).  The MFMA's
// k index is permuted alike for both operands: half h of the lanes takes k =
// 8 b + 4 h + j in step j of block b, which only reorders the sum.
// B's rows are the MFMA's first operand, so a lane owns 4 consecutive columns.
#include "common.h"
#include "gemm_f32.h"

typedef __attribute__((__vector_size__(16 * sizeof(float)))) float f32x16_t;

namespace {

// A tile of TILE x TILE outputs: stage depth and LDS pitches (floats).
template <int TILE> struct Shape {
  static constexpr int BK = TILE == 128 ? 16 : 32, PK = BK + 4, PN = TILE + 8;
  static constexpr int OPF = TILE * PK > BK * PN ? TILE * PK : BK * PN;
};

// One operand's stage: two float4 per thread.
template <bool KMAJ, int TILE> struct Stage {
  static constexpr int BK = Shape<TILE>::BK, PK = Shape<TILE>::PK, PN = Shape<TILE>::PN;
  static constexpr int KQ = BK / 4, RQ = TILE / 4;  // float4 per k-contiguous row / k row
  static_assert(TILE * BK == 4 * 2 * 256, "two float4 per thread");
  float4 v[2];
  __device__ __forceinline__ void load(const float* __restrict__ P, int64_t ld, int64_t r0,
                                       int64_t rows, int64_t k0, int64_t kend) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int c = threadIdx.x + 256 * i;
      const int64_t r = r0 + (KMAJ ? c / KQ : (c % RQ) * 4), k = k0 + (KMAJ ? (c % KQ) * 4 : c / RQ);
      // rows (KMAJ: k) come in whole groups of 4
      v[i] = r < rows && k < kend ? *reinterpret_cast<const float4*>(KMAJ ? P + r * ld + k : P + k * ld + r)
                                  : make_float4(0.f, 0.f, 0.f, 0.f);
    }
  }
  __device__ __forceinline__ void store(float* lds) const {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int c = threadIdx.x + 256 * i;
      *reinterpret_cast<float4*>(KMAJ ? lds + (c / KQ) * PK + (c % KQ) * 4
                                      : lds + (c / RQ) * PN + (c % RQ) * 4) = v[i];
    }
  }
  // the four k of block b for row `row`, this lane half
  static __device__ __forceinline__ float4 frag(const float* lds, int row, int b, int half) {
    if constexpr (KMAJ) return *reinterpret_cast<const float4*>(lds + row * PK + 8 * b + 4 * half);
    const float* p = lds + (8 * b + 4 * half) * PN + row;
    return make_float4(p[0], p[PN], p[2 * PN], p[3 * PN]);
  }
};

template <bool AK, bool BKM, int EPI, int TILE>
__global__ void __launch_bounds__(256, 2)
gemm_f32_kernel(const float* __restrict__ A, int64_t lda, const float* __restrict__ B, int64_t ldb,
                float* C, int64_t ldc, const float* R, int64_t ldr, int64_t M, int64_t N,
                int64_t K, float alpha, int64_t k_per_split, float* __restrict__ partial) {
  constexpr int BK = Shape<TILE>::BK, NB = TILE / 64;  // 32x32 blocks per wave and side
  typedef Stage<AK, TILE> SA;
  typedef Stage<BKM, TILE> SB;
  __shared__ __attribute__((aligned(16))) float lds[2][2][Shape<TILE>::OPF];
  const int64_t tiles_m = (M + TILE - 1) / TILE;
  // tile rows fastest: neighbouring workgroups share B's rows
  const int64_t m0 = (blockIdx.x % tiles_m) * TILE, n0 = (blockIdx.x / tiles_m) * TILE;
  const int64_t kbeg = (int64_t)blockIdx.y * k_per_split;
  const int64_t kend = kbeg + k_per_split < K ? kbeg + k_per_split : K;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int half = lane >> 5, col = lane & 31;
  const int wm = (wave >> 1) * (TILE / 2), wn = (wave & 1) * (TILE / 2);

  f32x16_t acc[NB][NB];
#pragma unroll
  for (int i = 0; i < NB; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;

  SA sa;
  SB sb;
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
      float4 fa[NB], fb[NB];
#pragma unroll
      for (int i = 0; i < NB; ++i) {
        fa[i] = SA::frag(la, wm + 32 * i + col, b, half);
        fb[i] = SB::frag(lb, wn + 32 * i + col, b, half);
      }
#pragma unroll
      for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int i = 0; i < NB; ++i)
#pragma unroll
          for (int j = 0; j < NB; ++j)
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
  for (int i = 0; i < NB; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j)
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

template <bool AK, bool BKM, int TILE>
void launch(const float* A, int64_t lda, const float* B, int64_t ldb, float* C, int64_t ldc,
            const float* R, int64_t ldr, int64_t M, int64_t N, int64_t K, float alpha, int epi,
            int64_t kps, int64_t nsplit, float* part, hipStream_t st) {
  const dim3 grid((unsigned)(((M + TILE - 1) / TILE) * ((N + TILE - 1) / TILE)), (unsigned)nsplit);
  if (epi == ALODLM_EPI_RESIDUAL)
    gemm_f32_kernel<AK, BKM, ALODLM_EPI_RESIDUAL, TILE><<<grid, 256, 0, st>>>(
        A, lda, B, ldb, C, ldc, R, ldr, M, N, K, alpha, kps, part);
  else if (epi == ALODLM_EPI_ACCUM)
    gemm_f32_kernel<AK, BKM, ALODLM_EPI_ACCUM, TILE><<<grid, 256, 0, st>>>(
        A, lda, B, ldb, C, ldc, R, ldr, M, N, K, alpha, kps, part);
  else
    gemm_f32_kernel<AK, BKM, ALODLM_EPI_STORE, TILE><<<grid, 256, 0, st>>>(
        A, lda, B, ldb, C, ldc, R, ldr, M, N, K, alpha, kps, part);
}

template <bool AK, bool BKM>
void launch_tile(const float* A, int64_t lda, const float* B, int64_t ldb, float* C, int64_t ldc,
                 const float* R, int64_t ldr, int64_t M, int64_t N, int64_t K, float alpha,
                 int epi, int64_t kps, int64_t nsplit, float* part, int tile, hipStream_t st) {
  if (tile == 128) launch<AK, BKM, 128>(A, lda, B, ldb, C, ldc, R, ldr, M, N, K, alpha, epi, kps, nsplit, part, st);
  else launch<AK, BKM, 64>(A, lda, B, ldb, C, ldc, R, ldr, M, N, K, alpha, epi, kps, nsplit, part, st);
}

// Tile side and splits of K (each keeping 128 of K) with the least modelled
// time: rounds of 256 workgroups at what a CU reaches of its share of the
// matrix rate (0.6 TFLOP/s: 0.79 large, 0.74 small), and a split's partial sums
// written and read at 5.5 TB/s plus a launch.  Four rounds of tiles and more
// run unsplit: their last one idles a fifth of the time at most, for partial
// sums of several times the output.
struct F32Plan {
  int tile;
  int64_t splits;
};
F32Plan plan(int64_t M, int64_t N, int64_t K, bool workspace) {
  F32Plan best{128, 1};
  double least = 1e30;
  for (int tile = 128; tile >= 64; tile -= 64) {
    const int64_t tiles = ((M + tile - 1) / tile) * ((N + tile - 1) / tile);
    const double each = 2.0 * tile * tile * (double)K / (0.6e6 * (tile == 64 ? 0.74 : 0.79));
    for (int64_t s = 1; s <= 16 && (s == 1 || (workspace && tiles < 1024 && K / s >= 128)); ++s) {
      const int64_t rounds = (tiles * s + 255) / 256;
      const double reduce = s > 1 ? 4.0 + 4e-6 / 5.5 * (double)(2 * s + 1) * (double)M * (double)N : 0.0;
      const double t = (double)rounds * each / (double)s + reduce;
      if (t < least) {
        least = t;
        best = F32Plan{tile, s};
      }
    }
  }
  return best;
}

}  // namespace

bool gemm_f32_eligible(const void* A, int64_t lda, int a_kmajor, const void* B, int64_t ldb,
                       int b_kmajor, int64_t M, int64_t N, int64_t K) {
  if (K < 1 || lda % 4 || ldb % 4) return false;
  if (((reinterpret_cast<uintptr_t>(A) | reinterpret_cast<uintptr_t>(B)) & 15) != 0) return false;
  if ((a_kmajor || b_kmajor) && K % 4) return false;
  return (a_kmajor || M % 4 == 0) && (b_kmajor || N % 4 == 0);
}

int64_t gemm_f32_splits(int64_t M, int64_t N, int64_t K) { return plan(M, N, K, true).splits; }

int64_t gemm_f32_launch(const float* A, int64_t lda, int a_kmajor, const float* B, int64_t ldb,
                        int b_kmajor, float* C, int64_t ldc, const float* R, int64_t ldr,
                        int64_t M, int64_t N, int64_t K, float alpha, int epi, float* workspace,
                        hipStream_t st) {
  const F32Plan p = plan(M, N, K, workspace != nullptr);
  const int64_t kps = ((K + p.splits - 1) / p.splits + 31) / 32 * 32;
  const int64_t nsplit = (K + kps - 1) / kps;
  float* part = nsplit > 1 ? workspace : nullptr;
  if (a_kmajor && b_kmajor) launch_tile<true, true>(A, lda, B, ldb, C, ldc, R, ldr, M, N, K, alpha, epi, kps, nsplit, part, p.tile, st);
  else if (a_kmajor) launch_tile<true, false>(A, lda, B, ldb, C, ldc, R, ldr, M, N, K, alpha, epi, kps, nsplit, part, p.tile, st);
  else if (b_kmajor) launch_tile<false, true>(A, lda, B, ldb, C, ldc, R, ldr, M, N, K, alpha, epi, kps, nsplit, part, p.tile, st);
  else launch_tile<false, false>(A, lda, B, ldb, C, ldc, R, ldr, M, N, K, alpha, epi, kps, nsplit, part, p.tile, st);
  return nsplit;
}
