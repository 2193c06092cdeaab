// bf16 GEMM for the products whose output is too small for the 256x256 kernel
// to fill the chip, and for weight gradients over a row count that is no
// multiple of 32:  C[m, n] = alpha * sum_k A(m, k) B(n, k).
//
// 128x128 block tile (32x128 or 64x128 for as few rows), 4 waves (2 x 2) of
// 16x16x32 MFMAs, 32-deep k stages in a ring of LDS buffers (at most 72 KB: two
// workgroups per CU, each covering the other's barriers and LDS latency) filled
// by direct buffer loads to LDS.  K is split over grid.y where the tiles are
// few.  Bound: L2 to LDS.  A 128x128 tile moves 16 KB per 32 k; the chip runs
// such a step in 0.275 us per workgroup and CU (15 TB/s, 0.95 PFLOP/s) with one
// or two workgroups on a CU, which is what the dispatch's cost rule uses; the
// 256x256 kernel (0.77 us per step of four times the work) is faster where its
// tiles fill the chip.
// Reads past the last k row return zeros through the buffer's range check, so
// m/n-contiguous operands take any K; rows and columns past the edge re-read
// the last valid ones (they feed outputs that are never stored).
//
// LDS layouts as in gemm_dl.hip, for 128 rows or columns: a k-contiguous
// operand as 64-byte rows with chunk ^ ((row / 2) % 4), read by ds_read_b128;
// an m/n-contiguous one as 256-byte k rows with chunk ^ (4 (k % 4) ^
// 2 ((k / 8) % 2)), read transposed by ds_read_b64_tr_b16.
#include "common.h"
#include "gemm_mid.h"
#include "lds_dma.h"

typedef __attribute__((__vector_size__(8 * sizeof(short)))) short bf16x8_t;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float f32x4_t;
typedef short v4s_t __attribute__((ext_vector_type(4)));
#define LDS_AS __attribute__((address_space(3)))

namespace {

constexpr int TN = 128, KD = 32, NW = 4;

// One operand: this wave's lane offsets into the buffer, the byte step from one
// k stage to the next, and the lane's fragment offsets within a stage.
// ROWS of the tile (128, or for a k-contiguous A 64 or 32).
template <bool KMAJ, int ROWS> struct Opnd {
  static_assert(KMAJ || ROWS == 128, "the transposed layout is for 128 columns");
  static constexpr int OPB = ROWS * KD * 2, SLOTS = OPB / 1024;  // bytes, 1 KB slots per stage
  // direct loads per wave and stage (two slots: two waves load each, the same bytes)
  static constexpr int PER = SLOTS < NW ? 1 : SLOTS / NW;
  uint32_t off[PER], slot[PER], step, fo[KMAJ ? 1 : 4];
  static __device__ __forceinline__ int swz(int x) {
    return KMAJ ? (x >> 1) & 3 : 4 * (x & 3) ^ 2 * ((x >> 3) & 1);
  }
  // rows (columns) r0 .. of an operand with `count` of them
  __device__ __forceinline__ void init(int64_t ld, int64_t r0, int64_t count, int wave, int lane) {
    step = (uint32_t)(KMAJ ? 2 * KD : 2 * KD * ld);
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int j = (wave + NW * i) % SLOTS;
      slot[i] = (uint32_t)j * 1024u;
      if (KMAJ) {
        const int r = 16 * j + (lane >> 2), c = (lane & 3) ^ swz(r);
        const int64_t rr = r0 + r < count ? r0 + r : count - 1;
        off[i] = (uint32_t)((rr * ld + 8 * c) * 2);
      } else {
        const int k = 4 * j + (lane >> 4), c = (lane & 15) ^ swz(k);
        const int64_t cc = r0 + 8 * c < count ? r0 + 8 * c : count - 8;
        off[i] = (uint32_t)((k * ld + cc) * 2);
      }
    }
  }
  // fragments of rows (columns) w0 + 16 idx + lane % 16 of the tile, k = 8
  // (lane / 16) + 0..7; w0 is the wave's first row (column)
  __device__ __forceinline__ void init_frag(int w0, int lane) {
    if constexpr (KMAJ) {
      const int row = w0 + (lane & 15);
      fo[0] = (uint32_t)(row * 64 + (((lane >> 4) ^ swz(row)) << 4));
    } else {
      const int s = lane & 15, k = 8 * (lane >> 4) + (s >> 2);
#pragma unroll
      for (int idx = 0; idx < 4; ++idx) {
        const int c = (w0 >> 3) + 2 * idx + ((s & 3) >> 1);
        fo[idx] = (uint32_t)(k * 256 + ((c ^ swz(k)) << 4) + (s & 1) * 8);
      }
    }
  }
  __device__ __forceinline__ bf16x8_t frag(const char* stage, int idx) const {
    if constexpr (KMAJ) {
      return *reinterpret_cast<const bf16x8_t*>(stage + fo[0] + idx * 16 * 64);
    } else {
      const char* p = stage + fo[idx];
      const v4s_t a = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LDS_AS v4s_t*)p);
      const v4s_t b = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LDS_AS v4s_t*)(p + 4 * 256));
      return __builtin_bit_cast(bf16x8_t, __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7));
    }
  }
};

// MB: 16-row blocks per wave (the tile has 32 MB rows).
template <bool AK, bool BKM, int EPI, int MB, int STAGES>
__global__ void __launch_bounds__(256, 2)
gemm_mid_kernel(const bf16_t* __restrict__ A, int64_t lda, const bf16_t* __restrict__ B,
                int64_t ldb, void* C, int64_t ldc, const bf16_t* R, int64_t ldr, int64_t M,
                int64_t N, int64_t K, float alpha, int64_t k_per_split,
                float* __restrict__ partial) {
  constexpr int TM = 32 * MB;
  typedef Opnd<AK, TM> OA;
  typedef Opnd<BKM, TN> OB;
  __shared__ __attribute__((aligned(1024))) char lds[STAGES * (OA::OPB + OB::OPB)];
  const int tiles_m = (int)((M + TM - 1) / TM), tiles_n = (int)((N + TN - 1) / TN);
  const int T = tiles_m * tiles_n;
  int t = blockIdx.x;
  if (T % 8 == 0) t = (t % 8) * (T / 8) + t / 8;  // contiguous tile chunk per XCD
  const int group = 8, per_group = group * tiles_n;
  const int g = t / per_group, first_m = g * group;
  const int gsize = (tiles_m - first_m) < group ? (tiles_m - first_m) : group;
  const int tm = first_m + (t % per_group) % gsize, tn = (t % per_group) / gsize;
  const int64_t m0 = __builtin_amdgcn_readfirstlane(tm * TM);
  const int64_t n0 = __builtin_amdgcn_readfirstlane(tn * TN);
  const int64_t kbeg = (int64_t)blockIdx.y * k_per_split;
  const int64_t kend = (kbeg + k_per_split) < K ? (kbeg + k_per_split) : K;
  const int ntiles = (int)((kend - kbeg + KD - 1) / KD);

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = (wave >> 1) * 16 * MB, wn = (wave & 1) * 64;

  OA oa;
  OB ob;
  oa.init(lda, m0, M, wave, lane);
  ob.init(ldb, n0, N, wave, lane);
  oa.init_frag(wm, lane);
  ob.init_frag(wn, lane);
  // the operands end with their last k row's (last row's) elements
  const v4i_t ra = buffer_of(A, 2 * (AK ? (M - 1) * lda + K : (K - 1) * lda + M));
  const v4i_t rb = buffer_of(B, 2 * (BKM ? (N - 1) * ldb + K : (K - 1) * ldb + N));
  uint32_t sa = (uint32_t)(kbeg / KD) * oa.step, sb = (uint32_t)(kbeg / KD) * ob.step;

  f32x4_t acc[MB][4];
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};

  // a stage: A's rows, then B's
  constexpr int STAGE = OA::OPB + OB::OPB, PL = OA::PER + OB::PER;
  const uint32_t l0 = lds_addr(lds);
  int tl = 0;  // the next tile to load; past the last one it is loaded again
  auto load = [&](int stage) {
    const uint32_t ls = l0 + (uint32_t)(stage * STAGE);
#pragma unroll
    for (int i = 0; i < OA::PER; ++i) dma16_buf(ra, oa.off[i], sa, ls + oa.slot[i]);
#pragma unroll
    for (int i = 0; i < OB::PER; ++i) dma16_buf(rb, ob.off[i], sb, ls + OA::OPB + ob.slot[i]);
    if (++tl < ntiles) {
      sa += oa.step;
      sb += ob.step;
    }
  };
#pragma unroll
  for (int s = 0; s < STAGES - 1; ++s) load(s);
  int cur = 0;
  for (int tt = 0; tt < ntiles; ++tt) {
    // tile tt's loads are done once at most the STAGES - 2 newest tiles' are in
    // flight; every wave has read tile tt-1, whose stage is filled next
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_waitcnt vmcnt(%0)\n\ts_barrier"
                 :: "n"((STAGES - 2) * PL) : "memory");
    load(cur == 0 ? STAGES - 1 : cur - 1);
    const char* pa = lds + cur * STAGE;
    const char* pb = pa + OA::OPB;
    cur = cur + 1 < STAGES ? cur + 1 : 0;
    bf16x8_t fa[MB], fb[4];
#pragma unroll
    for (int i = 0; i < MB; ++i) fa[i] = oa.frag(pa, i);
#pragma unroll
    for (int j = 0; j < 4; ++j) fb[j] = ob.frag(pb, j);
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int i = 0; i < MB; ++i)
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fb[j], fa[i], acc[i][j], 0, 0, 0);
  }
  // no load may land in LDS after the workgroup has gone
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");

  // lane: output row 16 i + lane % 16, columns 16 j + 4 (lane / 16) .. +3
  bf16_t* Cb = reinterpret_cast<bf16_t*>(C);
  float* Cf = partial ? partial + (int64_t)blockIdx.y * M * N : reinterpret_cast<float*>(C);
  const int64_t ldf = partial ? N : ldc;
  constexpr bool HALF = EPI == ALODLM_EPI_STORE || EPI == ALODLM_EPI_RESIDUAL;
  const bool fout = !HALF || partial != nullptr;
  const bool vec = fout ? ldf % 4 == 0 && reinterpret_cast<uintptr_t>(Cf) % 16 == 0
                        : ldc % 4 == 0 && reinterpret_cast<uintptr_t>(C) % 8 == 0 &&
                              (EPI != ALODLM_EPI_RESIDUAL ||
                               (ldr % 4 == 0 && reinterpret_cast<uintptr_t>(R) % 8 == 0));
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int64_t m = m0 + wm + i * 16 + (lane & 15), n = n0 + wn + j * 16 + 4 * (lane >> 4);
      if (m >= M || n >= N) continue;
      float v[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = alpha * acc[i][j][e];
      if (vec && n + 4 <= N) {
        if (fout) {
          float4* dst = reinterpret_cast<float4*>(Cf + m * ldf + n);
          if (EPI == ALODLM_EPI_ACCUM && !partial) {
            const float4 c = *dst;
            v[0] += c.x; v[1] += c.y; v[2] += c.z; v[3] += c.w;
          }
          *dst = make_float4(v[0], v[1], v[2], v[3]);
          continue;
        }
        if (EPI == ALODLM_EPI_RESIDUAL) {
          // reference order: x + round_bf16(proj), rounded once more
          const uint2 r = *reinterpret_cast<const uint2*>(R + m * ldr + n);
          v[0] = bf16_to_float((bf16_t)(r.x & 0xffff)) + round_bf16(v[0]);
          v[1] = bf16_to_float((bf16_t)(r.x >> 16)) + round_bf16(v[1]);
          v[2] = bf16_to_float((bf16_t)(r.y & 0xffff)) + round_bf16(v[2]);
          v[3] = bf16_to_float((bf16_t)(r.y >> 16)) + round_bf16(v[3]);
        }
        *reinterpret_cast<uint2*>(Cb + m * ldc + n) =
            make_uint2(pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]));
        continue;
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if (n + e >= N) continue;
        if (fout) {
          float* dst = Cf + m * ldf + n + e;
          *dst = EPI == ALODLM_EPI_ACCUM && !partial ? *dst + v[e] : v[e];
        } else if (EPI == ALODLM_EPI_RESIDUAL) {
          Cb[m * ldc + n + e] = float_to_bf16(bf16_to_float(R[m * ldr + n + e]) + round_bf16(v[e]));
        } else {
          Cb[m * ldc + n + e] = float_to_bf16(v[e]);
        }
      }
    }
}

template <bool AK, bool BKM, int MB, int STAGES>
void launch(const bf16_t* A, int64_t lda, const bf16_t* B, int64_t ldb, void* C, int64_t ldc,
            const bf16_t* R, int64_t ldr, int64_t M, int64_t N, int64_t K, float alpha, int epi,
            int64_t kps, int64_t nsplit, float* part, hipStream_t st) {
  const dim3 grid((unsigned)(((M + 32 * MB - 1) / (32 * MB)) * ((N + TN - 1) / TN)),
                  (unsigned)nsplit);
  if (epi == ALODLM_EPI_STORE)
    gemm_mid_kernel<AK, BKM, ALODLM_EPI_STORE, MB, STAGES><<<grid, 256, 0, st>>>(
        A, lda, B, ldb, C, ldc, R, ldr, M, N, K, alpha, kps, part);
  else if (epi == ALODLM_EPI_RESIDUAL)
    gemm_mid_kernel<AK, BKM, ALODLM_EPI_RESIDUAL, MB, STAGES><<<grid, 256, 0, st>>>(
        A, lda, B, ldb, C, ldc, R, ldr, M, N, K, alpha, kps, part);
  else if constexpr (MB == 4) {
    if (epi == ALODLM_EPI_ACCUM)
      gemm_mid_kernel<AK, BKM, ALODLM_EPI_ACCUM, MB, STAGES><<<grid, 256, 0, st>>>(
          A, lda, B, ldb, C, ldc, R, ldr, M, N, K, alpha, kps, part);
    else
      gemm_mid_kernel<AK, BKM, ALODLM_EPI_STORE_F32, MB, STAGES><<<grid, 256, 0, st>>>(
          A, lda, B, ldb, C, ldc, R, ldr, M, N, K, alpha, kps, part);
  }
}

template <bool AK, bool BKM>
void launch_rows(const bf16_t* A, int64_t lda, const bf16_t* B, int64_t ldb, void* C, int64_t ldc,
                 const bf16_t* R, int64_t ldr, int64_t M, int64_t N, int64_t K, float alpha,
                 int epi, int64_t kps, int64_t nsplit, float* part, int rows, hipStream_t st) {
  if constexpr (AK) {
    if (rows == 32) {
      launch<AK, BKM, 1, 6>(A, lda, B, ldb, C, ldc, R, ldr, M, N, K, alpha, epi, kps, nsplit, part, st);
      return;
    }
    if (rows == 64) {
      launch<AK, BKM, 2, 6>(A, lda, B, ldb, C, ldc, R, ldr, M, N, K, alpha, epi, kps, nsplit, part, st);
      return;
    }
  }
  launch<AK, BKM, 4, 4>(A, lda, B, ldb, C, ldc, R, ldr, M, N, K, alpha, epi, kps, nsplit, part, st);
}

}  // namespace

bool gemm_mid_eligible(const void* A, int64_t lda, int a_kmajor, const void* B, int64_t ldb,
                       int b_kmajor, int64_t M, int64_t N, int64_t K) {
  if (M < 8 || N < 8 || K < 1 || lda % 8 || ldb % 8) return false;
  if (((reinterpret_cast<uintptr_t>(A) | reinterpret_cast<uintptr_t>(B)) & 15) != 0) return false;
  // a k-contiguous row's chunks past K are not past the buffer
  if ((a_kmajor || b_kmajor) && K % KD) return false;
  if (!a_kmajor && M % 8) return false;
  if (!b_kmajor && N % 8) return false;
  // 32-bit buffer offsets, the zero-filled k rows past K included
  const int64_t ka = (K + KD - 1) / KD * KD;
  const int64_t abytes = 2 * (a_kmajor ? M : ka) * lda, bbytes = 2 * (b_kmajor ? N : ka) * ldb;
  return abytes < (1LL << 31) && bbytes < (1LL << 31);
}

int gemm_mid_rows(int a_kmajor, int64_t M, int epi) {
  if (!a_kmajor || (epi != ALODLM_EPI_STORE && epi != ALODLM_EPI_RESIDUAL)) return 128;
  return M <= 32 ? 32 : M <= 64 ? 64 : 128;
}

int64_t gemm_mid_launch(const bf16_t* A, int64_t lda, int a_kmajor, const bf16_t* B, int64_t ldb,
                        int b_kmajor, void* C, int64_t ldc, const bf16_t* R, int64_t ldr,
                        int64_t M, int64_t N, int64_t K, float alpha, int epi, int64_t splits,
                        float* workspace, hipStream_t st) {
  if (workspace == nullptr) splits = 1;
  const int64_t kps = ((K + splits - 1) / splits + KD - 1) / KD * KD;
  const int64_t nsplit = (K + kps - 1) / kps;
  float* part = nsplit > 1 ? workspace : nullptr;
  const int rows = gemm_mid_rows(a_kmajor, M, epi);
  if (a_kmajor && b_kmajor) launch_rows<true, true>(A, lda, B, ldb, C, ldc, R, ldr, M, N, K, alpha, epi, kps, nsplit, part, rows, st);
  else if (a_kmajor) launch_rows<true, false>(A, lda, B, ldb, C, ldc, R, ldr, M, N, K, alpha, epi, kps, nsplit, part, rows, st);
  else if (b_kmajor) launch_rows<false, true>(A, lda, B, ldb, C, ldc, R, ldr, M, N, K, alpha, epi, kps, nsplit, part, rows, st);
  else launch_rows<false, false>(A, lda, B, ldb, C, ldc, R, ldr, M, N, K, alpha, epi, kps, nsplit, part, rows, st);
  return nsplit;
}
