// One decoder layer as one host call (alodlm/model.py:49-76; a decoding window,
// alodlm/inference.py:83-88, and a differentiable call's forward and
// backward): the launches of the steps below are enqueued without returning
// to the caller between them, over one scratch allocation whose regions the
// steps share.  16 window rows keep the chip busy for 57 us per layer, and the
// separate calls with their output allocations took 95 us of host time, 36 us
// now.  Forward and backward of a 1.7B layer over 300 rows: 530 us a call and
// about 450 now (440 to 458 from card to card), with about 400 us of kernels;
// 2474 rows 1213 and 1199.
#include <algorithm>

#include "attention.h"
#include "common.h"

namespace {

constexpr int64_t FUSED_ROWS = 16;   // alodlm_norm_product's rows

#define RUN(call)           \
  do {                      \
    const int _rc = (call); \
    if (_rc) return _rc;    \
  } while (0)

struct Layer {
  int64_t rows, H, nq, nkv, dh, I;
  int dtype;
  float eps;
  void* stream;
  bool chain = false;  // products and attention as alodlm_gemm_chain sums them
  int64_t es() const { return dtype == ALODLM_BF16 ? 2 : 4; }
  int64_t QD() const { return nq * dh; }
  int64_t KD() const { return nkv * dh; }
  int64_t W() const { return QD() + 2 * KD(); }
  int64_t bytes(int64_t cols) const { return rows * cols * es(); }
  bool ok() const {
    return rows >= 0 && H > 0 && nq > 0 && nkv > 0 && dh > 0 && I > 0 &&
           (dtype == ALODLM_F32 || dtype == ALODLM_BF16);
  }
  // C = A w^T (+ R), w [N, K] or its copy w_t [K, N] where that serves the rows
  int product(const void* A, const void* w, const void* w_t, void* C, int64_t N, int64_t K,
              const void* R, float* ws) const {
    const bool copy = w_t != nullptr && rows > ALODLM_FEW_ROWS;
    return (chain ? alodlm_gemm_chain : alodlm_gemm)(
        A, K, 1, copy ? w_t : w, copy ? N : K, copy ? 0 : 1, C, N, R, R ? N : 0, rows, N, K, 1.f,
        R ? ALODLM_EPI_RESIDUAL : ALODLM_EPI_STORE, dtype, ws, stream);
  }
  // dA = dC w for the product above
  int input_grad(const void* dC, const void* w, void* dA, int64_t N, int64_t K, float* ws) const {
    return (chain ? alodlm_gemm_chain : alodlm_gemm)(dC, N, 1, w, K, 0, dA, K, nullptr, 0, rows, K,
                                                     N, 1.f, ALODLM_EPI_STORE, dtype, ws, stream);
  }
  // dw = dC^T A, in the storage dtype
  int weight_grad(const void* dC, const void* A, void* dw, int64_t N, int64_t K, float* ws) const {
    return alodlm_gemm(dC, N, 0, A, K, 0, dw, K, nullptr, 0, N, K, rows, 1.f, ALODLM_EPI_STORE,
                       dtype, ws, stream);
  }
  int norm(const void* x, const void* w, void* y, float* rstd) const {
    return alodlm_rmsnorm_fwd(x, w, y, rstd, rows, H, eps, dtype, stream);
  }
  int64_t product_workspace() const {
    return std::max(std::max(alodlm_gemm_workspace(rows, W(), H, ALODLM_EPI_STORE, dtype),
                             alodlm_gemm_workspace(rows, H, QD(), ALODLM_EPI_RESIDUAL, dtype)),
                    std::max(alodlm_gemm_workspace(rows, 2 * I, H, ALODLM_EPI_STORE, dtype),
                             alodlm_gemm_workspace(rows, H, I, ALODLM_EPI_RESIDUAL, dtype)));
  }
};

// Byte offsets of regions laid one after the other, each 256-byte aligned.
struct Regions {
  int64_t at = 0;
  int64_t take(int64_t bytes) {
    const int64_t here = at;
    at += (bytes + 255) / 256 * 256;
    return here;
  }
};

struct WindowScratch {
  int64_t qkv, q, o, x1, act, lse, h, gu, ws, total;
  explicit WindowScratch(const Layer& l) {
    Regions r;
    qkv = r.take(l.bytes(l.W()));
    q = r.take(l.bytes(l.QD()));
    o = r.take(l.bytes(l.QD()));
    x1 = r.take(l.bytes(l.H));
    act = r.take(l.bytes(l.I));
    lse = r.take(l.nq * l.rows * 4);
    h = r.take(l.bytes(l.H));
    gu = r.take(l.bytes(2 * l.I));
    ws = r.take(l.product_workspace() * 4);
    total = r.at;
  }
};

// What a forward keeps for its backward, besides its input and rotated keys.
struct Saved {
  int64_t rstd1, rstd2, lse, qkv, q, o, x1, gu, total;
  explicit Saved(const Layer& l) {
    Regions r;
    rstd1 = r.take(l.rows * 4);
    rstd2 = r.take(l.rows * 4);
    lse = r.take(l.nq * l.rows * 4);
    qkv = r.take(l.bytes(l.W()));
    q = r.take(l.bytes(l.QD()));
    o = r.take(l.bytes(l.QD()));
    x1 = r.take(l.bytes(l.H));
    gu = r.take(l.bytes(2 * l.I));
    total = r.at;
  }
};

// Forward: the norm outputs and the SwiGLU output are never live together.
struct ForwardScratch {
  int64_t h, ws, total;
  explicit ForwardScratch(const Layer& l) {
    Regions r;
    h = r.take(l.bytes(std::max(l.H, l.I)));
    ws = r.take(l.product_workspace() * 4);
    total = r.at;
  }
};

// Backward, three phases over the same bytes: {dgu, dact, act}, then
// {dgu, h2, dh2}, then {dx1, do | h1, dq | dh1, dk, dqkv} with dx1 written
// over dgu while dh2 behind it is read.
struct BackwardScratch {
  int64_t dgu, dact, act, h2, dh2, dx1, dout, dq, dk, dqkv, ws, total;
  BackwardScratch(const Layer& l, int64_t n_tiles, int64_t ds_blocks) {
    const int64_t wide = l.bytes(std::max(l.H, l.QD()));
    Regions a;
    dgu = a.take(std::max(l.bytes(2 * l.I), l.bytes(l.H)));
    Regions b = a, c;
    dact = a.take(l.bytes(l.I));
    act = a.take(l.bytes(l.I));
    h2 = b.take(l.bytes(l.H));
    dh2 = b.take(l.bytes(l.H));
    dx1 = c.take(l.bytes(l.H));
    dout = c.take(wide);
    dq = c.take(wide);
    dk = c.take(l.bytes(l.KD()));
    dqkv = c.take(l.bytes(l.W()));
    Regions r;
    r.at = std::max(a.at, std::max(b.at, c.at));
    const int S = ALODLM_EPI_STORE, t = l.dtype;
    int64_t n = std::max(alodlm_rmsnorm_bwd_workspace(l.rows, l.H),
                         alodlm_qknorm_rope_bwd_workspace(l.rows, l.nq, l.nkv, l.dh));
    n = std::max(n, alodlm_attention_bwd_workspace(l.rows, l.nq, l.nkv, l.dh, n_tiles, ds_blocks));
    const int64_t mats[4][2] = {{l.W(), l.H}, {l.H, l.QD()}, {2 * l.I, l.H}, {l.H, l.I}};
    for (const auto& m : mats) {
      n = std::max(n, alodlm_gemm_workspace(l.rows, m[1], m[0], S, t));
      n = std::max(n, alodlm_gemm_workspace(m[0], m[1], l.rows, S, t));
    }
    ws = r.take(n * 4);
    total = r.at;
  }
};

struct Memory {
  char* base;
  void* operator[](int64_t off) const { return base + off; }
  float* floats(int64_t off) const { return reinterpret_cast<float*>(base + off); }
};

}  // namespace

extern "C" int64_t alodlm_window_layer_scratch(int64_t rows, int64_t hidden, int64_t nq,
                                               int64_t nkv, int64_t dh, int64_t inter, int dtype) {
  const Layer l{rows, hidden, nq, nkv, dh, inter, dtype, 0.f, nullptr};
  return l.ok() ? WindowScratch(l).total : 0;
}

extern "C" int alodlm_window_layer(
    const void* x, const void* wqkv, const void* wqkv_t, const void* wo, const void* wo_t,
    const void* wgu, const void* wgu_t, const void* wd, const void* wd_t, const void* ln1,
    const void* ln2, const void* qn, const void* kn, const void* cos_tab, const void* sin_tab,
    void* kbuf, void* vbuf, int64_t prefix, int64_t base, const int64_t* bounds,
    const int32_t* row_segment, const int32_t* tiles, int64_t n_tiles, int64_t block_size,
    void* scratch, void* y, int64_t rows, int64_t hidden, int64_t nq, int64_t nkv, int64_t dh,
    int64_t inter, float eps, int dtype, void* stream) {
  const Layer l{rows, hidden, nq, nkv, dh, inter, dtype, eps, stream};
  ALODLM_CHECK_ARG(l.ok(), "window_layer: bad shape or dtype");
  ALODLM_CHECK_ARG(rows == 0 || (cos_tab && sin_tab), "window_layer: needs rotary tables");
  // the query rows start at the window, so the mask's row 0 is key row `prefix`
  ALODLM_CHECK_ARG(prefix >= 0 && base == prefix, "window_layer: bad prefix");
  const WindowScratch s(l);
  const Memory m{static_cast<char*>(scratch)};
  float* ws = m.floats(s.ws);
  const int64_t H = l.H, I = l.I, row = l.KD() * l.es();
  auto aligned = [](const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; };
  // rmsnorm(a) w^T, or silu(gate) * up of it
  auto norm_product = [&](const void* a, const void* norm, const void* w, const void* w_t, void* C,
                          int64_t N, bool swiglu) -> int {
    if (rows <= FUSED_ROWS && dtype == ALODLM_BF16 && H % 8 == 0 && aligned(a) && aligned(norm) &&
        aligned(w) && N * H * 2 < (1LL << 31))
      return alodlm_norm_product(a, H, norm, eps, w, H, C, swiglu ? N / 2 : N, rows, N, H, swiglu,
                                 dtype, stream);
    RUN(l.norm(a, norm, m[s.h], nullptr));
    RUN(l.product(m[s.h], w, w_t, swiglu ? m[s.gu] : C, N, H, nullptr, ws));
    return swiglu ? alodlm_swiglu_fwd(m[s.gu], C, rows, N / 2, dtype, stream) : ALODLM_OK;
  };
  char* kb = static_cast<char*>(kbuf);
  char* vb = static_cast<char*>(vbuf);
  RUN(norm_product(x, ln1, wqkv, wqkv_t, m[s.qkv], l.W(), false));
  RUN(alodlm_qknorm_rotary_window(m[s.qkv], qn, kn, cos_tab, sin_tab, m[s.q], kb + prefix * row,
                                  vb + prefix * row, rows, nq, nkv, dh, eps, dtype, stream));
  RUN(alodlm_attention_fwd(m[s.q], kb + base * row, vb + base * row, l.KD(), bounds, row_segment,
                           tiles, n_tiles, m[s.o], m.floats(s.lse), rows, nq, nkv, dh, block_size,
                           dtype, stream));
  RUN(l.product(m[s.o], wo, wo_t, m[s.x1], H, l.QD(), x, ws));
  RUN(norm_product(m[s.x1], ln2, wgu, wgu_t, m[s.act], 2 * I, true));
  return l.product(m[s.act], wd, wd_t, y, H, I, m[s.x1], ws);
}

extern "C" int64_t alodlm_layer_saved(int64_t rows, int64_t hidden, int64_t nq, int64_t nkv,
                                      int64_t dh, int64_t inter, int dtype) {
  const Layer l{rows, hidden, nq, nkv, dh, inter, dtype, 0.f, nullptr};
  return l.ok() ? Saved(l).total : 0;
}

extern "C" int64_t alodlm_layer_fwd_scratch(int64_t rows, int64_t hidden, int64_t nq, int64_t nkv,
                                            int64_t dh, int64_t inter, int dtype) {
  const Layer l{rows, hidden, nq, nkv, dh, inter, dtype, 0.f, nullptr};
  return l.ok() ? ForwardScratch(l).total : 0;
}

extern "C" int alodlm_layer_fwd(const void* x, const void* wqkv, const void* wo, const void* wgu,
                                const void* wd, const void* ln1, const void* ln2, const void* qn,
                                const void* kn, const void* cos_tab, const void* sin_tab,
                                const int64_t* positions, const float* inv_freq,
                                const int64_t* bounds, const int32_t* row_segment,
                                const int32_t* tiles, int64_t n_tiles, int64_t block_size, void* k,
                                void* v, void* saved, void* scratch, void* y, int64_t rows,
                                int64_t hidden, int64_t nq, int64_t nkv, int64_t dh, int64_t inter,
                                float eps, int chain, int dtype, void* stream) {
  const Layer l{rows, hidden, nq, nkv, dh, inter, dtype, eps, stream, chain != 0};
  ALODLM_CHECK_ARG(l.ok(), "layer_fwd: bad shape or dtype");
  ALODLM_CHECK_ARG(rows == 0 || (cos_tab ? sin_tab && v : positions && inv_freq && !v),
                   "layer_fwd: needs rotary tables with v, or positions without");
  const Saved s(l);
  const ForwardScratch t(l);
  const Memory m{static_cast<char*>(saved)}, tmp{static_cast<char*>(scratch)};
  void* h = tmp[t.h];
  float* ws = tmp.floats(t.ws);
  RUN(l.norm(x, ln1, h, m.floats(s.rstd1)));
  RUN(l.product(h, wqkv, nullptr, m[s.qkv], l.W(), l.H, nullptr, ws));
  int64_t ldv = l.KD();
  if (v) {
    RUN(alodlm_qknorm_rotary_window(m[s.qkv], qn, kn, cos_tab, sin_tab, m[s.q], k, v, rows, nq, nkv,
                                    dh, eps, dtype, stream));
  } else {
    RUN(alodlm_qknorm_rope_fwd(m[s.qkv], qn, kn, positions, inv_freq, m[s.q], k, rows, nq, nkv, dh,
                               eps, dtype, stream));
    v = static_cast<char*>(m[s.qkv]) + (l.QD() + l.KD()) * l.es();
    ldv = l.W();
  }
  RUN(attention_fwd(m[s.q], k, v, ldv, bounds, row_segment, tiles, n_tiles, m[s.o],
                    m.floats(s.lse), rows, nq, nkv, dh, block_size, dtype, l.chain, stream));
  RUN(l.product(m[s.o], wo, nullptr, m[s.x1], l.H, l.QD(), x, ws));
  RUN(l.norm(m[s.x1], ln2, h, m.floats(s.rstd2)));
  RUN(l.product(h, wgu, nullptr, m[s.gu], 2 * l.I, l.H, nullptr, ws));
  RUN(alodlm_swiglu_fwd(m[s.gu], h, rows, l.I, dtype, stream));
  return l.product(h, wd, nullptr, y, l.H, l.I, m[s.x1], ws);
}

extern "C" int64_t alodlm_layer_bwd_scratch(int64_t rows, int64_t hidden, int64_t nq, int64_t nkv,
                                            int64_t dh, int64_t inter, int64_t n_tiles,
                                            int64_t ds_blocks, int dtype) {
  const Layer l{rows, hidden, nq, nkv, dh, inter, dtype, 0.f, nullptr};
  return l.ok() ? BackwardScratch(l, n_tiles, ds_blocks).total : 0;
}

extern "C" int alodlm_layer_bwd(
    const void* dy, const void* x, const void* k, const void* saved, const void* wqkv,
    const void* wo, const void* wgu, const void* wd, const void* ln1, const void* ln2,
    const void* qn, const void* kn, const void* cos_tab, const void* sin_tab,
    const int64_t* positions, const float* inv_freq, const int64_t* bounds,
    const int32_t* row_segment, const int32_t* tiles, int64_t n_tiles, const int64_t* ds_base,
    int64_t ds_blocks, int64_t block_size, void* dwqkv, void* dwo, void* dwgu, void* dwd,
    float* dln1, float* dln2, float* dqn, float* dkn, void* scratch, void* dx, int64_t rows,
    int64_t hidden, int64_t nq, int64_t nkv, int64_t dh, int64_t inter, float eps, int chain,
    int dtype, void* stream) {
  const Layer l{rows, hidden, nq, nkv, dh, inter, dtype, eps, stream, chain != 0};
  ALODLM_CHECK_ARG(l.ok(), "layer_bwd: bad shape or dtype");
  ALODLM_CHECK_ARG(rows == 0 || (cos_tab ? sin_tab != nullptr : positions && inv_freq),
                   "layer_bwd: needs rotary tables or positions");
  const Saved s(l);
  const BackwardScratch t(l, n_tiles, ds_blocks);
  const Memory m{static_cast<char*>(const_cast<void*>(saved))}, tmp{static_cast<char*>(scratch)};
  float* ws = tmp.floats(t.ws);
  const int64_t H = l.H, I = l.I, W = l.W(), QD = l.QD(), KD = l.KD();
  // ---- MLP: y = x1 + act Wd^T (the SwiGLU backward also rewrites act)
  RUN(l.input_grad(dy, wd, tmp[t.dact], H, I, ws));
  RUN(alodlm_swiglu_bwd(tmp[t.dact], m[s.gu], tmp[t.dgu], tmp[t.act], rows, I, dtype, stream));
  RUN(l.weight_grad(dy, tmp[t.act], dwd, H, I, ws));
  RUN(l.norm(m[s.x1], ln2, tmp[t.h2], nullptr));
  RUN(l.input_grad(tmp[t.dgu], wgu, tmp[t.dh2], 2 * I, H, ws));
  RUN(l.weight_grad(tmp[t.dgu], tmp[t.h2], dwgu, 2 * I, H, ws));
  RUN(alodlm_rmsnorm_bwd(tmp[t.dh2], m[s.x1], m.floats(s.rstd2), ln2, dy, tmp[t.dx1], dln2, ws,
                         rows, H, dtype, stream));
  // ---- attention: x1 = x + o Wo^T
  RUN(l.input_grad(tmp[t.dx1], wo, tmp[t.dout], H, QD, ws));
  RUN(l.weight_grad(tmp[t.dx1], m[s.o], dwo, H, QD, ws));
  char* v = static_cast<char*>(m[s.qkv]) + (QD + KD) * l.es();
  char* dv = static_cast<char*>(tmp[t.dqkv]) + (QD + KD) * l.es();
  RUN(alodlm_attention_bwd(m[s.q], k, v, W, m[s.o], m.floats(s.lse), tmp[t.dout], bounds,
                           row_segment, tiles, n_tiles, tmp[t.dq], tmp[t.dk], dv, W, ws, ds_base,
                           ds_blocks, rows, nq, nkv, dh, block_size, dtype, stream));
  if (cos_tab)
    RUN(alodlm_qknorm_rotary_bwd(tmp[t.dq], tmp[t.dk], m[s.qkv], qn, kn, cos_tab, sin_tab,
                                 tmp[t.dqkv], dqn, dkn, ws, rows, nq, nkv, dh, eps, dtype, stream));
  else
    RUN(alodlm_qknorm_rope_bwd(tmp[t.dq], tmp[t.dk], m[s.qkv], qn, kn, positions, inv_freq,
                               tmp[t.dqkv], dqn, dkn, ws, rows, nq, nkv, dh, eps, dtype, stream));
  void* h1 = tmp[t.dout];
  void* dh1 = tmp[t.dq];
  RUN(l.norm(x, ln1, h1, nullptr));
  RUN(l.input_grad(tmp[t.dqkv], wqkv, dh1, W, H, ws));
  RUN(l.weight_grad(tmp[t.dqkv], h1, dwqkv, W, H, ws));
  return alodlm_rmsnorm_bwd(dh1, x, m.floats(s.rstd1), ln1, tmp[t.dx1], dx, dln1, ws, rows, H,
                            dtype, stream);
}
