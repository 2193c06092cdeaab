"""A decoding window's layer and its fused products, against the
separate entry points' arithmetic in float64.

* alodlm_norm_product: rmsnorm(x) W^T and silu(gate) * up of it for 1 to 16
  rows, row strides wider than the rows, widths off the 16-row blocks, K off
  the wave split.  Normalised rows are rounded to bf16 (2^-8 of each
  term, which average out over K: 2^-8 of the sum's root mean square per
  rounding, four of those allowed) and the outputs once (2^-8 of the value).
* Kernels.layer_window: a whole layer at row counts on every product path and
  prefixes from none to a long one, against float64; bf16 3e-2 and float32 1e-5
  of the outputs' norm; the cached rows before the window stay as they are."""

import pytest
import torch
import torch.nn.functional as F

from alodlm_amd import _lib as L
from alodlm_amd.engine import Dims
from alodlm_amd.layers import Kernels, LayerWeights, Rope, WindowMask
from tests.helpers import log

pytestmark = pytest.mark.gpu
DEV, EPS = "cuda", 1e-6


def _norm(x, w):
    return w * (x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + EPS))


@pytest.mark.parametrize("M,N,K", [(1, 16, 8), (3, 34, 40), (16, 4096, 2048), (16, 1056, 264),
                                   (15, 130, 4096), (7, 24576, 520)])
@pytest.mark.parametrize("swiglu", [0, 1])
def test_norm_product(M, N, K, swiglu):
    log(f"norm product M={M} N={N} K={K} swiglu={swiglu}")
    dtype = torch.bfloat16
    g = torch.Generator(device=DEV).manual_seed(M + N + K)
    r = lambda *s: torch.randn(*s, generator=g, device=DEV).to(dtype)
    x, W, w = 3 * r(M, K + 8), r(N, K + 8), 1 + 0.1 * r(K)
    cols = N // 2 if swiglu else N
    out = torch.full((M, cols), float("nan"), dtype=dtype, device=DEV)
    L.call("alodlm_norm_product", L.ptr(x), K + 8, L.ptr(w), EPS, L.ptr(W), K + 8, L.ptr(out), cols,
           M, N, K, swiglu, L.dtype_code(dtype), torch.cuda.current_stream().cuda_stream)
    y = _norm(x[:, :K].double(), w.double()) @ W[:, :K].double().T
    ref = F.silu(y[:, :cols]) * y[:, cols:] if swiglu else y
    err = (out.double() - ref).abs()
    step = 2.0 ** -8 * (4 * K ** 0.5 + y.abs())  # of a sum, and its stored rounding
    if swiglu:
        gate, up = y[:, :cols], y[:, cols:]
        bound = 1.2 * step[:, :cols] * up.abs() + F.silu(gate).abs() * step[:, cols:] \
            + 1.2 * step[:, :cols] * step[:, cols:] + 2.0 ** -7 * ref.abs()
    else:
        bound = step
    assert bool((err <= bound + 1e-6).all()), float((err - bound).max())


def test_norm_product_rejects_wide_or_unaligned():
    log("norm product argument checks")
    t = torch.zeros(17 * 72, dtype=torch.bfloat16, device=DEV)
    st = torch.cuda.current_stream().cuda_stream
    with pytest.raises(ValueError, match="16 rows"):
        L.call("alodlm_norm_product", L.ptr(t), 64, L.ptr(t), EPS, L.ptr(t), 64, L.ptr(t), 16, 17,
               16, 64, 0, L.BF16_CODE, st)
    with pytest.raises(ValueError, match="aligned"):
        L.call("alodlm_norm_product", L.ptr(t) + 2, 64, L.ptr(t), EPS, L.ptr(t), 64, L.ptr(t), 16,
               4, 16, 64, 0, L.BF16_CODE, st)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("copies", [False, True])
@pytest.mark.parametrize("rows,prefix", [(1, 0), (16, 40), (17, 300), (40, 5), (100, 0), (130, 129)])
def test_window_layer(rows, prefix, copies, dtype):
    log(f"window layer rows={rows} prefix={prefix} copies={copies} {dtype}")
    H, nq, nkv, dh, I = 256, 4, 2, 128, 384
    kernels = Kernels(Dims(H, nq, nkv, dh, I, 0, 1, EPS, 0.0), dtype, torch.device(DEV))
    g = torch.Generator(device=DEV).manual_seed(rows + prefix)
    r = lambda *s: torch.randn(*s, generator=g, device=DEV).to(dtype)
    W, QD = kernels.dims.qkv_width, nq * dh
    mats = [0.06 * r(*s) for s in ((W, H), (H, QD), (2 * I, H), (H, I))]
    norms = [1 + 0.1 * r(n) for n in (H, H, dh, dh)]
    extra = [m.T.contiguous() for m in mats] if copies else [None] * 4
    w = LayerWeights(*mats, *norms, wqkv_t=extra[0], wo_t=extra[1], wgu_t=extra[2], wd_t=extra[3])
    x, angle = r(rows, H), torch.randn(rows, dh // 2, generator=g, device=DEV).repeat(1, 2)
    cos, sin = angle.cos().to(dtype), angle.sin().to(dtype)
    kbuf, vbuf = r(prefix + rows + 3, nkv, dh), r(prefix + rows + 3, nkv, dh)
    k0, v0 = kbuf.clone(), vbuf.clone()
    mask = WindowMask(prefix, rows, dtype == torch.bfloat16, DEV, block_size=32)
    y = kernels.layer_window(w, x, Rope(cos=cos, sin=sin), mask, kbuf, vbuf)

    d = lambda t: t.double()
    qkv = _norm(d(x), d(norms[0])) @ d(mats[0]).T
    q, k, v = qkv.split([QD, nkv * dh, nkv * dh], 1)
    half = lambda t: torch.cat((-t[..., dh // 2:], t[..., :dh // 2]), -1)
    rot = lambda t, n: (_norm(t, d(n)) * d(cos)[:, None] + half(_norm(t, d(n))) * d(sin)[:, None])
    q, k = rot(q.view(rows, nq, dh), norms[2]), rot(k.view(rows, nkv, dh), norms[3])
    v = v.view(rows, nkv, dh)
    K, V = (torch.cat((d(t[:prefix]), n)).repeat_interleave(nq // nkv, 1)
            for t, n in ((k0, k), (v0, v)))
    allowed = (torch.arange(prefix + rows, device=DEV)
               <= torch.arange(prefix, prefix + rows, device=DEV)[:, None])
    s = torch.einsum("qhd,khd->hqk", q, K) * dh ** -0.5
    o = torch.einsum("hqk,khd->qhd", torch.softmax(s.masked_fill(~allowed, float("-inf")), -1), V)
    x1 = d(x) + o.reshape(rows, QD) @ d(mats[1]).T
    gu = _norm(x1, d(norms[1])) @ d(mats[2]).T
    ref = x1 + (F.silu(gu[:, :I]) * gu[:, I:]) @ d(mats[3]).T
    tol = 3e-2 if dtype == torch.bfloat16 else 1e-5
    rel = lambda a, b: float((a.double() - b).norm() / b.norm())
    assert rel(y, ref) <= tol
    assert rel(kbuf[prefix:prefix + rows], k) <= tol and rel(vbuf[prefix:prefix + rows], v) <= tol
    for now, before in ((kbuf, k0), (vbuf, v0)):
        assert torch.equal(now[:prefix], before[:prefix])
        assert torch.equal(now[prefix + rows:], before[prefix + rows:])
