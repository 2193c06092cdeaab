"""A differentiable layer as one host call each way against the same steps
called one by one.

alodlm_layer_fwd / alodlm_layer_bwd enqueue Kernels.layer_fwd's and layer_bwd's
launches over regions of one scratch allocation, so every output and gradient
is bit-identical; a region reused too early shows as a difference.  Sizes: one
row to several tiles, packs whose longest region is the MLP's or the
attention's (wide heads over a narrow MLP), block sizes with and without the
stored-dS backward, both storage types."""

import pytest
import torch

from alodlm_amd.engine import Dims
from alodlm_amd.layers import DualStreamMask, Kernels, LayerGrads, LayerWeights, Rope
from tests.helpers import log

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("tables", [True, False])
@pytest.mark.parametrize("H,nq,nkv,dh,I,lengths,block", [
    (64, 2, 1, 32, 96, (1,), 4), (128, 8, 2, 64, 64, (37, 5), 32), (256, 4, 2, 128, 768, (130,), 32),
    (256, 2, 2, 128, 1024, (129, 64, 1), 16), (64, 8, 4, 128, 40, (70,), 32)])
def test_layer_call_matches_steps(H, nq, nkv, dh, I, lengths, block, tables, dtype):
    log(f"layer call H={H} heads={nq}/{nkv}x{dh} I={I} lengths={lengths} block={block} tables={tables} {dtype}")
    kernels = Kernels(Dims(H, nq, nkv, dh, I, 0, 1, 1e-6, 0.0), dtype, torch.device(DEV))
    offsets = [0]
    for n in lengths:
        offsets.append(offsets[-1] + n)
    mask = DualStreamMask(offsets, block, torch.device(DEV))
    N, QD, KD, W = mask.rows, nq * dh, nkv * dh, kernels.dims.qkv_width
    g = torch.Generator(device=DEV).manual_seed(H + I + N)
    r = lambda *s: torch.randn(*s, generator=g, device=DEV).to(dtype)
    w = LayerWeights(*[0.06 * r(*s) for s in ((W, H), (H, QD), (2 * I, H), (H, I))],
                     *[1 + 0.1 * r(n) for n in (H, H, dh, dh)])
    angle = torch.randn(N, dh // 2, generator=g, device=DEV).repeat(1, 2)
    rope = Rope(cos=angle.cos().to(dtype), sin=angle.sin().to(dtype))
    if not tables:
        rope = Rope(positions=torch.arange(N, device=DEV) % 7,
                    inv_freq=torch.rand(dh // 2, generator=g, device=DEV))
    x, dy = r(N, H), r(N, H)

    def grads():
        mats = [torch.full(t.shape, float("nan"), dtype=dtype, device=DEV)
                for t in (w.wqkv, w.wo, w.wgu, w.wd)]
        return LayerGrads(*mats, *[torch.zeros(n, device=DEV) for n in (H, H, dh, dh)], stored=True)

    save, ref = [], grads()
    y0 = kernels.layer_fwd(w, x, mask, rope, save, keep=(True, False))
    dx0 = kernels.layer_bwd(dy, save[0], w, ref, mask, rope)
    got = grads()
    y, k, v, saved = kernels.layer_call_fwd(w, x, rope, mask)
    dx = kernels.layer_call_bwd(dy, x, k, saved, w, got, rope, mask)
    assert torch.equal(y, y0) and torch.equal(dx, dx0)
    assert torch.equal(k.view(N, KD), save[0][10])
    if tables:
        assert torch.equal(v.view(N, KD), save[0][3][:, QD + KD:])
    for name in ("wqkv", "wo", "wgu", "wd", "ln1", "ln2", "qn", "kn"):
        assert torch.equal(getattr(got, name), getattr(ref, name)), name


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_layer_call_of_no_rows(dtype):
    """No rows: empty outputs, zero weight gradients."""
    log(f"layer call of no rows {dtype}")
    H, nq, nkv, dh, I = 256, 2, 1, 128, 264
    kernels = Kernels(Dims(H, nq, nkv, dh, I, 0, 1, 1e-6, 0.0), dtype, torch.device(DEV))
    W, QD = kernels.dims.qkv_width, nq * dh
    shapes = ((W, H), (H, QD), (2 * I, H), (H, I))
    w = LayerWeights(*[torch.ones(s, device=DEV).to(dtype) for s in shapes],
                     *[torch.ones(n, device=DEV).to(dtype) for n in (H, H, dh, dh)])
    mask = DualStreamMask([0, 0], 32, torch.device(DEV))
    rope = Rope(cos=torch.empty(0, dh, dtype=dtype, device=DEV),
                sin=torch.empty(0, dh, dtype=dtype, device=DEV))
    x = torch.empty(0, H, dtype=dtype, device=DEV)
    g = LayerGrads(*[torch.full(s, float("nan"), dtype=dtype, device=DEV) for s in shapes],
                   *[torch.zeros(n, device=DEV) for n in (H, H, dh, dh)], stored=True)
    y, k, v, saved = kernels.layer_call_fwd(w, x, rope, mask)
    dx = kernels.layer_call_bwd(x, x, k, saved, w, g, rope, mask)
    assert y.shape == dx.shape == (0, H) and k.shape == v.shape == (0, nkv, dh)
    for t in (g.wqkv, g.wo, g.wgu, g.wd, g.ln1, g.ln2, g.qn, g.kn):
        assert not bool(t.any())
