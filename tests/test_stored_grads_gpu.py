"""Gradients written in the parameter dtype: the embedding scatter into a
storage-type table (bit-equal to the float32 table rounded, runs of one row up
to several chunks, both column widths, filtered rows), and a layer's projection
gradients stored by their products against the float32 accumulated ones (the
float32 sums of two kernels differ by a few units of float32; a bf16 store adds
half a unit of its last place, 2^-8)."""

import pytest
import torch

from alodlm_amd import _lib as L
from alodlm_amd.engine import Dims
from alodlm_amd.layers import (DualStreamMask, Kernels, LayerGrads, LayerWeights, Rope,
                               _LayerFunction)
from tests.helpers import log

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("rows,hidden", [(1, 8), (70, 33), (200, 40), (500, 2056)])
@pytest.mark.parametrize("filtered", [False, True])
def test_embed_scatter_storage_table(rows, hidden, dtype, filtered):
    log(f"embed scatter rows={rows} hidden={hidden} {dtype} filtered={filtered}")
    vocab, g = 37, torch.Generator().manual_seed(rows + hidden)
    ids = torch.randint(-1, vocab + 1, (rows,), generator=g)
    ids[rows // 3:] = 5  # a run of several chunks; ids outside the table take no part
    ids = ids.to(DEV)
    dout = torch.randn(rows, hidden, generator=g).to(dtype).to(DEV)
    exits = torch.randint(0, 3, (rows,), generator=g).to(torch.int32).to(DEV) if filtered else None
    st = torch.cuda.current_stream().cuda_stream
    plan = torch.empty(L.query("alodlm_embed_plan_size", rows), dtype=torch.int32, device=DEV)
    L.call("alodlm_embed_plan", L.ptr(ids), rows, vocab, L.ptr(plan), st)
    ws = torch.empty(L.query("alodlm_embed_scatter_workspace", rows, hidden), device=DEV)
    tables = []
    for name, t in (("alodlm_embed_scatter_add", torch.float32), ("alodlm_embed_scatter", dtype)):
        table = torch.zeros(vocab, hidden, dtype=t, device=DEV)
        L.call(name, L.ptr(dout), L.ptr(plan), L.ptr(exits), 1, L.ptr(table), L.ptr(ws), rows,
               hidden, vocab, L.dtype_code(dtype), st)
        tables.append(table)
    assert torch.equal(tables[0].to(dtype), tables[1])


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("lengths", [[3], [40, 25], [160]])
def test_layer_gradients_stored(lengths, dtype):
    log(f"stored layer gradients lengths={lengths} {dtype}")
    H, nq, nkv, dh, I = 256, 2, 1, 128, 264
    kernels = Kernels(Dims(H, nq, nkv, dh, I, 0, 1, 1e-6, 0.0), dtype, torch.device(DEV))
    g = torch.Generator(device=DEV).manual_seed(sum(lengths))
    rand = lambda *s: torch.randn(*s, generator=g, device=DEV)
    W, QD = kernels.dims.qkv_width, nq * dh
    shapes = [(W, H), (H, QD), (2 * I, H), (H, I)]
    mats = [(0.05 * rand(*s)).to(dtype) for s in shapes]
    norms = [(1 + 0.05 * rand(n)).to(dtype) for n in (H, H, dh, dh)]
    offsets = [0]
    for n in lengths:
        offsets.append(offsets[-1] + n)
    N = 2 * offsets[-1]
    mask = DualStreamMask(offsets, 32, torch.device(DEV))
    angle = rand(N, dh)
    rope = Rope(cos=angle.cos().to(dtype), sin=angle.sin().to(dtype))
    x, dy = rand(N, H).to(dtype), rand(N, H).to(dtype)
    results = []
    for stored in (True, False):
        save = []
        w = LayerWeights(*mats, *norms)
        kernels.layer_fwd(w, x, mask, rope, save, keep=(True, False))
        t = dtype if stored else torch.float32
        out = [torch.full(s, float("nan") if stored else 0.0, dtype=t, device=DEV) for s in shapes]
        gn = [torch.zeros(n, device=DEV) for n in (H, H, dh, dh)]
        dx = kernels.layer_bwd(dy, save[0], w, LayerGrads(*out, *gn, stored=stored), mask, rope)
        results.append((dx, out, gn))
    (dx, got, gn), (dx2, ref, gn2) = results
    assert torch.equal(dx, dx2)
    for a, b in zip(gn, gn2):
        assert torch.equal(a, b)
    for a, b in zip(got, ref):
        bound = 2.0 ** -20 * N ** 0.5 * b.abs().max()
        if dtype == torch.bfloat16:
            bound = bound + 2.0 ** -8 * b.abs()
        assert bool(((a.float() - b).abs() <= bound).all())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("trained", [(0,), (1, 4), (3, 6), tuple(range(11))])
def test_gradients_hold_their_own_memory(trained, dtype):
    """A parameter's gradient holds no memory of parameters that are not
    trained: its storage is its own size, or its group's (q|k|v, gate|up: one
    product writes them) when the whole group is trained.  Values do not depend
    on which parameters are."""
    log(f"gradient storage, trained parameters {trained} {dtype}")
    H, nq, nkv, dh, I = 256, 2, 1, 128, 264
    kernels = Kernels(Dims(H, nq, nkv, dh, I, 0, 1, 1e-6, 0.0), dtype, torch.device(DEV))
    g = torch.Generator(device=DEV).manual_seed(7)
    shapes = [(nq * dh, H), (nkv * dh, H), (nkv * dh, H), (H, nq * dh), (I, H), (I, H), (H, I),
              (H,), (H,), (dh,), (dh,)]
    mask = DualStreamMask([0, 40, 65], 32, torch.device(DEV))
    rope = Rope(positions=torch.arange(mask.rows, device=DEV) % 40,
                inv_freq=torch.rand(dh // 2, generator=g, device=DEV))
    data = [0.05 * torch.randn(*s, generator=g, device=DEV) + (len(s) == 1) for s in shapes]
    x, dy = (torch.randn(mask.rows, H, generator=g, device=DEV).to(dtype) for _ in range(2))

    def grads(which):
        params = [t.to(dtype, copy=True).requires_grad_(i in which) for i, t in enumerate(data)]
        _LayerFunction.apply(kernels, mask, rope, False, x, *params)[0].backward(dy)
        return [p.grad for p in params]
    full, got = grads(range(11)), grads(trained)
    groups = ((0, 1, 2), (3,), (4, 5), (6,))
    for i, t in enumerate(got):
        assert (t is not None) == (i in trained)
        if t is None:
            continue
        assert torch.equal(t, full[i]), i
        if i < 7:
            group = next(m for m in groups if i in m)
            owners = group if set(group) <= set(trained) else (i,)
            size = sum(data[j].numel() for j in owners) * t.element_size()
            held = t.untyped_storage().nbytes()
            assert held == size, i
