"""ALoDLM.rollout and the fused step in bf16: a row's sums run in one order
whatever the other rows of the pack, and every output of a rollout against 64
bits.

Both apply their layers once per depth to their own outputs, so a product summed
in another order reaches every later depth; the word-embedding gradient, whose
few nonzero rows dilute the table's root mean square, shows it at single
elements by more than that root mean square, and the step's loss, a difference
of credits, by some percent."""

import pytest
import torch

from alodlm_amd import _lib as L
from alodlm_amd.batch import build_batch
from alodlm_amd.layers import DualStreamMask, LayerWeights, Rope, _LayerFunction
from perf import cases
from tests.helpers import log

pytestmark = pytest.mark.gpu
DEV, BF16 = "cuda", torch.bfloat16


def _product(name, A, B, b_kmajor, R, N):
    M, K = A.shape
    C = torch.full((M, N), float("nan"), dtype=BF16, device=DEV)
    epi = L.EPI_STORE if R is None else L.EPI_RESIDUAL
    ws = torch.empty(max(1, L.query("alodlm_gemm_workspace", M, N, K, epi, L.BF16_CODE)),
                     device=DEV)
    L.call(name, L.ptr(A), K, 1, L.ptr(B), K if b_kmajor else N, b_kmajor, L.ptr(C), N, L.ptr(R),
           N, M, N, K, 1.0, epi, L.BF16_CODE, L.ptr(ws), torch.cuda.current_stream().cuda_stream)
    return C


# a K with many splits, one of no whole 32-deep stage, columns of no whole tile,
# and the small products of narrow models
@pytest.mark.parametrize("N,K,b_kmajor,residual", [
    (2048, 6144, 1, True), (2048, 12288, 0, False), (4096, 2048, 1, False), (520, 1056, 1, True),
    (264, 200, 0, False), (72, 40, 1, False), (256, 16384, 0, False)])
def test_chain_product_rows(N, K, b_kmajor, residual):
    """alodlm_gemm_chain gives a row the same bits in products of 1 to 300 rows,
    on every tile and kernel the row counts reach, within a bf16 store's half
    unit (2^-8) and the float32 sum's rounding (K terms: K^0.5 2^-22 of the sum
    of their sizes) of float64."""
    log(f"chain product N={N} K={K} b_kmajor={b_kmajor} residual={residual}")
    g = torch.Generator(device=DEV).manual_seed(N + K)
    A = torch.randn(300, K, generator=g, device=DEV).to(BF16)
    W = (0.05 * torch.randn(N, K, generator=g, device=DEV)).to(BF16)
    R = torch.randn(300, N, generator=g, device=DEV).to(BF16) if residual else None
    B = W if b_kmajor else W.T.contiguous()
    # K >= 16384 splits from 256 rows on
    full = _product("alodlm_gemm_chain", A[:255] if K >= 16384 else A, B, b_kmajor,
                    R, N)
    s = A[:len(full)].double() @ W.double().T
    sizes = A[:len(full)].double().abs() @ W.double().abs().T
    ref = s if R is None else R[:len(full)].double() + s
    # a residual output is rounded twice (the product, then the sum)
    bound = 2.0 ** -8 * (ref.abs() + (s.abs() if residual else 0)) + K ** 0.5 * 2.0 ** -22 * sizes
    assert bool(((full.double() - ref).abs() <= bound).all())
    for m in (1, 7, 16, 27, 33, 48, 64, 65, 128, 200, 255):
        part = _product("alodlm_gemm_chain", A[:m], B, b_kmajor, R, N)
        assert torch.equal(part, full[:m]), m


def _segment(model, length, seed):
    gen = torch.Generator().manual_seed(seed)
    ids = torch.randint(0, 500, (length,), generator=gen)
    probs, counts, perms = [], [], []
    for left in range(0, length, model.config.block_size):
        n = min(model.config.block_size, length - left)
        probs.append(0.5)
        counts.append(round(0.5 * n))
        perms.append(torch.randperm(n, generator=gen))
    uniforms = [torch.rand(2 * length, generator=gen) for _ in range(model.config.max_depth - 1)]
    return ids, (probs, counts, perms), uniforms


def _rollout(model, segments):
    ids = torch.cat([s[0] for s in segments])
    bounds = [0]
    for s in segments:
        bounds.append(bounds[-1] + len(s[0]))
    draws = tuple(sum((s[1][i] for s in segments), []) for i in range(3))
    c = model.config
    batch = build_batch(ids.to(DEV), ids.to(DEV), torch.tensor(bounds), c.block_size,
                        c.mask_token_id, draws=draws)
    u = [torch.cat(t).to(DEV) for t in zip(*(s[2] for s in segments))]
    with torch.no_grad():
        return model.rollout(batch, exit_uniforms=u)


@pytest.mark.parametrize("length", [5, 20, 40, 130])
def test_rollout_rows_do_not_depend_on_the_pack(length):
    """A segment's logits, gates and exits are bit-identical alone and beside
    other segments (10 to 690 rows of a 1.7B layer: the row counts of every
    tile, of K splits and of the few-row kernels)."""
    log(f"rollout of {length} tokens alone and in a pack")
    model = cases._model("1.7b", 1, 512, 511, BF16, cases._generator(length))
    segments = [_segment(model, n, n) for n in (length, 200, 15)]
    alone, packed = _rollout(model, segments[:1]), _rollout(model, segments)
    n = 2 * length
    for a, b in zip(alone[0] + alone[1], packed[0] + packed[1]):
        assert torch.equal(a, b[:n])
    assert torch.equal(alone[2], packed[2][:n])


def _step(model, segments):
    ids = torch.cat([s[0] for s in segments])
    bounds = [0]
    for s in segments:
        bounds.append(bounds[-1] + len(s[0]))
    draws = tuple(sum((s[1][i] for s in segments), []) for i in range(3))
    u = [torch.cat(t).to(DEV) for t in zip(*(s[2] for s in segments))]
    with torch.no_grad():
        return model.engine().forward(ids.to(DEV), ids.to(DEV), torch.tensor(bounds), False,
                                      exit_uniforms=u, draws=draws)[1]


@pytest.mark.parametrize("length", [5, 20, 40, 130])
def test_step_rows_do_not_depend_on_the_pack(length):
    """The fused step's gates, exits and per-row cross-entropies of a segment are
    bit-identical alone and beside other segments, and its gates and exits are
    the rollout's."""
    log(f"step of {length} tokens alone and in a pack")
    model = cases._model("1.7b", 1, 512, 511, BF16, cases._generator(length))
    segments = [_segment(model, n, n) for n in (length, 200, 15)]
    alone, packed = _step(model, segments[:1]), _step(model, segments)
    n = 2 * length
    for name in ("gates", "ce", "entropy"):
        assert torch.equal(alone[name], packed[name][:, :n]), name
    assert torch.equal(alone["exits"], packed["exits"][:n])
    _, gates, exits = _rollout(model, segments)
    assert torch.equal(torch.stack(gates), packed["gates"].to(BF16))
    assert torch.equal(exits, packed["exits"].long())


@pytest.mark.parametrize("length", [3, 20, 130])
def test_layer_input_gradient_does_not_depend_on_the_pack(length):
    """The same of one layer's backward: dx of a segment's rows."""
    log(f"layer input gradient of {length} tokens alone and in a pack")
    gen = cases._generator(length)
    model = cases._model("1.7b", 1, 256, 255, BF16, gen)
    kernels, layer = model.engine(), model.backbone.model.layers[0]
    x = torch.randn(2 * (length + 200), 2048, generator=gen, device=DEV).to(BF16)
    dy = torch.randn(x.shape, generator=gen, device=DEV).to(BF16)
    positions = torch.arange(len(x), device=DEV) % 211
    grads = []
    for offsets in ([0, length], [0, length, length + 200]):
        n = 2 * offsets[-1]
        h = x[:n].clone().requires_grad_(True)
        rope = Rope(positions=positions[:n].contiguous(), inv_freq=kernels.inv_freq)
        y = _LayerFunction.apply(kernels, DualStreamMask(offsets, 32, torch.device(DEV)), rope,
                                 True, h, *LayerWeights.module_tensors(layer))[0]
        grads.append(torch.autograd.grad(y, h, dy[:n])[0])
    assert torch.equal(grads[0], grads[1][:2 * length])


@pytest.mark.parametrize("segments", ["60,37", "24"])
def test_rollout_against_64_bits(segments):
    """Every output of a full-vocabulary rollout, and the gradient of every
    parameter, against float64 of the same inputs.  Some hundred bf16 roundings
    lie between the embedding and its gradient (a dozen a layer call and depth,
    forward and backward): 100^0.5 times the rms of one (2^-9 / 3^0.5 of a
    value, up to twice that near a power of two) is 0.02 of the norm, bounded
    by 0.04; a single element is bounded by 8 of these over its own size or the
    root mean square of its row or of its tensor's nonzero rows."""
    log(f"rollout segments={segments} against float64")
    case = {"kind": "rollout", "segments": segments, "layers": 1}
    out, ref = cases.run(cases.prepare(case, 3)), cases.exact(case, 3)
    assert torch.equal(out["exits"], ref["exits"])
    pairs = list(zip(out["logits"], ref["logits"])) + list(zip(out["grads"], ref["grads"]))
    for i, (got, want) in enumerate(pairs):
        got, want = got.double(), want.double()
        diff = got - want
        assert float(diff.norm()) <= 0.04 * float(want.norm()), i
        if want.dim() == 2:
            live = want.abs().amax(1) > 0
            assert not bool(got[~live].any()), i
            diff, want = diff[live], want[live]
        rms = want.pow(2).mean(-1, keepdim=True).sqrt().clamp(min=float(want.pow(2).mean().sqrt()))
        size = torch.maximum(want.abs(), rms)
        assert float((diff.abs() / size).max()) <= 8 * 0.04, i
    # a mean of float32 terms over the bf16 logits
    assert abs(float(out["loss"]) - float(ref["loss"])) <= 1e-3 * float(ref["loss"])
