"""float32 attention of head_dim 128 on the matrix cores: forward and backward
under the dual-stream mask (ragged segments, streams and segments crossing the
32-row tiles, grouped heads, several block sizes) through sparse_attention, and
the decoding window's form through the C ABI, against float64 softmax
attention.

Bound: scores are dots of 128 products and outputs weighted means, each a
float32 sum of unit-scale terms: 1e-5 of the largest value (at least 1) covers their
rounding (about 128 eps) with the exponential's (eps times the scores' size)."""

import pytest
import torch

from alodlm_amd import _lib as L
from alodlm_amd.attention import sparse_attention, sparse_plan
from alodlm_amd.layers import DualStreamMask, WindowMask
from tests.helpers import log

pytestmark = pytest.mark.gpu
DEV, DH = "cuda", 128


def _reference(q, k, v, allowed):
    group = q.shape[1] // k.shape[1]
    k, v = k.repeat_interleave(group, 1), v.repeat_interleave(group, 1)
    s = torch.einsum("qhd,khd->hqk", q, k) * DH ** -0.5
    p = torch.softmax(s.masked_fill(~allowed, float("-inf")), -1)
    return torch.einsum("hqk,khd->qhd", p, v)


def _close(got, ref):
    # terms of unit scale that may cancel exactly (one key: dQ = dK = 0)
    err = float((got.double().cpu() - ref).abs().max()) / max(1.0, float(ref.abs().max()))
    assert err <= 1e-5, err


@pytest.mark.parametrize("lengths,block", [([1], 32), ([31], 32), ([33, 5, 64], 32),
                                           ([17, 90], 8), ([200], 64)])
@pytest.mark.parametrize("nq,nkv", [(2, 1), (3, 3)])
def test_dual_stream(lengths, block, nq, nkv):
    log(f"f32 attention lengths={lengths} block={block} heads={nq}/{nkv}")
    offsets = [0]
    for n in lengths:
        offsets.append(offsets[-1] + n)
    N = 2 * offsets[-1]
    g = torch.Generator().manual_seed(N + nq)
    q, k, v, do = (torch.randn(N, h, DH, generator=g) for h in (nq, nkv, nkv, nq))
    plan = sparse_plan([2 * o for o in offsets], block, "sdpa")
    allowed = DualStreamMask(offsets, block, DEV).dense().cpu()
    leaves = [t.to(DEV).requires_grad_(True) for t in (q, k, v)]
    out = sparse_attention(*leaves, plan)
    out.backward(do.to(DEV))
    ref_leaves = [t.double().requires_grad_(True) for t in (q, k, v)]
    ref = _reference(*ref_leaves, allowed)
    ref.backward(do.double())
    _close(out.detach(), ref.detach())
    for leaf, r in zip(leaves, ref_leaves):
        _close(leaf.grad, r.grad)


@pytest.mark.parametrize("prefix,window", [(0, 1), (0, 40), (5, 16), (300, 16), (31, 33)])
def test_window(prefix, window):
    log(f"f32 attention window prefix={prefix} rows={window}")
    nq, nkv = 4, 2
    g = torch.Generator().manual_seed(prefix + window)
    q = torch.randn(window, nq, DH, generator=g)
    k, v = (torch.randn(prefix + window, nkv, DH, generator=g) for _ in range(2))
    mask = WindowMask(prefix, window, False, DEV, block_size=32)
    qd, kd, vd = q.to(DEV), k.to(DEV), v.to(DEV)
    o = torch.empty_like(qd)
    lse = torch.empty(nq, window, device=DEV)
    shift = mask.base * nkv * DH * 4
    L.call("alodlm_attention_fwd", L.ptr(qd), L.ptr(kd) + shift, L.ptr(vd) + shift, nkv * DH,
           L.ptr(mask.boundaries), L.ptr(mask.row_segment), None, 0, L.ptr(o), L.ptr(lse), window,
           nq, nkv, DH, 32, L.F32_CODE, torch.cuda.current_stream().cuda_stream)
    allowed = torch.arange(prefix + window) <= torch.arange(prefix, prefix + window)[:, None]
    _close(o, _reference(q.double(), k.double(), v.double(), allowed))


@pytest.mark.parametrize("which", ["q", "k", "v", "do"])
@pytest.mark.parametrize("value", [float("nan"), float("inf")])
def test_hidden_rows_take_no_part(which, value):
    """A row holding a NaN or infinity reaches only the rows that the mask lets
    see it: the outputs and query gradients of the other queries, and the key
    and value gradients of keys none of the reached queries sees, are those of
    a pack without it (within the float32 bound: the affected tiles are summed
    row by row).  Segments of one 32-row tile share it."""
    log(f"f32 attention with {value} in {which}")
    offsets, nq, nkv = [0, 33, 38, 102], 4, 2
    N = 2 * offsets[-1]
    g = torch.Generator().manual_seed(5)
    t = {n: torch.randn(N, h, DH, generator=g) for n, h in
         (("q", nq), ("k", nkv), ("v", nkv), ("do", nq))}
    plan = sparse_plan([2 * o for o in offsets], 8, "sdpa")
    allowed = DualStreamMask(offsets, 8, DEV).dense().cpu()

    def run(t):
        leaves = [t[n].to(DEV).requires_grad_(True) for n in ("q", "k", "v")]
        out = sparse_attention(*leaves, plan)
        out.backward(t["do"].to(DEV))
        return [out.detach().cpu()] + [x.grad.cpu() for x in leaves]
    clean = run(t)
    for row in (12, 20, 66, 75, 150, N - 1):  # clean and noisy rows of every segment
        bad = dict(t)
        bad[which] = t[which].clone()
        bad[which][row, :, 17] = value
        reached = allowed[:, row] if which in ("k", "v") else torch.arange(N) == row
        keys = ~allowed[reached].any(0)
        assert bool((~reached).any()) and bool(keys.any())
        for got, ref, rows in zip(run(bad), clean, (~reached, ~reached, keys, keys)):
            assert bool(got[rows].isfinite().all()), (row, value)
            _close(got[rows], ref[rows].double())


def test_window_rows_before_a_bad_one():
    """A window row whose value is not finite leaves the rows before it alone."""
    log("f32 attention window with infinite later rows")
    nq, nkv, prefix, window = 4, 2, 21, 24
    g = torch.Generator().manual_seed(9)
    q = torch.randn(window, nq, DH, generator=g)
    k, v = (torch.randn(prefix + window, nkv, DH, generator=g) for _ in range(2))
    allowed = torch.arange(prefix + window) <= torch.arange(prefix, prefix + window)[:, None]
    ref = _reference(q.double(), k.double(), v.double(), allowed)
    v[prefix + 10] = float("inf")
    mask = WindowMask(prefix, window, False, DEV, block_size=32)
    qd, kd, vd = q.to(DEV), k.to(DEV), v.to(DEV)
    o, lse = torch.empty_like(qd), torch.empty(nq, window, device=DEV)
    shift = mask.base * nkv * DH * 4
    L.call("alodlm_attention_fwd", L.ptr(qd), L.ptr(kd) + shift, L.ptr(vd) + shift, nkv * DH,
           L.ptr(mask.boundaries), L.ptr(mask.row_segment), None, 0, L.ptr(o), L.ptr(lse), window,
           nq, nkv, DH, 32, L.F32_CODE, torch.cuda.current_stream().cuda_stream)
    _close(o[:10], ref[:10])
    assert not bool(o[10:].isfinite().any())
