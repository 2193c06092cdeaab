"""The bf16 head_dim-128 forward for few query tiles (32-row workgroups whose
waves share the keys) through the C ABI against float64 softmax attention of
the same bf16 values: dual-stream packs (segments and streams ending inside a
tile, several block sizes, grouped heads) and decoding windows after prefixes
of 0 to 3000 rows; output and log-sum-exp.

Bound: probabilities are rounded to bf16 for the second product (2^-8 of each
term), the output once more (2^-8 of the value): 2^-7 of the largest value of
unit-scale rows; the log-sum-exp is a float32 sum of float32 scores (1e-4)."""

import pytest
import torch

from alodlm_amd import _lib as L
from alodlm_amd.layers import DualStreamMask, WindowMask
from tests.helpers import log

pytestmark = pytest.mark.gpu
DEV, DH = "cuda", 128


def _check(q, k, v, shift_rows, mask, allowed, block):
    N, nq, nkv = q.shape[0], q.shape[1], k.shape[1]
    assert mask.tiles.shape[0] * nq < 256, "the case must take the few-tile kernel"
    o = torch.full_like(q, float("nan"))
    lse = torch.empty(nq, N, device=DEV)
    shift = shift_rows * nkv * DH * 2
    L.call("alodlm_attention_fwd", L.ptr(q), L.ptr(k) + shift, L.ptr(v) + shift, nkv * DH,
           L.ptr(mask.boundaries), L.ptr(mask.row_segment), L.ptr(mask.tiles),
           mask.tiles.shape[0], L.ptr(o), L.ptr(lse), N, nq, nkv, DH, block, L.BF16_CODE,
           torch.cuda.current_stream().cuda_stream)
    kf, vf = (t.double().repeat_interleave(nq // nkv, 1) for t in (k, v))
    s = torch.einsum("qhd,khd->hqk", q.double(), kf) * DH ** -0.5
    s = s.masked_fill(~allowed, float("-inf"))
    ref = torch.einsum("hqk,khd->qhd", torch.softmax(s, -1), vf)
    assert float((o.double() - ref).abs().max()) <= 2.0 ** -7 * float(ref.abs().max())
    assert float((lse.double() - torch.logsumexp(s, -1)).abs().max()) <= 1e-4


def _rand(rows, heads, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    return torch.randn(rows, heads, DH, generator=g, device=DEV).to(torch.bfloat16)


@pytest.mark.parametrize("lengths,block", [([1], 32), ([31, 2], 32), ([130, 33], 8), ([257], 64),
                                           ([100, 5, 64], 32)])
@pytest.mark.parametrize("nq,nkv", [(2, 1), (16, 8)])
def test_dual_stream(lengths, block, nq, nkv):
    log(f"few-tile attention lengths={lengths} block={block} heads={nq}/{nkv}")
    offsets = [0]
    for n in lengths:
        offsets.append(offsets[-1] + n)
    N = 2 * offsets[-1]
    mask = DualStreamMask(offsets, block, torch.device(DEV))
    _check(_rand(N, nq, 1), _rand(N, nkv, 2), _rand(N, nkv, 3), 0, mask, mask.dense(), block)


@pytest.mark.parametrize("prefix,window", [(0, 1), (0, 300), (7, 16), (128, 32), (3000, 27),
                                           (255, 130)])
@pytest.mark.parametrize("nq,nkv", [(4, 1), (16, 8)])
def test_window(prefix, window, nq, nkv):
    log(f"few-tile attention window prefix={prefix} rows={window} heads={nq}/{nkv}")
    mask = WindowMask(prefix, window, True, DEV, block_size=32)
    total = prefix + window
    q = _rand(mask.q_rows, nq, prefix + window)
    allowed = (torch.arange(total, device=DEV)
               <= torch.arange(total - mask.q_rows, total, device=DEV)[:, None])
    _check(q, _rand(total, nkv, 4), _rand(total, nkv, 5), mask.base, mask, allowed, 32)
