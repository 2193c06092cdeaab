"""The bf16 head_dim-128 forward on 128-row query tiles (packs and windows of 256
and more workgroups) through the C ABI against float64 softmax attention of the
same bf16 values: ragged dual-stream packs, whose tiles end inside a stream and
whose last keys are the pack's last rows, and wide decoding windows after
prefixes that are no multiple of the tile, whose cached keys lie at negative
rows; output and log-sum-exp.

Bound: probabilities are rounded to bf16 for the second product (2^-8 of each
term), the output once more (2^-8 of the value): 2^-7 of the largest value of
unit-scale rows; the log-sum-exp is a float32 sum of float32 scores (1e-4)."""

import pytest
import torch

from alodlm_amd import _lib as L
from alodlm_amd.layers import DualStreamMask, WindowMask
from tests.helpers import log
from tests.test_attention_few_gpu import _rand

pytestmark = pytest.mark.gpu
DEV, DH, NQ, NKV = "cuda", 128, 16, 8


def _check(q, k, v, shift_rows, mask, allowed, block):
    N = q.shape[0]
    assert mask.tiles.shape[0] * NQ >= 256, "the case must take the 128-row tiles"
    # rows beyond the pack are never read: they would spread
    pad = lambda t: torch.cat((t, torch.full_like(t[:64], float("nan"))))
    q, k, v = pad(q), pad(k), pad(v)
    o, lse = torch.full_like(q, 7.0), torch.empty(NQ, N, device=DEV)
    shift = shift_rows * NKV * DH * 2
    L.call("alodlm_attention_fwd", L.ptr(q), L.ptr(k) + shift, L.ptr(v) + shift, NKV * DH,
           L.ptr(mask.boundaries), L.ptr(mask.row_segment), L.ptr(mask.tiles),
           mask.tiles.shape[0], L.ptr(o), L.ptr(lse), N, NQ, NKV, DH, block, L.BF16_CODE,
           torch.cuda.current_stream().cuda_stream)
    assert bool((o[N:] == 7.0).all())
    for h in range(NQ):  # a head at a time: the scores are [rows, keys] in float64
        hk = h // (NQ // NKV)
        s = q[:N, h].double() @ k[:-64, hk].double().T * DH ** -0.5
        s = s.masked_fill(~allowed, float("-inf"))
        ref = torch.softmax(s, -1) @ v[:-64, hk].double()
        err = float((o[:N, h].double() - ref).abs().max())
        assert err <= 2.0 ** -7 * float(ref.abs().max()), h
        assert float((lse[h].double() - torch.logsumexp(s, -1)).abs().max()) <= 1e-4, h


@pytest.mark.parametrize("lengths,block", [([61, 402, 17, 757], 16), ([61, 402, 17, 757], 32),
                                           ([1000, 25], 64), ([1] * 12 + [129, 3], 32)])
def test_ragged_pack(lengths, block):
    log(f"128-row tiles, pack lengths={lengths} block={block}")
    offsets = [0]
    for n in lengths:
        offsets.append(offsets[-1] + n)
    N = 2 * offsets[-1]
    mask = DualStreamMask(offsets, block, torch.device(DEV))
    _check(_rand(N, NQ, 1), _rand(N, NKV, 2), _rand(N, NKV, 3), 0, mask, mask.dense(), block)


@pytest.mark.parametrize("prefix,window", [(77, 2100), (100, 1930), (0, 1921), (1, 2047),
                                           (300, 2048), (2500, 1985)])
def test_wide_window(prefix, window):
    log(f"128-row tiles, window prefix={prefix} rows={window}")
    mask = WindowMask(prefix, window, True, DEV, block_size=32)
    total = prefix + window
    allowed = (torch.arange(total, device=DEV)
               <= torch.arange(prefix, total, device=DEV)[:, None])
    _check(_rand(window, NQ, prefix), _rand(total, NKV, 4), _rand(total, NKV, 5), mask.base, mask,
           allowed, 32)
