"""autoregressive_loss against torch's cross-entropy in float64: value (the
per-token terms in float32: 1e-5 of the value), gradient (float32: its
exponentials to 1e-5; bf16: half a unit of the last place, 2^-8 of the value),
exact zeros in every row without a target, logits left as they were, an
upstream factor, vocabularies on both row-kernel paths and off the 8-column
groups, ignored labels, segments of one token, more rows than one sweep of the
row selection, and a pack without a target."""

import pytest
import torch
import torch.nn.functional as F

from alodlm_amd.loss import autoregressive_loss
from tests.helpers import log

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("lengths,vocab", [([2], 16), ([5, 1, 9], 1003), ([300, 41, 700], 264),
                                           ([40, 3], 151936)])
def test_against_torch(lengths, vocab, dtype):
    log(f"autoregressive_loss lengths={lengths} vocab={vocab} {dtype}")
    offsets = [0]
    for n in lengths:
        offsets.append(offsets[-1] + n)
    N = 2 * offsets[-1]
    g = torch.Generator(device=DEV).manual_seed(N + vocab)
    logits = (2 * torch.randn(N, vocab, generator=g, device=DEV)).to(dtype)
    labels = torch.randint(0, vocab, (offsets[-1],), generator=g, device=DEV)
    if offsets[-1] > 2:
        labels[::5] = -100
    rows, targets = [], []
    for a, b in zip(offsets, offsets[1:]):
        for i in range(b - a - 1):
            if int(labels[a + 1 + i]) != -100:
                rows.append(2 * a + i)
                targets.append(int(labels[a + 1 + i]))
    ref_in = logits.double().requires_grad_(True)
    ref = F.cross_entropy(ref_in[rows], torch.tensor(targets, device=DEV))
    ref_grad = torch.autograd.grad(0.37 * ref, ref_in)[0]
    x = logits.clone().requires_grad_(True)
    loss = autoregressive_loss(x, labels, torch.tensor([2 * o for o in offsets], device=DEV))
    grad = torch.autograd.grad(0.37 * loss, x)[0]
    assert torch.equal(x.detach(), logits)
    assert abs(float(loss) - float(ref)) <= 1e-5 * abs(float(ref))
    # the stored softmax - onehot and its scaled copy are each rounded
    rel = 2 * 2.0 ** -8 if dtype == torch.bfloat16 else 1e-5
    err = (grad.double() - ref_grad).abs()
    assert bool((err <= rel * ref_grad.abs() + 1e-6 * ref_grad.abs().max()).all())
    other = torch.ones(N, dtype=torch.bool, device=DEV)
    other[rows] = False
    assert not bool(grad[other].any())


def test_no_target():
    log("autoregressive_loss without a target")
    logits = torch.randn(8, 24, device=DEV, requires_grad=True)
    labels = torch.full((4,), -100, device=DEV)
    loss = autoregressive_loss(logits, labels, torch.tensor([0, 2, 8], device=DEV))
    assert float(loss.detach()) == 0.0 and loss.requires_grad
