"""The head_dim-128 bf16 q/k norm + rotary kernels driven by caller tables:
forward bit-equal to the same rows through the generic kernel (an unaligned
output takes it), backward within the bf16 rounding of its float32 sums, for
row counts on both sides of the head-group split and head counts that leave a
group part empty; tables whose two halves differ; adjacent and separate norm
gradients."""

import pytest
import torch

from alodlm_amd import _lib as L
from tests.helpers import log

pytestmark = pytest.mark.gpu
DEV, DH, EPS = "cuda", 128, 1e-6


def _inputs(rows, nq, nkv):
    g = torch.Generator(device=DEV).manual_seed(rows + nq)
    r = lambda *s: torch.randn(*s, generator=g, device=DEV).to(torch.bfloat16)
    return (r(rows, (nq + 2 * nkv) * DH), 1 + 0.1 * r(DH), 1 + 0.1 * r(DH), r(rows, DH), r(rows, DH),
            r(rows, nq * DH), r(rows, nkv * DH))


@pytest.mark.parametrize("rows", [1, 5, 300, 4097])
@pytest.mark.parametrize("nq,nkv", [(2, 1), (16, 8), (5, 5)])
def test_tables(rows, nq, nkv):
    log(f"rope tables rows={rows} heads={nq}/{nkv}")
    qkv, wq, wk, cos, sin, dq, dk = _inputs(rows, nq, nkv)
    st = torch.cuda.current_stream().cuda_stream
    outs = []
    for shift in (0, 1):  # an output one element off 16 bytes runs the generic kernel
        q = torch.empty(rows * nq * DH + 8, dtype=torch.bfloat16, device=DEV)[shift:]
        k = torch.empty(rows * nkv * DH + 8, dtype=torch.bfloat16, device=DEV)[shift:]
        L.call("alodlm_qknorm_rotary_fwd", L.ptr(qkv), L.ptr(wq), L.ptr(wk), L.ptr(cos),
               L.ptr(sin), L.ptr(q), L.ptr(k), rows, nq, nkv, DH, EPS, L.BF16_CODE, st)
        outs.append((q[:rows * nq * DH].clone(), k[:rows * nkv * DH].clone()))
    # the two kernels sum a head's squares in another order, so a normalised
    # value may round to the neighbouring bf16 (2^-7 of it), twice, which moves
    # its two products by as much
    heads = qkv.view(rows, nq + 2 * nkv, DH)[:, :nq + nkv].float()
    w = torch.cat((wq.float().expand(nq, DH), wk.float().expand(nkv, DH)))
    t = (w * heads * torch.rsqrt(heads.pow(2).mean(-1, keepdim=True) + EPS)).abs()
    swapped = torch.cat((t[..., DH // 2:], t[..., :DH // 2]), -1)
    bound = 2.0 ** -6 * (t * cos.float().abs()[:, None] + swapped * sin.float().abs()[:, None])
    for (a, b), limit, n in zip(zip(*outs), bound.split([nq, nkv], 1), (nq, nkv)):
        err = (a.float() - b.float()).abs().view(rows, n, DH)
        assert bool((err <= 2 * limit + 1e-6).all())
        assert float((a != b).float().mean()) < 0.02
    grads = []
    for shift in (0, 1):
        dqkv = torch.zeros(qkv.numel() + 8, dtype=torch.bfloat16, device=DEV)[shift:]
        gn = torch.zeros(2 * DH + 8, device=DEV)
        gq, gk = gn[:DH], (gn[DH:2 * DH] if shift == 0 else gn[DH + 4:2 * DH + 4])
        ws = torch.empty(L.query("alodlm_qknorm_rope_bwd_workspace", rows, nq, nkv, DH), device=DEV)
        L.call("alodlm_qknorm_rotary_bwd", L.ptr(dq), L.ptr(dk), L.ptr(qkv), L.ptr(wq), L.ptr(wk),
               L.ptr(cos), L.ptr(sin), L.ptr(dqkv), L.ptr(gq), L.ptr(gk), L.ptr(ws), rows, nq, nkv,
               DH, EPS, L.BF16_CODE, st)
        grads.append((dqkv[:qkv.numel()].view(rows, -1)[:, :(nq + nkv) * DH].float(), gq.clone(),
                      gk.clone()))
    (a, aq, ak), (b, bq, bk) = grads
    assert bool(((a - b).abs() <= 2.0 ** -7 * b.abs() + 2.0 ** -8 * b.abs().max()).all())
    for u, v in ((aq, bq), (ak, bk)):
        assert float((u - v).abs().max()) <= 2.0 ** -9 * float(v.abs().max()) + 1e-4
