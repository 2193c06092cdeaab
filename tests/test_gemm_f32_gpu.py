"""The float32 matrix-core products through the C ABI against float64: every
operand layout and epilogue at the edges of the 64x64 and 128x128 tiles (2044
x 1924: one round of the large ones) and their 32- and 16-deep k stages, split
and unsplit K, row strides wider than the rows.

Bound: a float32 sum of K products of unit normals errs by at most K eps times
the sum's absolute terms; in practice the partial sums grow like sqrt(k), which
gives sqrt(K) eps sqrt(K): four of those standard deviations are allowed."""

import pytest
import torch

from alodlm_amd import _lib as L
from tests.helpers import log

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("M,N,K", [(72, 4, 4), (68, 132, 20), (128, 128, 16), (132, 260, 36),
                                   (256, 128, 1000), (700, 384, 2048), (2048, 516, 700),
                                   (2044, 1924, 52)])
@pytest.mark.parametrize("ak,bk", [(1, 1), (1, 0), (0, 1), (0, 0)])
@pytest.mark.parametrize("epi", [0, 1, 2, 3])
def test_float32_products(M, N, K, ak, bk, epi):
    log(f"gemm f32 M={M} N={N} K={K} ak={ak} bk={bk} epi={epi}")
    g = torch.Generator().manual_seed(M + N + K)
    A = torch.randn(M, K, generator=g).to(DEV)
    B = torch.randn(N, K, generator=g).to(DEV)
    wide = lambda t: torch.nn.functional.pad(t, (0, 4)).contiguous()
    Ad, Bd = wide(A if ak else A.T), wide(B if bk else B.T)
    R = torch.randn(M, N, generator=g).to(DEV)
    C = torch.randn(M, N, generator=g).to(DEV)
    ref = 0.5 * (A.double() @ B.double().T)
    if epi in (1, 2):
        ref = ref + (R if epi == 1 else C).double()
    need = L.query("alodlm_gemm_workspace", M, N, K, epi, L.F32_CODE)
    outs = []
    for ws in (torch.empty(max(need, 1), device=DEV), None):
        out = C.clone()
        L.call("alodlm_gemm", L.ptr(Ad), Ad.shape[1], ak, L.ptr(Bd), Bd.shape[1], bk, L.ptr(out),
               N, L.ptr(R), N, M, N, K, 0.5, epi, L.F32_CODE, L.ptr(ws),
               torch.cuda.current_stream().cuda_stream)
        err = float((out.double() - ref).abs().max())
        bound = 4 * 2.0 ** -24 * (K ** 0.5) * (K ** 0.5) + 2.0 ** -23 * float(ref.abs().max())
        assert err <= bound, (err, bound)
