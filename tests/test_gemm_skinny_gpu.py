"""Products of a few rows with an [out, in] weight (the decoder's windows)
through the C ABI against float64: both storage types, plain and residual
epilogues, at the edges of the 16-row blocks on both sides, of the K split
between waves and of the row limit above which the tile kernels take over.

Bounds: the float32 sum of K products errs by at most K eps sum|a||b|, in
practice by about sqrt(K) eps of its root mean square; a bf16 output adds half
a unit of its last place (2^-8 of the value) and, with a residual, a unit of
the rounded product's (2^-7), where its sum lies between two bf16 values."""

import pytest
import torch

from alodlm_amd import _lib as L
from tests.helpers import log

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("M,N,K", [
    (1, 16, 8), (5, 33, 40), (16, 4096, 2048), (16, 12304, 264), (17, 4112, 520),
    (32, 130, 2056), (33, 6144, 1032), (48, 2048, 6144), (49, 50, 4104), (64, 96, 1024),
    (65, 96, 1024), (9, 4130, 776), (20, 1000, 72), (48, 4096, 8200)])
@pytest.mark.parametrize("epi", [0, 1])
def test_few_rows(M, N, K, dtype, epi):
    log(f"gemm few rows M={M} N={N} K={K} {dtype} epi={epi}")
    g = torch.Generator().manual_seed(M * 131 + N + K)
    pad = 8  # row strides wider than the rows
    A = torch.randn(M, K + pad, generator=g).to(dtype).to(DEV)
    W = torch.randn(N, K + pad, generator=g).to(dtype).to(DEV)
    R = torch.randn(M, N, generator=g).to(dtype).to(DEV)
    C = torch.full((M, N), float("nan"), dtype=dtype, device=DEV)
    code = L.dtype_code(dtype)
    need = L.query("alodlm_gemm_workspace", M, N, K, epi, code)
    ws = torch.empty(max(need, 1), device=DEV)
    L.call("alodlm_gemm", L.ptr(A), K + pad, 1, L.ptr(W), K + pad, 1, L.ptr(C), N, L.ptr(R), N,
           M, N, K, 0.5, epi, code, L.ptr(ws), torch.cuda.current_stream().cuda_stream)
    ref = 0.5 * (A[:, :K].double() @ W[:, :K].double().T)
    if epi == 1:
        ref = R.double() + ref.to(dtype).double()
    err = (C.double() - ref).abs()
    eps = 2.0 ** -23 * K ** 0.5
    bound = 4 * eps * (0.5 * K ** 0.5)  # four standard deviations of the sum's error
    if dtype == torch.bfloat16:
        bound = bound + 2.0 ** -8 * ref.abs()
        if epi == 1:
            bound = bound + 2.0 ** -7 * (ref - R.double()).abs()
    assert bool((err <= bound + 1e-6).all()), float((err - bound).max())
