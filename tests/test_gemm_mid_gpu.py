"""The 128-column-tile bf16 products (128, 64 or 32 tile rows) through the C ABI
against float64, at the edges of the tiles, of the 32-deep k stages (any K for
m/n-contiguous operands: rows past K must read as zeros, also where memory
after the operand holds NaN) and of the K splits, every epilogue.

Bounds: float outputs 4 sqrt(K) eps of the sum's root mean square (the float32
accumulation's rounding); a bf16 output adds half a unit of its last place
(2^-8 of the value) and, with a residual, a unit of the rounded product's
(2^-7)."""

import pytest
import torch

from alodlm_amd import _lib as L
from tests.helpers import log

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _operand(rows, K, kmajor, g):
    """rows x K values stored k- or row-contiguous with NaN after the last
    element."""
    t = torch.randn(rows, K, generator=g).to(torch.bfloat16)
    flat = (t if kmajor else t.T).contiguous().flatten()
    buf = torch.full((flat.numel() + 65536,), float("nan"), dtype=torch.bfloat16)
    buf[:flat.numel()] = flat
    return t, buf.to(DEV), K if kmajor else rows


@pytest.mark.parametrize("M,N,K,ak,bk", [
    (17, 136, 64, 1, 1), (32, 128, 32, 1, 0), (33, 264, 2048, 1, 1), (64, 2048, 6144, 1, 0),
    (65, 136, 96, 1, 1), (128, 128, 992, 1, 0), (150, 2048, 4096, 1, 1), (777, 520, 2048, 1, 1),
    (300, 2048, 6144, 1, 0), (2474, 2048, 12288, 1, 0), (136, 40, 33, 0, 0), (256, 264, 1, 0, 0),
    (512, 384, 301, 0, 0), (2048, 1024, 2474, 0, 0), (264, 136, 2048, 0, 1)])
@pytest.mark.parametrize("epi", [0, 1, 2, 3])
def test_products(M, N, K, ak, bk, epi):
    log(f"gemm 128-tile M={M} N={N} K={K} ak={ak} bk={bk} epi={epi}")
    g = torch.Generator().manual_seed(M + N + K + epi)
    A, Ad, lda = _operand(M, K, ak, g)
    B, Bd, ldb = _operand(N, K, bk, g)
    R = torch.randn(M, N, generator=g).to(torch.bfloat16).to(DEV)
    half = epi in (0, 1)
    C = torch.randn(M, N, generator=g).to(torch.bfloat16 if half else torch.float32).to(DEV)
    prod = 0.5 * (A.to(DEV).double() @ B.to(DEV).double().T)
    ref = prod
    if epi == 1:
        ref = R.double() + prod.to(torch.bfloat16).double()
    elif epi == 2:
        ref = C.double() + prod
    bound = 4 * 2.0 ** -23 * K ** 0.5 * (0.5 * K ** 0.5) + 2.0 ** -22 * ref.abs()
    if half:
        bound = bound + 2.0 ** -8 * ref.abs()
    if epi == 1:
        bound = bound + 2.0 ** -7 * prod.abs()
    need = L.query("alodlm_gemm_workspace", M, N, K, epi, L.BF16_CODE)
    for ws in (torch.full((max(need, 1),), float("nan"), device=DEV), None):
        out = C.clone()
        L.call("alodlm_gemm", L.ptr(Ad), lda, ak, L.ptr(Bd), ldb, bk, L.ptr(out), N, L.ptr(R), N,
               M, N, K, 0.5, epi, L.BF16_CODE, L.ptr(ws),
               torch.cuda.current_stream().cuda_stream)
        err = (out.double() - ref).abs()
        assert bool((err <= bound + 1e-6).all()), float((err - bound).max())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("epi", [0, 1, 2, 3])
@pytest.mark.parametrize("ak,bk", [(0, 0), (1, 1)])
def test_empty_sum(epi, ak, bk, dtype):
    """K = 0 (the weight gradient of no rows): zeros are stored, the residual is
    copied, an accumulated output stays."""
    log(f"gemm K=0 ak={ak} bk={bk} epi={epi} {dtype}")
    M, N = 264, 136
    f32 = epi in (L.EPI_ACCUM, L.EPI_STORE_F32)
    C = torch.randn(M, N, device=DEV).to(torch.float32 if f32 else dtype)
    R, before = torch.randn(M, N, device=DEV).to(dtype), C.clone()
    A, B = torch.zeros(8, device=DEV, dtype=dtype), torch.zeros(8, device=DEV, dtype=dtype)
    L.call("alodlm_gemm", L.ptr(A), 8 if ak else M, ak, L.ptr(B), 8 if bk else N, bk, L.ptr(C), N,
           L.ptr(R), N, M, N, 0, 1.0, epi, L.dtype_code(dtype), None,
           torch.cuda.current_stream().cuda_stream)
    want = R if epi == L.EPI_RESIDUAL else before if epi == L.EPI_ACCUM else torch.zeros_like(C)
    assert torch.equal(C, want)
