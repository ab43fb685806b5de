"""GPU tests of the few-row projections (cvh_gemv_bf16_*): against float64 at the bound of the GEMM tests, and
their fused layer boundaries against the plain projection followed by the standalone kernels, bit for bit."""
import pytest
import torch

from cppvllm_amd import _lib, ops
from tests.test_gpu_gemm import _check, _inputs
from tests._util import say

pytestmark = pytest.mark.gpu
DEV = "cuda"
BF = torch.bfloat16


def _gain(n, seed):
    return (torch.rand((n,), generator=torch.Generator().manual_seed(seed)) + 0.5).to(BF).to(DEV)


def _eq(a, b):
    assert torch.equal(a.view(torch.int16), b.view(torch.int16))


@pytest.mark.parametrize("M", [1, 2, 3, 4])
@pytest.mark.parametrize("N,K", [(16, 512), (4096, 1024), (48, 1536), (96, 2048)])
def test_norm_linear_rows(M, N, K):
    """rms_norm + projection: the normed rows are cvh_rms_norm's, the products within the GEMM bound of
    float64; columns do not depend on the width of the matrix (a slice of it gives the same bits)."""
    say(f"norm_linear_rows M={M} N={N} K={K}")
    x, w = _inputs(M, N, K, M + N + K)
    x *= 3.0
    xd, wd, gain = x.to(DEV), w.to(DEV), _gain(K, K)
    y = torch.full((M, N), float("nan"), dtype=BF, device=DEV)
    ops.norm_linear_rows(y, xd, gain, 1e-6, wd)
    xn = torch.empty_like(xd)
    ops.fused.rms_norm(xn, xd, gain, 1e-6)
    torch.cuda.synchronize()
    _check(y, xn, w)
    y16 = torch.empty((M, 16), dtype=BF, device=DEV)
    ops.norm_linear_rows(y16, xd, gain, 1e-6, wd[-16:].contiguous())
    torch.cuda.synchronize()
    _eq(y16, y[:, -16:].contiguous())


@pytest.mark.parametrize("M", [1, 2, 3, 4])
@pytest.mark.parametrize("N,K", [(16, 512), (1024, 2048), (1024, 3072), (80, 4096), (32, 2560)])
def test_linear_residual_rows(M, N, K):
    """From a zero residual the result is the projection within the GEMM bound of float64; from any other it is
    that projection through cvh_add_rms_norm's residual add, bit for bit."""
    say(f"linear_residual_rows M={M} N={N} K={K}")
    x, w = _inputs(M, N, K, M + N + K)
    xd, wd = x.to(DEV), w.to(DEV)
    y = torch.zeros((M, N), dtype=BF, device=DEV)
    ops.linear_residual_rows(y, xd, wd)
    resid = (torch.randn((M, N), generator=torch.Generator().manual_seed(7)) * 2).to(BF).to(DEV)
    want = resid.clone()
    ops.fused.add_rms_norm(want, y, torch.ones(N, dtype=BF, device=DEV), torch.empty_like(y), 1e-6)
    ops.linear_residual_rows(resid, xd, wd)
    torch.cuda.synchronize()
    _check(y, x, w)
    _eq(resid, want)


@pytest.mark.parametrize("M", [1, 2, 3, 4])
@pytest.mark.parametrize("I,K", [(16, 512), (3072, 1024), (48, 2048)])
def test_norm_linear_swiglu_rows(M, I, K):
    """Equal to norm_linear_rows over the interleaved weight followed by cvh_swiglu, bit for bit."""
    say(f"norm_linear_swiglu_rows M={M} I={I} K={K}")
    x, w = _inputs(M, 2 * I, K, M + I + K)
    wi, xd, gain = ops.interleave_gate_up(w).to(DEV), x.to(DEV), _gain(K, K)
    act = torch.full((M, I), float("nan"), dtype=BF, device=DEV)
    ops.norm_linear_swiglu_rows(act, xd, gain, 1e-6, wi)
    gu = torch.empty((M, 2 * I), dtype=BF, device=DEV)
    ops.norm_linear_rows(gu, xd, gain, 1e-6, wi)
    want = torch.empty_like(act)
    ops.fused.swiglu(want, ops.deinterleave_gate_up(gu.t().contiguous()).t().contiguous())
    torch.cuda.synchronize()
    _eq(act, want)


def test_unsupported_shapes():
    s = torch.cuda.current_stream().cuda_stream
    t = torch.zeros((8, 8192), dtype=BF, device=DEV)
    p = t.data_ptr()
    L = _lib.lib()
    for M, N, K in ((5, 16, 512), (1, 8, 512), (1, 16, 768), (1, 16, 4608)):
        assert L.cvh_gemv_bf16_residual(p, p, p, M, N, K, s) == _lib.CVH_ERR_UNSUPPORTED
    assert L.cvh_gemv_bf16_norm(p, p, p, 1e-6, p, 1, 16, 2560, s) == _lib.CVH_ERR_UNSUPPORTED
    assert L.cvh_gemv_bf16_norm_swiglu(p, p, p, 1e-6, p, 1, 24, 512, s) == _lib.CVH_ERR_UNSUPPORTED
    assert L.cvh_gemv_bf16_norm(p, p, None, 1e-6, p, 1, 16, 512, s) == _lib.CVH_ERR_INVALID_ARG
    assert L.cvh_gemv_bf16_residual(p, p, p, 0, 16, 512, s) == _lib.CVH_OK
