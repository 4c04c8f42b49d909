"""Equal activation rows of one call give equal bits wherever in the call they lie, whatever kernel the library
chooses: every number of rows at which it changes, both fp16 layouts, int8 and int4 weights, real-valued data."""
import pytest
import torch

from fastgate_amd import capi
from helpers import capi_gemm, ptr, stream_ptr

pytestmark = pytest.mark.gpu

SIZES = [(1024, 4096), (2048, 2048), (5120, 5120), (8192, 2048), (4864, 8320), (1152, 16384)]


def _rows(M, K, g, device):
    A = torch.randn((3, K), generator=g, device=device).half()
    pick = torch.arange(M, device=device) % 3
    return A[pick].contiguous(), pick


@pytest.mark.parametrize("layout", [capi.FG_W_KN, capi.FG_W_NK])
@pytest.mark.parametrize("N,K", SIZES)
def test_fp16(device, layout, N, K):
    g = torch.Generator(device=device)
    g.manual_seed(9990 + N + K)
    W = (torch.randn((K, N) if layout == capi.FG_W_KN else (N, K), generator=g, device=device) * 0.02).half()
    for M in (4, 5, 8, 9, 16, 17, 31, 33, 48, 65, 100, 129, 160, 256, 520):
        A, pick = _rows(M, K, g, device)
        C = torch.empty((M, N), dtype=torch.half, device=device)
        capi_gemm(A, W, C, layout)
        assert torch.equal(C, C[:3][pick]), (M, capi.plan(M, N, K, layout).as_dict())


@pytest.mark.parametrize("bits,most", [(8, 16), (4, 4)])
@pytest.mark.parametrize("N,K", SIZES)
def test_quantised_weights(device, bits, most, N, K):
    g = torch.Generator(device=device)
    g.manual_seed(9995 + N + K)
    W = torch.randint(-128, 128, (N, K * bits // 8), generator=g, device=device, dtype=torch.int8)
    scale = (torch.rand(N, generator=g, device=device) * 0.009 + 0.001).half()
    run = capi.lib().fg_gemv_w8a16 if bits == 8 else capi.lib().fg_gemv_w4a16
    for M in range(4, most + 1):
        x, pick = _rows(M, K, g, device)
        y = torch.empty((M, N), dtype=torch.half, device=device)
        capi.check(run(ptr(W), ptr(x), ptr(scale), 1.0, 3.0, ptr(y), M, N, K, stream_ptr()), "gemv")
        assert torch.equal(y, y[:3][pick]), M
