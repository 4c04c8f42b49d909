"""int8 weights against two to sixteen activation rows held in LDS as one panel: K at and below every panel size
and just beyond the largest of each row count, few and many column tiles a workgroup, every number of rows."""
import numpy as np
import pytest
import torch

import oracle
from fastgate_amd import capi
from helpers import assert_close_f16, gen, normal, ptr, stream_ptr

pytestmark = pytest.mark.gpu


def _run(Wd, x, scale, scalar_scale, zp, device):
    M, K = x.shape
    N = Wd.shape[0]
    y = torch.full((M + 1, N), 5.0, dtype=torch.half, device=device)  # a row behind the result stays as it is
    xd = x.to(device)
    capi.check(capi.lib().fg_gemv_w8a16(ptr(Wd), ptr(xd), ptr(scale), scalar_scale, zp, ptr(y), M, N, K, stream_ptr()),
               "fg_gemv_w8a16")
    torch.cuda.synchronize()
    assert bool((y[M] == 5.0).all())
    return y[:M].cpu()


# columns: under one tile a CU, one to two, a last round partly filled, several workgroups a CU
@pytest.mark.parametrize("K", [128, 512, 640, 1024, 1152, 1536, 2048, 2176, 2560, 3072, 3200, 4096, 4224, 5120, 5248, 6144,
                               6272, 7168, 7296, 8192, 8320])
@pytest.mark.parametrize("N", [2176, 4224, 9088, 17536])
def test_whole_numbers_are_exact(device, N, K):
    # |w + 128| < 256 and |x| <= 4: the magnitudes of a sum stay below 256 * 4 * 8320 < 2^24, so every partial sum and
    # the zero point's share (128 + 3) * sum of x are exact in fp32 in any order, the scales are powers of two, and the
    # only rounding is the last one
    g = torch.Generator(device=device)
    g.manual_seed(9700 + N + K)
    Wd = torch.randint(-128, 128, (N, K), generator=g, dtype=torch.int8, device=device)
    W = Wd.double().t().contiguous()
    scale = torch.pow(2.0, torch.randint(-3, 2, (N,), generator=g, device=device).float()).half()
    for M in (2, 3, 4, 5, 6, 8, 9, 13, 16):
        x = torch.randint(-4, 5, (M, K), generator=g, device=device).half()
        got = _run(Wd, x, scale, 2.0 ** -7, 3.0, device)
        xd = x.double()
        want = ((xd @ W - 3.0 * xd.sum(1, keepdim=True)) * scale.double() * 2.0 ** -7).half().cpu()
        assert torch.equal(got, want), (M, N, K)


@pytest.mark.parametrize("M", [3, 7, 16])
@pytest.mark.parametrize("N,K", [(2176, 2560), (8448, 4096)])
def test_real_and_broken_rows(device, M, N, K):
    g = gen(9800 + M + K)
    Wd = torch.randint(-128, 128, (N, K), generator=g, dtype=torch.int8).to(device)
    scale = (torch.rand(N, generator=g) * 0.009 + 0.001).half().to(device)
    x = normal((M, K), g)
    x[1, 5] = float("inf")
    x[2, K - 1] = float("nan")
    got = _run(Wd, x, scale, 0.5, 3.0, device).numpy()
    rows = [m for m in range(M) if m not in (1, 2)]
    cols = np.array([0, 1, 15, 16, 31, N // 2 + 7, N - 16, N - 1])
    ref, _ = oracle.gemv_w8a16(Wd.cpu().numpy()[cols], x.numpy()[rows], scale.cpu().numpy()[cols], 0.5, 3.0)
    assert_close_f16(got[rows][:, cols], ref, "finite rows")
    w = Wd[:, 5].cpu().numpy().astype(np.float32) - 3.0
    assert (np.isnan(got[1]) == (w == 0)).all() and (np.sign(got[1][w != 0]) == np.sign(w[w != 0])).all()
    assert np.isinf(got[1][w != 0]).all() and np.isnan(got[2]).all()


@pytest.mark.parametrize("unit", [2.0 ** -24, 32.0])  # subnormal activations; the largest halves
@pytest.mark.parametrize("M,N,K", [(2, 2176, 512), (4, 4224, 4096), (8, 2176, 5120), (16, 2176, 3072)])
def test_smallest_and_largest_activations_are_exact(device, M, N, K, unit):
    # 32 activations a row are not zero.  In units, |x| <= 2047: the magnitudes of w + 128 times x stay below
    # 32 * 2047 * 255 < 2^24, so every partial sum is exact in fp32 in any order
    g = gen(9900 + M + K + int(unit))
    Wd = torch.randint(-128, 128, (N, K), generator=g, dtype=torch.int8)
    scalar = 1.0 if unit < 1 else 2.0 ** -14
    m = torch.zeros((M, K), dtype=torch.int64)
    top = 511 if unit < 1 else 2047
    for row in range(M):
        at = torch.randperm(K, generator=g)[:32]
        m[row, at] = torch.randint(1, top + 1, (32,), generator=g) * (torch.randint(0, 2, (32,), generator=g) * 2 - 1)
    got = _run(Wd.to(device), (m.double() * unit).half(), None, scalar, 0.0, device).numpy()
    want = ((m.numpy() @ Wd.numpy().astype(np.int64).T) * (unit * scalar)).astype(np.float32).astype(np.float16)
    assert (want != 0).mean() > 0.99
    assert (got == want).all(), (M, N, K)
