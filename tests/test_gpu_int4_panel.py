"""int4 weights against two to four activation rows held in LDS as one panel: K at and beside the panel
sizes (and beyond the largest, where the row-load kernel takes over), one and several column tiles a
workgroup.  Single weights picked out come back exactly; sums are held to the oracle."""
import numpy as np
import pytest
import torch

import oracle
from fastgate_amd import capi
from helpers import assert_close_f16, gen, normal, ptr, stream_ptr

pytestmark = pytest.mark.gpu

PANELS = (2048, 4096, 6144, 8192, 12288, 16384)
KS = (128, *[k + d for k in PANELS for d in (-128, 0, 128)])


def _run(Wd, x, scale, scalar_scale, zp, device):
    M, K = x.shape
    N = Wd.shape[0]
    y = torch.full((M + 1, N), 5.0, dtype=torch.half, device=device)  # a row behind the result stays as it is
    xd = x.to(device)
    capi.check(capi.lib().fg_gemv_w4a16(ptr(Wd), ptr(xd), ptr(scale), scalar_scale, zp, ptr(y), M, N, K, stream_ptr()),
               "fg_gemv_w4a16")
    torch.cuda.synchronize()
    assert bool((y[M] == 5.0).all())
    return y[:M].cpu().numpy()


@pytest.mark.parametrize("K", KS)
@pytest.mark.parametrize("N", [2176, 7168])  # 136 tiles of 16 columns, one a workgroup; 448, more than CUs
def test_panel_sizes(device, N, K):
    g = torch.Generator(device=device)
    g.manual_seed(9300 + N + K)
    Wd = torch.randint(0, 256, (N, K // 2), generator=g, dtype=torch.uint8, device=device)
    W = Wd.cpu().numpy()
    scale = (torch.rand(N, generator=g, device=device) * 0.009 + 0.001).half()
    cols = np.array(sorted({0, 1, 15, 16, 31, 32, N // 2 + 7, N - 33, N - 16, N - 1}))
    for M in (2, 3, 4):
        x = normal((M, K), gen(9400 + M + K))
        got = _run(Wd, x, scale, 0.5, 7.5, device)
        ref, _ = oracle.gemv_w4a16(W[cols], x.numpy(), scale.cpu().numpy()[cols], 0.5, 7.5)
        assert_close_f16(got[:, cols], ref, "M=%d N=%d K=%d" % (M, N, K))
        # x = e_k: the output is the weight, at positions over a 128-k load and at the end of K
        for k in sorted({0, 1, 7, 8, 30, 63, 64, 127, K // 2 + 21, K - 97, K - 2, K - M}):
            if k < 0 or k + M > K:
                continue
            x = torch.zeros((M, K), dtype=torch.half)
            for m in range(M):
                x[m, k + m] = 1.0
            got = _run(Wd, x, None, 1.0, 8.0, device)
            for m in range(M):
                b = W[:, (k + m) // 2]
                want = (b >> 4 if (k + m) % 2 else b & 15).astype(np.float32) - 8.0
                assert (got[m].astype(np.float32) == want).all(), (M, K, k, m)


@pytest.mark.parametrize("N,K", [(2176, 4096), (7168, 6272)])
def test_broken_rows_stay_alone(device, N, K):
    g = gen(9500 + K)
    Wd = torch.randint(0, 256, (N, K // 2), generator=g, dtype=torch.uint8).to(device)
    x = normal((4, K), g)
    x[1, 5] = float("inf")
    x[3, K - 1] = float("nan")
    got = _run(Wd, x, None, 1.0, 8.0, device)
    ref, _ = oracle.gemv_w4a16(Wd.cpu().numpy()[:64], x.numpy()[[0, 2]], None, 1.0, 8.0)
    assert_close_f16(got[[0, 2]][:, :64], ref, "finite rows")
    w = (Wd[:, 2] >> 4).cpu().numpy().astype(np.float32) - 8.0  # k = 5: the high nibble of byte 2
    assert (np.isnan(got[1]) == (w == 0)).all() and (np.sign(got[1][w != 0]) == np.sign(w[w != 0])).all()
    assert np.isinf(got[1][w != 0]).all() and np.isnan(got[3]).all()


@pytest.mark.parametrize("unit", [2.0 ** -24, 32.0])  # subnormal activations up to 511 units; the largest halves
@pytest.mark.parametrize("N,K", [(2176, 512), (2176, 4096), (7168, 2048), (2176, 12288)])
def test_smallest_and_largest_activations_are_exact(device, N, K, unit):
    # 512 activations a row are not zero.  In units, |x| <= 2047 and weights below 16 keep the sum of all
    # magnitudes below 512 * 2047 * 15 < 2^24, so every partial sum is exact in fp32 in any order and the
    # only rounding is the last one
    g = gen(9900 + K + int(unit))
    Wd = torch.randint(0, 256, (N, K // 2), generator=g, dtype=torch.uint8)
    W = torch.stack((Wd & 15, Wd >> 4), dim=-1).flatten(1).numpy().astype(np.int64) - 8
    scalar = 1.0 if unit < 1 else 2.0 ** -14
    for M in (2, 3, 4):
        m = torch.zeros((M, K), dtype=torch.int64)
        top = 511 if unit < 1 else 2047
        for row in range(M):
            at = torch.randperm(K, generator=g)[:512]
            m[row, at] = torch.randint(1, top + 1, (512,), generator=g) * (torch.randint(0, 2, (512,), generator=g) * 2 - 1)
            m[row, at[:64]] = top
        x = (m.double() * unit).half()
        assert (x.double() / unit == m.double()).all()
        got = _run(Wd.to(device), x, None, scalar, 8.0, device)
        want = ((m.numpy() @ W.T) * (unit * scalar)).astype(np.float32).astype(np.float16)
        assert (want != 0).mean() > 0.99
        assert (got == want).all(), (M, N, K)


# tiles of 16 columns that a workgroup walks over: the last round partly filled, one to four workgroups a CU, every
# panel size (the largest shares its LDS between the waves' strips and their sums; 12288 with sixteen waves, where there
# are no more tiles than CUs, and with eight)
@pytest.mark.parametrize("N,K", [(33024, 128), (17408, 1024), (33024, 896), (8320, 1152), (12416, 2048), (8320, 2176),
                                 (8320, 4224), (8320, 8192), (4224, 12160), (8320, 12416), (4224, 16384), (4224, 2176),
                                 (2176, 3072), (2176, 4736), (4224, 5120), (8320, 4992), (2176, 8320), (4224, 10240),
                                 (2176, 12416), (4224, 14336), (4096, 11008), (3072, 12288), (24704, 1152), (2176, 4352),
                                 (8320, 4352)])
def test_many_tiles_a_workgroup_are_exact(device, N, K):
    # |x| <= 8 and weights below 16: every sum is a whole number below 2^24, the scale a power of two
    g = torch.Generator(device=device)
    g.manual_seed(9950 + N + K)
    Wd = torch.randint(0, 256, (N, K // 2), generator=g, dtype=torch.uint8, device=device)
    W = torch.stack((Wd & 15, Wd >> 4), dim=-1).flatten(1).double() - 8.0
    for M in (2, 3, 4):
        x = torch.randint(-8, 9, (M, K), generator=g, device=device).half()
        scale = torch.pow(2.0, torch.randint(-3, 2, (N,), generator=g, device=device).float()).half()
        got = _run(Wd, x, scale, 2.0 ** -6, 8.0, device)
        want = (x.double() @ W.t() * scale.double() * 2.0 ** -6).half().cpu().numpy()
        assert (got == want).all(), (M, N, K)
