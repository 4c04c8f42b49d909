"""int8 x int8 products of two to eight activation rows, which the kernel that holds them in LDS as one panel
and the v_dot4 kernel share between them: K at and beside the panel sizes, sizes on both sides of each line
of the rule, workgroups that walk over several column tiles, whole int8 range, exact to the bit; nothing is
written behind the result."""
import pytest
import torch

from fastgate_amd import capi
from helpers import ptr, stream_ptr

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N", [2048, 2304, 4096])
@pytest.mark.parametrize("K", (128, *[k + d for k in (2048, 4096, 6144, 8192, 12288, 16384) for d in (-128, 0, 128)]))
def test_panel_sizes_are_exact(device, N, K):
    g = torch.Generator(device=device)
    g.manual_seed(9600 + N + K)
    W = torch.randint(-128, 128, (N, K), generator=g, dtype=torch.int8, device=device)
    W64 = W.double().t()
    for M in range(2, 9):
        x = torch.randint(-128, 128, (M, K), generator=g, dtype=torch.int8, device=device)
        acc = torch.full((M + 1, N), -3, dtype=torch.int32, device=device)
        st = capi.lib().fg_gemv_i8i8_i32(ptr(W), ptr(x), ptr(acc), M, N, K, stream_ptr())
        assert st == capi.FG_OK
        want = (x.double() @ W64).round().int()  # below 2^53: exact
        assert torch.equal(acc[:M], want), (M, N, K)
        assert bool((acc[M] == -3).all())


# on 256 CUs the v_dot4 kernel runs, on three or four waves: two rows everywhere but at K = 2304; three rows at N=5120
# K=8192, N=8320 K=7808 and K > 8192; four at K > 8192.  The panel kernel has the rest
@pytest.mark.parametrize("N,K", [(2176, 2304), (2176, 4992), (3072, 6144), (4224, 9088), (5120, 5120), (2176, 8192),
                                 (5120, 8192), (8320, 7808), (5120, 9216), (2176, 10368), (3072, 11264)])
def test_few_rows_beside_the_panel_are_exact(device, N, K):
    # K that gives every wave of the v_dot4 kernel a piece, and K that does not
    g = torch.Generator(device=device)
    g.manual_seed(9700 + N + K)
    W = torch.randint(-128, 128, (N, K), generator=g, dtype=torch.int8, device=device)
    for M in (2, 3, 4):
        x = torch.randint(-128, 128, (M, K), generator=g, dtype=torch.int8, device=device)
        acc = torch.full((M + 1, N), -3, dtype=torch.int32, device=device)
        assert capi.lib().fg_gemv_i8i8_i32(ptr(W), ptr(x), ptr(acc), M, N, K, stream_ptr()) == capi.FG_OK
        assert torch.equal(acc[:M], (x.double() @ W.double().t()).round().int()), (M, N, K)
        assert bool((acc[M] == -3).all())


# both sides of every line between the panel, one piece a wave, and two pieces a wave
@pytest.mark.parametrize("N,K", [(8192, 2048), (8320, 2048), (14336, 512), (14336, 640), (28672, 1536), (28672, 1664),
                                 (16384, 2048), (16512, 2048), (8320, 7808), (9216, 8064), (9344, 8064), (3072, 4096), (2944, 4096), (3072, 4224), (4096, 6144),
                                 (4096, 6272), (4224, 4096), (8192, 4096), (16384, 4096), (8192, 7296), (8064, 8192),
                                 (8192, 8192), (12288, 11264), (12288, 11392), (12160, 11392), (12288, 12288),
                                 (2176, 12288), (2176, 12416)])
def test_lines_of_the_rule_are_exact(device, N, K):
    g = torch.Generator(device=device)
    g.manual_seed(9800 + N + K)
    W = torch.randint(-128, 128, (N, K), generator=g, dtype=torch.int8, device=device)
    W64 = W.double().t()
    for M in (2, 3, 4):
        x = torch.randint(-128, 128, (M, K), generator=g, dtype=torch.int8, device=device)
        acc = torch.full((M + 1, N), -3, dtype=torch.int32, device=device)
        assert capi.lib().fg_gemv_i8i8_i32(ptr(W), ptr(x), ptr(acc), M, N, K, stream_ptr()) == capi.FG_OK
        assert torch.equal(acc[:M], (x.double() @ W64).round().int()), (M, N, K)
        assert bool((acc[M] == -3).all())


# column tiles that a workgroup walks over (the last round partly filled; one to four workgroups a CU), and both sides
# of the rule's lines for five rows and more, for narrow outputs and for two rows
@pytest.mark.parametrize("N,K", [(128, 128), (33024, 256), (33024, 512), (17408, 640), (17408, 1024), (14464, 1152),
                                 (8320, 2048), (8320, 2176), (12416, 4096), (4224, 4224), (8320, 5248), (8320, 8064),
                                 (512, 4096), (1024, 4096), (1024, 4224), (896, 6144), (1024, 6272), (1536, 8192),
                                 (1408, 8192), (1536, 8320), (2048, 12416), (2176, 12416), (3584, 5120), (3456, 5120),
                                 (7168, 6144), (4224, 8192), (4224, 12288), (4224, 16384), (4224, 1152), (8320, 1536),
                                 (2176, 2560), (8320, 2432), (4224, 3072), (4224, 5120), (2176, 5120), (2176, 7168),
                                 (4224, 6272), (4096, 8320), (4096, 10240), (8192, 9344), (2176, 8320), (4224, 10240),
                                 (4224, 14336), (4224, 12416)])
def test_many_tiles_and_narrow_outputs_are_exact(device, N, K):
    g = torch.Generator(device=device)
    g.manual_seed(9850 + N + K)
    W = torch.randint(-128, 128, (N, K), generator=g, dtype=torch.int8, device=device)
    W64 = W.double().t()
    for M in range(2, 9):
        x = torch.randint(-128, 128, (M, K), generator=g, dtype=torch.int8, device=device)
        acc = torch.full((M + 1, N), -3, dtype=torch.int32, device=device)
        assert capi.lib().fg_gemv_i8i8_i32(ptr(W), ptr(x), ptr(acc), M, N, K, stream_ptr()) == capi.FG_OK
        assert torch.equal(acc[:M], (x.double() @ W64).round().int()), (M, N, K)
        assert bool((acc[M] == -3).all())
