"""The kernel for more than 16 activation rows, through the library's plans and through forced splits and
completions: rows at and beside the edges of its row blocks, columns and K that leave a last tile, an odd
number of steps and fewer steps than splits.  Every output against an fp32 product on the device,
a spread of columns against the oracle, whole numbers bit for bit."""
import ctypes

import numpy as np
import pytest
import torch

import oracle
from fastgate_amd import capi
from helpers import ATOL, RTOL, assert_close_f16, capi_gemm, make_plan, ptr, stream_ptr

pytestmark = pytest.mark.gpu

KN, NK = capi.FG_W_KN, capi.FG_W_NK
EDGES = (17, 32, 33, 64, 65, 96, 97, 128, 129, 255, 256, 300)


def _inputs(M, N, K, layout, device, whole=False, seed=0):
    g = torch.Generator(device=device)
    g.manual_seed(9000 + seed + M + N + K)
    if whole:
        A = torch.randint(-2, 3, (M, K), generator=g, device=device).half()
        W = torch.randint(-3, 4, (K, N) if layout == KN else (N, K), generator=g, device=device).half()
    else:
        A = torch.randn((M, K), generator=g, device=device).half()
        W = (torch.randn((K, N) if layout == KN else (N, K), generator=g, device=device) * 0.02).half()
    return A, W


def _product(A, W, layout):
    return A.float() @ (W.float() if layout == KN else W.float().t())


def _close(C, ref32, what):
    assert torch.isfinite(C).all(), what
    worst = ((C.float() - ref32).abs() - (ATOL + RTOL * ref32.abs())).max().item()
    assert worst <= 0.0, "%s: %.4g beyond the tolerance" % (what, worst)


@pytest.mark.parametrize("layout", [KN, NK])
@pytest.mark.parametrize("N,K", [(2048, 2176), (8320, 640), (1152, 4224), (33024, 512), (4096, 11008)])
def test_rows_at_the_edges_of_the_row_blocks(device, layout, N, K):
    for M in EDGES:
        A, W = _inputs(M, N, K, layout, device)
        out = torch.full((M + 1, N), -7.0, dtype=torch.half, device=device)  # a row behind C that stays as it is
        p = capi_gemm(A, W, out[:M], layout)
        what = "M=%d N=%d K=%d layout=%d %s" % (M, N, K, layout, p.as_dict())
        _close(out[:M], _product(A, W, layout), what)
        assert bool((out[M] == -7.0).all()), what
        if M in (33, 129):
            cols = torch.tensor(sorted({0, 1, 63, 64, 127, N // 2 + 5, N - 65, N - 1}), device=device)
            sub = (W[:, cols].t() if layout == KN else W[cols]).contiguous().cpu().numpy()
            ref, _ = oracle.gemm_f16(A.cpu().numpy(), sub, oracle.W_NK)
            assert_close_f16(out[:M][:, cols].cpu().numpy(), ref, what)


@pytest.mark.parametrize("layout", [KN, NK])
@pytest.mark.parametrize("M", [33, 96, 130])
def test_splits_and_completions_agree(device, layout, M):
    # whole numbers: every split and completion gives the exact sum; 40 splits leave workgroups without a step
    N, K = 1920, 2304
    A, W = _inputs(M, N, K, layout, device, whole=True)
    exact = _product(A, W, layout).half()
    for splitk in (1, 2, 5, 17, 40):
        for fused in ((0, 1, 2, 3) if layout == KN else (0, 1, 2)):
            p = capi.plan(M, N, K, layout, splitk)
            if fused == 2 and (splitk > 31 or M * N > 262144):
                continue
            if fused == 3 and splitk > 32:
                continue
            p.fused = fused
            C = torch.full((M, N), float("nan"), dtype=torch.half, device=device)
            for _ in range(2):  # the second call finds the header as the first left it
                capi_gemm(A, W, C, layout, plan=p)
                assert torch.equal(C, exact), (splitk, fused)
    # two passes and the counters add the same partials in the same order
    A, W = _inputs(M, N, K, layout, device, seed=1)
    got = []
    for fused in (0, 1):
        p = capi.plan(M, N, K, layout, 3)
        p.fused = fused
        got.append(torch.empty((M, N), dtype=torch.half, device=device))
        capi_gemm(A, W, got[-1], layout, plan=p)
    assert torch.equal(got[0], got[1])


@pytest.mark.parametrize("layout", [KN, NK])
@pytest.mark.parametrize("splitk", [1, 3])
def test_accumulate_bias_activation_and_pitch(device, layout, splitk):
    M, N, K = 70, 1664, 2688
    L = capi.lib()
    A, W = _inputs(M, N, K, layout, device)
    ref = _product(A, W, layout)
    C0 = torch.randn((M, N), device=device).half()
    C = C0.clone()
    capi_gemm(A, W, C, layout, accumulate=True, splitk=splitk)
    _close(C, ref + C0.float(), "accumulate")
    bias = torch.randn(N, device=device).half()
    ws = torch.zeros(capi.plan(M, N, K, layout, splitk).workspace_bytes + 16, dtype=torch.uint8, device=device)
    st = L.fg_gemm_f16_bias_act(ptr(A), ptr(W), ptr(bias), 4, ptr(C), M, N, K, layout, splitk, None, ptr(ws),
                                ws.numel(), stream_ptr())
    assert st == capi.FG_OK
    _close(C, torch.nn.functional.silu(ref + bias.float()), "bias and silu")
    if layout == KN:
        dense = torch.empty_like(C)
        capi_gemm(A, W, dense, layout, splitk=splitk)
        wide = torch.full((K, N + 136), float("nan"), dtype=torch.half, device=device)
        wide[:, :N] = W
        st = L.fg_gemm_f16_pitched(ptr(A), ptr(wide), ptr(C), M, N, K, N + 136, 0, splitk, ptr(ws), ws.numel(),
                                   stream_ptr())
        assert st == capi.FG_OK and torch.equal(C, dense)


@pytest.mark.parametrize("layout", [KN, NK])
def test_infinities_and_nan_stay_in_their_rows(device, layout):
    M, N, K = 50, 2048, 2304
    A, W = _inputs(M, N, K, layout, device)
    A[3, 100] = float("inf")
    A[49, K - 1] = float("nan")
    C = torch.empty((M, N), dtype=torch.half, device=device)
    capi_gemm(A, W, C, layout)
    ref = _product(A, W, layout)
    col = (W[100] if layout == KN else W[:, 100]) != 0
    assert bool(torch.isinf(C[3][col]).all()) and bool((torch.sign(C[3][col].float()) == torch.sign(ref[3][col])).all())
    assert bool(torch.isnan(C[49]).all())
    rest = [m for m in range(M) if m not in (3, 49)]
    _close(C[rest], ref[rest], "rows beside them")


@pytest.mark.parametrize("layout", [KN, NK])
def test_replayed_graph_gives_the_eager_result(device, layout):
    M, N, K = 48, 2048, 4352
    A, W = _inputs(M, N, K, layout, device)
    C, want = (torch.empty((M, N), dtype=torch.half, device=device) for _ in range(2))
    p = capi.plan(M, N, K, layout)
    assert p.splitk > 1
    ws = torch.zeros(p.workspace_bytes, dtype=torch.uint8, device=device)

    def call(out):
        st = capi.lib().fg_gemm_f16_planned(ptr(A), ptr(W), ptr(out), M, N, K, layout, 0, ctypes.byref(p), ptr(ws),
                                            ws.numel(), stream_ptr())
        capi.check(st, "fg_gemm_f16_planned")

    call(C)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        call(C)
    for i in range(4):
        A.copy_(torch.randn((M, K), device=device).half())
        C.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        call(want)
        assert torch.equal(C, want), i


@pytest.mark.parametrize("M", [33, 65])
def test_nk_rows_of_16_mi_elements(device, M):
    # a row of W is 32 MiB, a tile's rows together more than 2 GiB; -1, 0 and 1 keep every partial sum a
    # whole number below 2^24, exact in fp32 in any order
    N, K = 128, 1 << 24
    g = torch.Generator(device=device)
    g.manual_seed(9100 + M)
    A = torch.randint(-1, 2, (M, K), generator=g, dtype=torch.int8, device=device).half()
    W = torch.randint(-1, 2, (N, K), generator=g, dtype=torch.int8, device=device).half()
    want = torch.zeros((M, N), device=device)
    for k in range(0, K, 1 << 20):
        want += A[:, k:k + (1 << 20)].float() @ W[:, k:k + (1 << 20)].float().t()
    C = torch.full((M + 1, N), -7.0, dtype=torch.half, device=device)
    for splitk in (0, 1):
        capi_gemm(A, W, C[:M], NK, splitk=splitk)
        assert torch.equal(C[:M], want.half()), splitk
        assert bool((C[M] == -7.0).all())


@pytest.mark.parametrize("M", [33, 130])
def test_rows_32_mib_apart_give_the_dense_result(device, M):
    # a pitch whose offsets over the rows of a step leave 32 bits: the same tile, split and order of sums
    N, K, ldw = 8320, 640, 1 << 24
    A, W = _inputs(M, N, K, KN, device)
    wide = torch.empty((K - 1) * ldw + N, dtype=torch.half, device=device)
    torch.as_strided(wide, (K, N), (ldw, 1)).copy_(W)
    ws = torch.zeros(1 << 26, dtype=torch.uint8, device=device)
    for splitk in (0, 1, 2, 7):  # seven splits of five or ten steps: some have one step, some two
        dense = torch.empty((M, N), dtype=torch.half, device=device)
        p = capi_gemm(A, W, dense, KN, splitk=splitk)
        assert p.workspace_bytes <= ws.numel()
        _close(dense, _product(A, W, KN), "dense")
        C = torch.full((M, N), float("nan"), dtype=torch.half, device=device)
        st = capi.lib().fg_gemm_f16_pitched(ptr(A), ptr(wide), ptr(C), M, N, K, ldw, 0, splitk, ptr(ws), ws.numel(),
                                            stream_ptr())
        assert st == capi.FG_OK and torch.equal(C, dense), splitk


def test_16_mi_columns(device):
    # dense [K,N] weights as far apart: windows of columns against the product
    M, N, K = 17, 1 << 24, 512
    g = torch.Generator(device=device)
    g.manual_seed(9200)
    A = torch.randint(-2, 3, (M, K), generator=g, device=device).half()
    W = torch.empty((K, N), dtype=torch.half, device=device)
    for k in range(0, K, 64):
        W[k:k + 64] = torch.randint(-3, 4, (64, N), generator=g, dtype=torch.int8, device=device)
    C = torch.full((M, N), float("nan"), dtype=torch.half, device=device)
    capi_gemm(A, W, C, KN)
    for n in range(0, N, 1 << 21):
        assert torch.equal(C[:, n:n + (1 << 21)], _product(A, W[:, n:n + (1 << 21)], KN).half()), n


def _form(p):
    return p.stagger - 2  # include/fastgate.h: 2 + the number of the tile


FORMS = range(7)


@pytest.mark.parametrize("layout", [KN, NK])
@pytest.mark.parametrize("form", FORMS)
def test_every_form_at_the_edges_of_its_rows(device, layout, form):
    # whole numbers, so every form and split gives the exact sum; 40 splits of 33 steps or fewer leave
    # workgroups without a step
    N, K = 1280, 2176
    for M in (17, 31, 32, 33, 63, 65, 95, 97, 127, 129, 300):
        A, W = _inputs(M, N, K, layout, device, whole=True)
        exact = _product(A, W, layout).half()
        for splitk in (1, 3, 40):
            p = make_plan(capi.FG_KERNEL_KN_MFMA, tile_n=128, m_block=16, waves=8, splitk=splitk, stagger=2 + form) if \
                layout == KN else make_plan(capi.FG_KERNEL_NK_MFMA_R, tile_n=64, m_block=32, waves=8, splitk=splitk,
                                            stagger=2 + form, band=128)
            C = torch.full((M + 1, N), -7.0, dtype=torch.half, device=device)
            capi_gemm(A, W, C[:M], layout, plan=p)
            assert _form(p) == form  # kept: the tile fits the shape
            assert torch.equal(C[:M], exact), (M, splitk)
            assert bool((C[M] == -7.0).all())


# the library's own plans, one at least for every form of either layout
LIBRARY = [(KN, 31, 11008, 1024, 0), (KN, 24, 14336, 3072, 1), (KN, 64, 6144, 4096, 2), (KN, 96, 10240, 1024, 3),
           (KN, 128, 11008, 3072, 4), (KN, 200, 10240, 4096, 5), (KN, 48, 28672, 1024, 6), (NK, 32, 3072, 11008, 0),
           (NK, 17, 13824, 5120, 1), (NK, 32, 8192, 11008, 1), (NK, 31, 10240, 3072, 1), (NK, 17, 6144, 5120, 1), (NK, 64, 6144, 8192, 2),
           (NK, 96, 10240, 3072, 3), (NK, 128, 11008, 5120, 4), (NK, 200, 13824, 5120, 5), (NK, 48, 28672, 3072, 6)]


@pytest.mark.parametrize("layout,M,N,K,form", LIBRARY)
def test_library_plans_of_the_tiled_kernel(device, layout, M, N, K, form):
    for splitk in (0, 1, 2, 5):
        p = capi.plan(M, N, K, layout, splitk)
        if splitk == 0:
            assert _form(p) == form, p.as_dict()
        A, W = _inputs(M, N, K, layout, device, whole=True)
        C = torch.full((M, N), float("nan"), dtype=torch.half, device=device)
        capi_gemm(A, W, C, layout, plan=p)
        assert torch.equal(C, _product(A, W, layout).half()), splitk


# row blocks that share weight tiles walk K in exchanged steps (2 3 0 1): every remainder of the fours, K ranges of a
# split that start anywhere, two, three and five blocks, both sides of the rule between the two walks
@pytest.mark.parametrize("layout", [KN, NK])
@pytest.mark.parametrize("form", FORMS)
def test_row_blocks_side_by_side_are_exact(device, layout, form):
    rows = (32, 32, 64, 96, 128, 128, 64)[form]
    for N, K in ((384, 128), (384, 256), (640, 384), (384, 640), (640, 896), (384, 1920), (384, 2048), (384, 2304)):
        for M in (rows + 1, 2 * rows, 2 * rows + 3, 4 * rows + 3):
            A, W = _inputs(M, N, K, layout, device, whole=True)
            exact = _product(A, W, layout).half()
            for splitk in (1, 2, 5):
                p = make_plan(capi.FG_KERNEL_KN_MFMA, tile_n=128, m_block=16, waves=8, splitk=splitk,
                              stagger=2 + form) if layout == KN else \
                    make_plan(capi.FG_KERNEL_NK_MFMA_R, tile_n=64, m_block=32, waves=8, splitk=splitk,
                              stagger=2 + form, band=128)
                C = torch.full((M + 1, N), -7.0, dtype=torch.half, device=device)
                capi_gemm(A, W, C[:M], layout, plan=p)
                assert torch.equal(C[:M], exact), (M, N, K, splitk)
                assert bool((C[M] == -7.0).all())


# a row's sums do not depend on the row block it lies in: equal rows give equal bits, whatever block of a call they are
# in, and again in the next call.  Every remainder of the fours, K ranges of a split, few and many workgroups
@pytest.mark.parametrize("layout", [KN, NK])
@pytest.mark.parametrize("form", FORMS)
def test_equal_rows_give_equal_bits(device, layout, form):
    rows = (32, 32, 64, 96, 128, 128, 64)[form]
    M, distinct = 3 * rows + 5, 7
    pick = torch.arange(M, device=device) % distinct
    for N, K in ((640, 640), (640, 1152), (384, 1664), (640, 2304), (384, 4096), (384, 6144), (8320, 1024)):
        A, W = _inputs(distinct, N, K, layout, device, seed=form)
        for splitk in (1, 3, 5):
            p = make_plan(capi.FG_KERNEL_KN_MFMA, tile_n=128, m_block=16, waves=8, splitk=splitk, stagger=2 + form) if \
                layout == KN else make_plan(capi.FG_KERNEL_NK_MFMA_R, tile_n=64, m_block=32, waves=8, splitk=splitk,
                                            stagger=2 + form, band=128)
            C = torch.empty((M, N), dtype=torch.half, device=device)
            for _ in range(2):
                capi_gemm(A[pick].contiguous(), W, C, layout, plan=p)
                _close(C[:distinct], _product(A, W, layout), (N, K, splitk))
                assert torch.equal(C, C[:distinct][pick]), (N, K, splitk)


@pytest.mark.parametrize("layout", [KN, NK])
@pytest.mark.parametrize("M,N,K", [(256, 13824, 1152), (256, 5120, 5120), (160, 10240, 1664), (48, 1024, 4736)])
def test_equal_rows_of_the_librarys_plans_give_equal_bits(device, layout, M, N, K):
    pick = torch.arange(M, device=device) % 7
    A, W = _inputs(7, N, K, layout, device)
    C = torch.empty((M, N), dtype=torch.half, device=device)
    capi_gemm(A[pick].contiguous(), W, C, layout)
    assert torch.equal(C, C[:7][pick])
