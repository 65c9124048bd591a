"""The FP16 / BF16 product with K split over workgroups (fp32 planes, added by a second kernel): every tile that has the form, share
counts that do and do not divide the K stages, a last stage that K cuts short, both B layouts and types, against a float64 product;
the library's own choice through the Python entry point, eager and captured."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu
TILES = {"128x128": 3, "64x128": 4, "64x64": 6}


def _operands(M, N, K, dtype, bt, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    A = torch.randn((M, K), generator=g, device="cuda").to(dtype)
    B = torch.randn((N, K) if bt else (K, N), generator=g, device="cuda").to(dtype)
    return A, B, A.double() @ (B.double().t() if bt else B.double())


def _check(C, ref, A, B, bt):
    # |error| <= K additions and products in fp32 of a row's magnitude sum, then half a step of the type
    K = A.shape[1]
    mag = A.double().abs() @ (B.double().abs().t() if bt else B.double().abs())
    half_step = 2.0 ** (-11 if C.dtype == torch.float16 else -8)
    assert ((C.double() - ref).abs() <= K * 2.0 ** -24 * mag + half_step * ref.abs() + 2.0 ** -24).all()


def _call(A, B, C, bt, tile, split, ws):
    from llmmm_amd import _lib
    cfg = _lib.GemmCfg(tile, split, 0, 0)
    M, K = A.shape
    return _lib.lib.llmmm_fp16_gemm_ws(0 if A.dtype == torch.float16 else 1, A.data_ptr(), B.data_ptr(), C.data_ptr(), M, C.shape[1], K, int(bt), ws.data_ptr(),
                                       ws.numel() * 4, ctypes.byref(cfg), torch.cuda.current_stream().cuda_stream)


@pytest.mark.parametrize("tile", list(TILES))
@pytest.mark.parametrize("M,N,K,split", [(128, 128, 128, 2), (128, 256, 80, 2), (256, 128, 1040, 8), (384, 640, 1488, 5), (1152, 128, 336, 6), (128, 1408, 2000, 3),
                                         (640, 384, 976, 7), (256, 256, 4096, 4)])
def test_shares_against_float64(tile, M, N, K, split):
    for bt, dtype in ((False, torch.float16), (True, torch.bfloat16), (False, torch.bfloat16), (True, torch.float16)):
        A, B, ref = _operands(M, N, K, dtype, bt, seed=M + K)
        C = torch.full((M, N), float("nan"), dtype=dtype, device="cuda")
        ws = torch.full((split * M * N,), float("nan"), device="cuda")
        assert _call(A, B, C, bt, TILES[tile], split, ws) == 0
        _check(C, ref, A, B, bt)
        first = C.clone()
        ws.fill_(float("inf"))
        assert _call(A, B, C, bt, TILES[tile], split, ws) == 0
        assert torch.equal(C, first)


def test_non_finite_operands():
    A, B, _ = _operands(128, 128, 512, torch.bfloat16, True, seed=3)
    A[5, 400], A[7, 3], B[9, 100] = float("inf"), float("nan"), float("inf")
    C, ws = torch.empty((128, 128), dtype=torch.bfloat16, device="cuda"), torch.empty(4 * 128 * 128, device="cuda")
    assert _call(A, B, C, True, 6, 4, ws) == 0
    ref = A.double() @ B.double().t()
    assert torch.equal(torch.isnan(C), torch.isnan(ref)) and torch.equal(torch.isinf(C), torch.isinf(ref))


@pytest.mark.parametrize("bt", [False, True])
def test_the_library_choice_eager_and_captured(bt):
    import llmmm_amd
    from llmmm_amd import _lib
    M, N, K = 384, 640, 5264
    assert _lib.lib.llmmm_fp16_gemm_workspace(M, N, K) >= 2 * M * N * 4
    A, B, ref = _operands(M, N, K, torch.float16, bt, seed=1)
    C = llmmm_amd.fp16_gemm(A, B, b_transposed=bt)
    _check(C, ref, A, B, bt)
    out = torch.empty_like(C)
    s = torch.cuda.Stream()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        llmmm_amd.fp16_gemm(A, B, out, b_transposed=bt)
    for seed in (2, 3, 4):
        A.copy_(_operands(M, N, K, torch.float16, bt, seed)[0])
        out.fill_(float("nan"))
        g.replay()
        assert torch.equal(llmmm_amd.fp16_gemm(A, B, b_transposed=bt), out)
        torch.cuda.synchronize()


def test_without_room_nothing_is_split():
    from llmmm_amd import _lib
    M, N, K = 384, 640, 5264
    A, B, ref = _operands(M, N, K, torch.float16, False, seed=1)
    C, D = (torch.empty((M, N), dtype=torch.float16, device="cuda") for _ in range(2))
    ws = torch.zeros(M * N, device="cuda")
    st = torch.cuda.current_stream().cuda_stream
    assert _lib.lib.llmmm_fp16_gemm_ws(0, A.data_ptr(), B.data_ptr(), C.data_ptr(), M, N, K, 0, ws.data_ptr(), ws.numel() * 4, None, st) == 0
    assert _lib.lib.llmmm_fp16_gemm(0, A.data_ptr(), B.data_ptr(), D.data_ptr(), M, N, K, 0, st) == 0
    assert torch.equal(C, D) and not ws.any()
    assert _call(A, B, C, False, 6, 4, ws) == _lib.ERR_WORKSPACE
