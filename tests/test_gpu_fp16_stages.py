"""The FP16 / BF16 kernels where their K loop and their tile order can go wrong: every tile at K around one stage (64), one k step (32), the depth
of each ring and its wrap-around, with both B layouts; and tile counts that the eight XCDs do not divide.  Reference: the float64 product of the
rounded inputs.  Bound per element: the result's own rounding (half an ulp: 2^-11 f16, 2^-8 bf16, relative) plus fp32 accumulation,
K * 2^-23 * sum |a b| (K sums and products of fp32, each within 2^-24, twice that for the order)."""
import pytest
import torch

pytestmark = pytest.mark.gpu
TILES = {"256x256": (0, 256, 256), "128x256": (1, 128, 256), "256x128": (2, 256, 128), "128x128": (3, 128, 128), "64x128": (4, 64, 128), "64x64": (6, 64, 64)}


def _check(lib, M, N, K, dtype, bt, tile):
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    A = (torch.rand((M, K), generator=g, device="cuda") * 2 - 1).to(dtype)
    B = (torch.rand((K, N), generator=g, device="cuda") * 2 - 1).to(dtype)
    C = torch.full((M, N), float("nan"), dtype=dtype, device="cuda")
    lib.fp16_gemm(A, B.t().contiguous() if bt else B, C, b_transposed=bt, tile=tile)
    a, b = A.double(), B.double()
    ref = a @ b
    ulp = 2.0 ** -11 if dtype == torch.float16 else 2.0 ** -8
    bound = ref.abs() * ulp + K * 2.0 ** -23 * (a.abs() @ b.abs()) + 2.0 ** -25
    d = (C.double() - ref).abs()
    assert bool((d <= bound).all()), "M=%d N=%d K=%d %s bt=%s tile=%d: worst %.3g of the bound" % (M, N, K, dtype, bt, tile, float((d / bound).nan_to_num(9e9).max()))


@pytest.mark.parametrize("tile", sorted(TILES))
@pytest.mark.parametrize("bt", [False, True])
def test_k_around_stages_and_ring_depths(lib, tile, bt):
    tid, bm, bn = TILES[tile]
    for K in (16, 32, 48, 64, 80, 112, 128, 144, 192, 208, 256, 272, 320, 336, 384, 400, 448, 528):
        _check(lib, max(bm, 128), max(bn, 128), K, torch.float16, bt, tid)
    _check(lib, max(bm, 128), max(bn, 128), 1040, torch.bfloat16, bt, tid)


@pytest.mark.parametrize("bt", [False, True])
@pytest.mark.parametrize("M,N", [(384, 640), (1152, 384), (128, 1408), (1408, 128), (1280, 1792)])
def test_tile_counts_that_eight_does_not_divide(lib, M, N, bt):
    # 15, 27, 11, 11 and 140 tiles of 128 x 128; the last with both ring depths' neighbours 64 x 128 and 64 x 64
    for tile in ("128x128", "64x128", "64x64"):
        _check(lib, M, N, 96, torch.bfloat16, bt, TILES[tile][0])


def test_more_128x128_tiles_than_compute_units(lib):
    _check(lib, 2304, 2048, 80, torch.float16, False, TILES["128x128"][0])  # 288 tiles: the shallow rings, two workgroups per CU
    _check(lib, 2304, 2048, 192, torch.bfloat16, True, TILES["128x128"][0])


@pytest.mark.parametrize("bt", [False, True])
def test_deep_rings_around_their_first_k(lib, bt):
    """128 x 128 tiles: the shallow rings up to K = 1008, the deep ones from 1024 on, at every kind of K tail."""
    for K in (1008, 1024, 1040, 1056, 1072, 1088, 1136, 1152, 1200, 1264, 1328, 1360):
        _check(lib, 256, 128, K, torch.float16, bt, TILES["128x128"][0])
