"""The tile and split the FP8 GEMM chooses by itself, over shapes at the edges of its rule: host arithmetic, no GPU.  (What the chosen
kernels compute is compared with the oracle in test_gpu_fp8_gemm.py and test_gpu_random_shapes.py.)"""
import pytest

TILES = {0: (256, 256), 1: (128, 256), 2: (256, 128), 3: (128, 128), 5: (128, 160)}
SKINNY = 8


@pytest.fixture(scope="module")
def query():
    import llmmm_amd as lib
    from llmmm_amd import _lib
    return lambda M, N, K, out=None: lib.query_config(_lib.OUT_BF16 if out is None else out, M, N, K)


# one tile, one slice; just up to and beyond one workgroup per CU; shapes only 128 x 128 tiles divide; long and short K; one row of tiles
@pytest.mark.parametrize("M", [128, 256, 384, 640, 1024, 2048, 4096])
@pytest.mark.parametrize("N,K", [(128, 128), (128, 512), (256, 16384), (384, 128), (1152, 256), (2816, 22016), (16384, 384), (18176, 18560), (32768, 128)])
def test_tile_divides_and_split_fits(query, M, N, K):
    tile, split = query(M, N, K)[:2]
    if tile == SKINNY:
        assert M == 128
        return
    bm, bn = TILES[tile]
    assert M % bm == 0 and N % bn == 0
    assert 1 <= split <= 8
    if split > 1:
        assert (M // bm) * (N // bn) * split <= 256, "a split puts at most one workgroup on each of the 256 CUs"
        assert K >= 256 * split, "shares of two 128-wide slices or more"


# 33 .. 64 rows: streaming, but for large and for wide matrices; 65 .. 127 rows: always a row tail of 128 x 128 tiles; 32 and fewer: streaming
@pytest.mark.parametrize("M,N,K,tile", [(32, 32768, 4096, SKINNY), (33, 32768, 4096, 3), (64, 1152, 17920, SKINNY), (64, 12416, 1152, 3), (40, 16512, 1408, 3),
                                        (65, 1152, 17920, 3), (65, 128, 128, 3), (127, 2304, 7808, 3), (1, 128, 128, SKINNY)])
def test_few_rows(query, M, N, K, tile):
    assert query(M, N, K)[0] == tile


def test_large_launches_keep_the_large_tiles(query):
    assert query(1024, 18176, 18560)[:2] == (0, 1)
    assert query(4096, 18176, 18560)[:2] == (0, 1)
