"""Codes of quotients on and next to the rounding boundaries through the row kernels, several chunks of a thread in doubt at once, beside blocks whose maximum
lies on either side of what the quotients take without a division, blocks of zeros, infinities and NaN: bit for bit against the oracle.

Rows of +-1 with eps = 0 have the norm 1 exactly, so that the quantised values are the norm's weights with the rows' signs."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _weights(oracle, K, rng):
    vals = oracle.e4m3_decode(np.arange(0, 0x7F, dtype=np.uint8)).astype(np.float64)
    mids = (vals[:-1] + vals[1:]) / 2  # 126 ties
    edges = [np.float32(2.0 ** e) for e in (-126, -91, -90, -61, -60, 0, 99, 100, 101, 120, 127)]
    edges += [np.nextafter(e, np.float32(d), dtype=np.float32) for e in edges for d in (0, np.inf)]
    w = np.zeros((K // 128, 128), np.float32)
    for b in range(K // 128):
        amax = edges[rng.integers(len(edges))] if b % 4 == 3 else np.float32(rng.uniform(1, 2) * 2.0 ** rng.integers(-20, 20))
        s = np.float32(amax / np.float32(448))
        v = (mids * float(s)).astype(np.float32)
        v = np.minimum((v.view(np.int32) + rng.integers(-3, 4, v.shape)).astype(np.int32), np.float32(amax).view(np.int32)).clip(0).astype(np.int32).view(np.float32)
        w[b, 0], w[b, 1:127] = amax, v
    w[1::9] = 0
    if K >= 1024:
        w[5, 17] = np.nan
        w[6, 3] = np.inf
    return w.reshape(K)


@pytest.mark.parametrize("K", [128, 2048, 2560, 4096, 5120, 8192, 10240])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_rows_in_doubt(lib, oracle, K, dtype):
    rng = np.random.default_rng(K)
    w = _weights(oracle, K, rng)
    x = rng.choice(np.float32([1, -1]), (5, K))
    with np.errstate(all="ignore"):
        rq, rs = oracle.rmsnorm_quant(x, w, 0.0)
    tw = torch.from_numpy(w).cuda()
    q, s = lib.rmsnorm_quantize_activation(torch.from_numpy(x).cuda().to(dtype), tw, 0.0)
    assert np.array_equal(s.cpu().numpy().view(np.uint32), rs.view(np.uint32))
    assert np.array_equal(q.cpu().numpy(), rq), np.argwhere(q.cpu().numpy() != rq)[:5]
    # behind a product of zeros: the add + norm + quantiser kernel on the same rows
    A, As = torch.zeros((5, 128), dtype=torch.uint8, device="cuda"), torch.zeros((1, 5), device="cuda")
    B, Bs = torch.zeros((K, 128), dtype=torch.uint8, device="cuda"), torch.zeros((K // 128, 1), device="cuda")
    res = torch.from_numpy(x).cuda().to(dtype)
    from llmmm_amd import _lib
    q, s = lib.fp8_gemm_add_rmsnorm_quant(A, As, B, Bs, res, torch.empty_like(res), tw, 0.0, 5, K, 128, tile=_lib.TILE_SKINNY, split_k=1)
    assert np.array_equal(s.cpu().numpy().view(np.uint32), rs.view(np.uint32))
    assert np.array_equal(q.cpu().numpy(), rq), np.argwhere(q.cpu().numpy() != rq)[:5]
