"""The quantisers' block scale amax / 448 is the correctly rounded quotient: block maxima with mantissas over the whole binade, from the smallest magnitudes to the
largest, on either side of every magnitude where the kernels take another way, of zeros, infinities and NaN.  (Every mantissa: test_quotient_cpu.py.)"""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu

EDGES = (-149, -126, -117, -90, -61, -60, 0, 8, 99, 100, 101, 120, 127)


def _blocks(exponents, count, rng):
    """Block maxima: uniform mantissas over the exponents; first the edges and their neighbours, both infinities' magnitude, zero."""
    amax = np.ldexp(rng.uniform(1, 2, count), rng.integers(exponents[0], exponents[1] + 1, count)).astype(np.float32)
    e = np.float32([2.0 ** k for k in EDGES])
    edge = np.concatenate([e, np.nextafter(e, np.float32(0)), np.nextafter(e, np.float32(np.inf)), np.float32([0, 0, np.inf, np.finfo(np.float32).max])])
    amax[:edge.size] = edge
    return amax


@pytest.mark.parametrize("exponents", [(-149, -126), (-126, -88), (-64, -56), (-10, 10), (90, 127)])
@pytest.mark.parametrize("quant_m", [1, 128])
def test_scales_and_codes_over_magnitudes(exponents, quant_m):
    import torch

    import llmmm_amd
    rng = np.random.default_rng(1000 + exponents[0] + quant_m)
    mb, nb = (1024, 4) if quant_m == 1 else (8, 32)
    amax = _blocks(exponents, mb * nb, rng).reshape(mb, 1, nb, 1)
    with np.errstate(invalid="ignore", over="ignore"):
        x = (amax * rng.uniform(-0.99, 0.99, (mb, quant_m, nb, 128)).astype(np.float32)).astype(np.float32)
    x[:, :, :, 3] = np.where(np.isnan(x[:, :, :, 3]), -np.inf, x[:, :, :, 3])  # (blocks of an infinity times zero: NaN beside it)
    r, c = rng.integers(0, quant_m, (mb, nb)), rng.integers(0, 128, (mb, nb))
    i, j = np.meshgrid(np.arange(mb), np.arange(nb), indexing="ij")
    x[i, r, j, c] = amax[:, 0, :, 0] * rng.choice(np.float32([1, -1]), (mb, nb))
    x[0, :, 1 % nb] = np.nan  # nothing but NaN
    x[mb - 1, 0, 0, 5] = np.nan
    x = np.ascontiguousarray(x.reshape(mb * quant_m, nb * 128))
    m, _ = np.frexp(np.abs(amax[np.isfinite(amax) & (amax > 1e-37)]))
    assert exponents[1] < -120 or (2 * m.min() < 1.1 and 1.3 < 2 * np.median(m) < 1.7)  # the whole binade
    rq, rs = oracle.quant_fp8(x, quant_m, quant_m == 1)
    t = torch.from_numpy(x).cuda()
    q, s = llmmm_amd.quantize_activation(t) if quant_m == 1 else llmmm_amd.quantize_weight(t)
    assert np.array_equal(s.cpu().numpy().view(np.uint32).ravel(), rs.view(np.uint32).ravel())
    assert np.array_equal(q.cpu().numpy(), rq)


@pytest.mark.parametrize("M,N", [(1, 4), (127, 132), (128, 128), (129, 260), (300, 384)])
@pytest.mark.parametrize("quant_m", [1, 128])
def test_scales_of_zero(M, N, quant_m):
    """Zeros of both signs, blocks that hold NaN beside them, values so small that their scale rounds to zero: codes 0, next to blocks that have a scale."""
    import torch

    import llmmm_amd
    rng = np.random.default_rng(M + N + quant_m)
    x = rng.choice(np.float32([0, -0.0]), (M, N))
    x[M // 2, N // 2] = np.nan
    if N > 256:
        x[:, 128:256] = rng.choice(np.float32([2.0 ** -149, -2.0 ** -147, 0]), (M, 128))
        x[:, 256:] = rng.standard_normal((M, N - 256))
    rq, rs = oracle.quant_fp8(x, quant_m, quant_m == 1)
    t = torch.from_numpy(x).cuda()
    q, s = llmmm_amd.quantize_activation(t) if quant_m == 1 else llmmm_amd.quantize_weight(t)
    assert not rq[:, :min(N, 256)].any()
    assert np.array_equal(s.cpu().numpy().view(np.uint32).ravel(), rs.view(np.uint32).ravel())
    assert np.array_equal(q.cpu().numpy(), rq)
