"""The quantisers' block scale amax / 448 is the correctly rounded quotient for every amax, also where the short form does not hold
(zero, the smallest and the largest magnitudes, infinity)."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("exponents", [(0, 1), (20, 44), (110, 140), (235, 255)])
@pytest.mark.parametrize("quant_m", [1, 128])
def test_scales_and_codes_over_magnitudes(exponents, quant_m):
    import torch

    import llmmm_amd
    rng = np.random.default_rng(exponents[0] * 1000 + quant_m)
    M, N = 1024, 512
    bits = (rng.integers(exponents[0], exponents[1], (M, 1), endpoint=False).astype(np.uint32) << 23) | rng.integers(0, 1 << 23, (M, N), dtype=np.uint32)
    x = bits.view(np.float32) * rng.choice(np.float32([1, -1, 0.5, 0.001, 0]), (M, N))
    x[:256, :128] = 0  # whole blocks of zeros
    x = np.ascontiguousarray(x, dtype=np.float32)
    rq, rs = oracle.quant_fp8(x, quant_m, quant_m == 1)
    t = torch.from_numpy(x).cuda()
    q, s = llmmm_amd.quantize_activation(t) if quant_m == 1 else llmmm_amd.quantize_weight(t)
    assert np.array_equal(s.cpu().numpy().view(np.uint32).ravel(), rs.view(np.uint32).ravel())
    assert np.array_equal(q.cpu().numpy(), rq)
