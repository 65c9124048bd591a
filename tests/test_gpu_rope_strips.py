"""The QKV projection with per-head RMSNorm and rotary embedding in column strips (M <= 16, bf16): one launch, the four strips of a head
exchanging partial sums of squares.  The oracle's bits on the strip kernel's own fp32 result, which sums K in the same ranges."""
import ctypes

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _case(lib, oracle, M, K, n_q, n_kv, seed, norm=True, pre=False, rows=512, fp8=False):
    N = (n_q + 2 * n_kv) * 128
    rng = np.random.default_rng(seed)
    X = rng.standard_normal((M, K)).astype(np.float32)
    X[:, ::53] *= 10
    t = [torch.from_numpy(a).cuda() for a in oracle.quant_fp8(X, 1, True)]
    w = torch.randn((N, K), generator=torch.Generator(device="cuda").manual_seed(seed), device="cuda") * 0.05
    b, bs = lib.quantize_weight(w)
    if pre:
        b = lib.preshuffle_weight(b)
    inv = 1e4 ** (-np.arange(64) / 64.0)
    ang = np.arange(rows)[:, None] * inv[None, :]
    cos, sin = np.cos(ang).astype(np.float32), np.sin(ang).astype(np.float32)
    pos = rng.integers(-2, rows + 2, M).astype(np.int32)  # some beyond the table: clamped
    qw, kw = (rng.uniform(0.5, 1.5, 128).astype(np.float32) for _ in range(2)) if norm else (None, None)
    g = lambda a: None if a is None else torch.from_numpy(a).cuda()
    C = torch.empty((M, N), dtype=torch.float32, device="cuda")
    how = {"tile": lib._lib.TILE_STRIP} if M <= 16 else {"tile": lib._lib.TILE_SKINNY, "split_k": 1}  # (beyond 16 rows: K in one range)
    lib.fp8_gemm_blockwise_quant_A_1x128__B_128x128__output_fp32(t[0], t[1], b, bs, C, M, N, K, b_preshuffled=pre, **how)
    want = oracle.qk_norm_rope(C.cpu().numpy(), qw, kw, 1e-6, cos, sin, pos, n_q, n_kv)
    want = oracle.requant_c_1x128(want) if fp8 else oracle.f32_to_bf16_bits(want)
    args = (t[0], t[1], b, bs, g(qw), g(kw), 1e-6, g(cos), g(sin), g(pos), n_q, n_kv, M, N, K)
    return (lambda: lib.fp8_gemm_qkv_rope(*args, b_preshuffled=pre, out_fp8=fp8)), want, t


def _bits(out):
    return out.view(torch.int16).cpu().numpy().view(np.uint16)


def _timeouts(lib):
    n = ctypes.c_uint(7)
    assert lib._lib.lib.llmmm_probe_strip_exchange_timeouts(ctypes.byref(n)) == 0
    return n.value


@pytest.mark.parametrize("K,n_q,n_kv", [(1024, 27, 3), (1152, 32, 8), (2560, 32, 8), (3968, 48, 8), (4096, 32, 8)])
@pytest.mark.parametrize("pre", [False, True])
def test_oracle_bits(lib, oracle, K, n_q, n_kv, pre):
    for M in (1, 2, 7, 8) + ((15, 16) if K == 4096 else ()):
        call, want, _ = _case(lib, oracle, M, K, n_q, n_kv, M + K, pre=pre)
        assert np.array_equal(_bits(call()), want), M
    call, want, _ = _case(lib, oracle, 3, K, n_q, n_kv, K, norm=False, pre=pre)
    assert np.array_equal(_bits(call()), want)
    assert _timeouts(lib) == 0


# (heads, K) whose 16-row groups, or only whose 32-row ones, fit one round of the chip; the first and last rows of a group
@pytest.mark.parametrize("M,K,n_q,n_kv", [(48, 2560, 32, 8), (49, 2560, 32, 8), (64, 2560, 32, 8), (65, 2560, 32, 8), (80, 2560, 32, 8), (81, 2560, 32, 8), (100, 2560, 32, 8),
                                          (128, 2560, 32, 8), (17, 2048, 16, 8), (33, 2048, 16, 8), (127, 2048, 16, 8), (128, 2048, 16, 8)])
def test_whole_heads_in_row_groups(lib, oracle, M, K, n_q, n_kv):
    call, want, _ = _case(lib, oracle, M, K, n_q, n_kv, M, pre=M % 2 == 0)
    assert np.array_equal(_bits(call()), want)
    call, (codes, scales), _ = _case(lib, oracle, M, K, n_q, n_kv, M, norm=M % 3 != 0, fp8=True)
    q, s = call()
    assert np.array_equal(q.cpu().numpy(), codes) and np.array_equal(s.cpu().numpy().view(np.uint32), scales.view(np.uint32))


def test_back_to_back_and_captured(lib, oracle):
    """Other shapes, row counts and heads without norm in turn on one stream: the slots' buffers alternate per head."""
    cases = [_case(lib, oracle, *c) for c in ((1, 1024, 27, 3, 1), (8, 2560, 32, 8, 2), (3, 1152, 32, 8, 3, False), (8, 1024, 27, 3, 4), (16, 4096, 32, 8, 5))]
    for _ in range(5):
        outs = [c[0]() for c in cases]
        for o, c in zip(outs, cases):
            assert np.array_equal(_bits(o), c[1])
    s = torch.cuda.Stream()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        outs = [c[0]() for c in cases for _ in range(2)]
    for _ in range(3):
        for o in outs:
            o.zero_()
        g.replay()
        eager = cases[1][0]()
        torch.cuda.synchronize()
        assert all(np.array_equal(_bits(o), cases[i // 2][1]) for i, o in enumerate(outs)) and np.array_equal(_bits(eager), cases[1][1])
    assert _timeouts(lib) == 0


def test_non_finite_rows(lib, oracle):
    call, _, t = _case(lib, oracle, 6, 2560, 32, 8, 9)
    clean = call()
    t[0][2, 5] = 0x7F           # NaN code: the whole row
    t[1][3, 4] = float("inf")   # an infinite slice scale
    out = call().float()
    assert torch.isnan(out[2]).all() and not torch.isfinite(out[4]).any()
    keep = [0, 1, 3, 5]
    assert torch.equal(out[keep], clean.float()[keep]) and _timeouts(lib) == 0
