"""The SwiGLU output in one launch (64 gate + 64 up columns per workgroup, row maxima exchanged between the two workgroups of a 1x128
group), from the weight-streaming kernel and from 128 x 128 tiles, against the same kernel through an fp32 plane and the reduce
kernel: the same sums and the same arithmetic, so the same bits."""
import ctypes

import numpy as np
import pytest
import torch

from helpers import fp8_inputs

pytestmark = pytest.mark.gpu


def _call(t, M, N, K, pre, split=0, out=None, ws=None, tile=None):
    from llmmm_amd import _lib
    C, Cs = out if out else (torch.full((M, N // 2), 0x55, dtype=torch.uint8, device="cuda"), torch.full((N // 256, M), -1.0, device="cuda"))
    ws = torch.empty(M * N, device="cuda") if ws is None else ws
    cfg = _lib.GemmCfg(tile if tile is not None else _lib.TILE_AUTO if not split else _lib.TILE_SKINNY if M <= 32 else _lib.TILE_128x128, split, 1 if pre else 0, 0)
    rc = _lib.lib.llmmm_fp8_gemm_ex(_lib.OUT_FP8Q_SWIGLU, t[0].data_ptr(), t[1].data_ptr(), t[2].data_ptr(), t[3].data_ptr(), C.data_ptr(), Cs.data_ptr(), M, N,
                                    K, ws.data_ptr(), ws.numel() * 4, ctypes.byref(cfg), torch.cuda.current_stream().cuda_stream)
    assert rc == 0, _lib.lib.llmmm_last_error().decode()
    return C, Cs


def _same(a, b):
    return torch.equal(a[0], b[0]) and torch.equal(a[1].view(torch.int32), b[1].view(torch.int32))


def _inputs(oracle, M, N, K, seed, pre):
    import llmmm_amd
    t = [torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in fp8_inputs(oracle, M, N, K, seed=seed)]
    return [t[0], t[1], llmmm_amd.preshuffle_weight(t[2]) if pre else t[2], t[3]], t


def _timeouts():
    from llmmm_amd import _lib
    n = ctypes.c_uint(7)
    assert _lib.lib.llmmm_probe_strip_exchange_timeouts(ctypes.byref(n)) == 0
    return n.value


@pytest.mark.parametrize("N,K", [(12288, 512), (19456, 2560), (31744, 512), (32256, 512), (32768, 640), (12288, 5120)])
@pytest.mark.parametrize("pre", [False, True])
def test_bits_of_the_plane_route(oracle, N, K, pre):
    t, _ = _inputs(oracle, 32, N, K, 5, pre)
    for M in (1, 2, 8, 9, 15, 16, 17, 24, 25, 32):
        s = [t[0][:M].contiguous(), t[1][:, :M].contiguous(), t[2], t[3]]
        if M <= 16 or K <= 2560:
            assert _same(_call(s, M, N, K, pre), _call(s, M, N, K, pre, split=1)), M
    assert _timeouts() == 0


@pytest.mark.parametrize("N,K", [(256, 128), (512, 256), (768, 384), (12288, 640), (19456, 2560), (32000, 128), (65536, 128)])
@pytest.mark.parametrize("pre", [False, True])
def test_bits_of_the_plane_route_tiles(oracle, N, K, pre):
    from llmmm_amd import _lib
    t, _ = _inputs(oracle, 128, N, K, 6, pre)
    for M in (1, 16, 17, 33, 64, 65, 100, 112, 113, 127, 128):
        s = [t[0][:M].contiguous(), t[1][:, :M].contiguous(), t[2], t[3]]
        want = _call(s, M, N, K, pre, split=1, tile=_lib.TILE_128x128)
        guard = torch.full((M + 4, N // 2), 0x55, dtype=torch.uint8, device="cuda"), torch.full((N // 256 + 1, M), -1.0, device="cuda")
        got = _call(s, M, N, K, pre, tile=_lib.TILE_128x128, out=guard)
        assert _same((got[0][:M], got[1][:-1]), want), M
        assert (guard[0][M:] == 0x55).all() and (guard[1][-1] == -1.0).all()
    assert _timeouts() == 0


@pytest.mark.parametrize("M,N,K", [(17, 49152, 4096), (20, 51200, 4224), (32, 65536, 4096), (33, 33024, 640), (64, 33024, 256), (65, 33024, 128), (100, 37888, 512), (127, 33024, 384)])
@pytest.mark.parametrize("pre", [False, True])
def test_row_tails_in_wide_tiles(oracle, M, N, K, pre):
    """More 128-column tiles than CUs: 256-column tiles of fewer than 128 rows, which hold whole groups."""
    if K < 4096:
        t, _ = _inputs(oracle, M, N, K, M, pre)
    else:  # (the weights of 1024 columns over and over, told apart by their scales)
        t, _ = _inputs(oracle, M, 1024, K, M, pre)
        t[2], t[3] = t[2].repeat(N // 1024, 1), t[3].repeat(N // 1024, 1) * torch.linspace(0.5, 1.5, N // 128, device="cuda")[:, None]
    guard = torch.full((M + 4, N // 2), 0x55, dtype=torch.uint8, device="cuda"), torch.full((N // 256 + 1, M), -1.0, device="cuda")
    got, want = _call(t, M, N, K, pre, out=guard), _call(t, M, N, K, pre, split=1)
    assert _same((got[0][:M], got[1][:-1]), want)
    assert (guard[0][M:] == 0x55).all() and (guard[1][-1] == -1.0).all()


def test_launches_that_change_rows_and_shapes(oracle):
    """Exchange slots are kept per block of 16 rows: launches of other row counts and widths on one stream, other maxima each time."""
    from llmmm_amd import _lib
    cases = []
    for i, (M, N, K) in enumerate([(1, 12288, 512), (32, 19456, 512), (16, 12288, 640), (17, 32768, 512), (3, 19456, 512), (32, 12288 + 4096, 512),
                                   (48, 12288, 512), (128, 19456, 256), (100, 12288, 256), (33, 24576, 128)]):
        t, _ = _inputs(oracle, M, N, K, 10 + i, True)
        t[1] = t[1] * (2.0 ** i)
        cases.append((t, M, N, K, _call(t, M, N, K, True, split=1)))
    outs = [[(torch.empty_like(c[4][0]), torch.empty_like(c[4][1])) for c in cases] for _ in range(4)]
    ws = torch.empty(128 * 32768, device="cuda")
    for o in outs:
        for c, out in zip(cases, o):
            _call(c[0], c[1], c[2], c[3], True, out=out, ws=ws, tile=_lib.TILE_128x128 if c[1] > 32 else None)
    for o in outs:
        for x, c in zip(o, cases):
            assert _same(x, c[4]), c[1:4]
    assert _timeouts() == 0


@pytest.mark.parametrize("M", [16, 100])
def test_captured_with_other_work_between_replays(oracle, M):
    from llmmm_amd import _lib
    N, K = 19456, 512
    tile = _lib.TILE_128x128 if M > 32 else None
    t, _ = _inputs(oracle, M, N, K, 3, False)
    out, ws = (torch.empty((M, N // 2), dtype=torch.uint8, device="cuda"), torch.empty((N // 256, M), device="cuda")), torch.empty(M * N, device="cuda")
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        _call(t, M, N, K, False, out=out, ws=ws, tile=tile)
    side.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=side):
        for _ in range(3):
            _call(t, M, N, K, False, out=out, ws=ws, tile=tile)
    for rep in range(4):
        t[1].mul_(3.0)
        want = _call(t, M, N, K, False, split=1)
        out[0].fill_(0)
        out[1].fill_(0)
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        assert _same(out, want), rep
    assert _timeouts() == 0


@pytest.mark.parametrize("M", [5, 40])
def test_non_finite_operands(oracle, M):
    from llmmm_amd import _lib
    N, K = 19456, 512
    t, _ = _inputs(oracle, M, N, K, 4, False)
    t[0][1, 7] = 0x7F            # NaN code
    t[1][2, 3] = float("inf")
    t[1][:, 4] = 0.0             # a row of zeros
    t[0][2] = 0
    a, b = _call(t, M, N, K, False, tile=_lib.TILE_128x128 if M > 32 else None), _call(t, M, N, K, False, split=1)
    assert torch.equal(a[0], b[0]) and torch.equal(torch.nan_to_num(a[1], nan=-2.0), torch.nan_to_num(b[1], nan=-2.0))


def test_beside_a_stream_of_large_products(oracle):
    """Launches of both forms beside a stream that fills the chip: their workgroups get a few CUs at a time, in the order of their ids."""
    import llmmm_amd
    from llmmm_amd import _lib
    big = torch.randn((4096, 4096), device="cuda").half()
    cases = []
    for M in (16, 100):
        t, _ = _inputs(oracle, M, 19456, 512, M, False)
        cases.append((t, M, _call(t, M, 19456, 512, False, split=1)))
    a, b = torch.cuda.Stream(), torch.cuda.Stream()
    outs = []
    torch.cuda.synchronize()
    with torch.cuda.stream(a):
        for _ in range(12):
            llmmm_amd.fp16_gemm(big, big)
    for _ in range(10):
        for t, M, want in cases:
            with torch.cuda.stream(b):
                outs.append((_call(t, M, 19456, 512, False, tile=_lib.TILE_128x128 if M > 32 else None), want))
    torch.cuda.synchronize()
    assert all(_same(x, w) for x, w in outs) and _timeouts() == 0
