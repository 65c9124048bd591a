"""The native side of the Python entry points (llmmm_amd/csrc/binding.cpp): what it refuses, how, and the streams it takes."""
import pytest
import torch

import llmmm_amd

M, N, K = 4, 256, 1024


def _fp8_args(device):
    t = lambda shape, dtype=torch.uint8: torch.zeros(shape, dtype=dtype, device=device)  # noqa: E731
    f32 = torch.float32
    return {"A": t((M, K)), "As": t((K // 128, M), f32), "Bt": t((N, K)), "Bs": t((N // 128, K // 128), f32), "C": t((M, N)), "Cs": t((N // 128, M), f32)}


def _gemm(a, **over):
    a = dict(a, **over)
    llmmm_amd.fp8_gemm_blockwise_quant_A_1x128__B_128x128__C_1x128__output_fp8(a["A"], a["As"], a["Bt"], a["Bs"], a["C"], a["Cs"], M, N, K)


def test_host_tensors_are_refused_everywhere():
    a, x = _fp8_args("cpu"), torch.zeros((M, K))
    w, h = torch.ones(N), torch.zeros((M, N), dtype=torch.bfloat16)
    tab, pos = torch.zeros((8, 64)), torch.zeros(M, dtype=torch.int32)
    half = torch.zeros((256, 256), dtype=torch.float16)
    calls = [lambda: _gemm(a), lambda: llmmm_amd.quantize_activation(x), lambda: llmmm_amd.quantize_weight(x), lambda: llmmm_amd.preshuffle_weight(a["Bt"]),
             lambda: llmmm_amd.rmsnorm_quantize_activation(x, w, 1e-6), lambda: llmmm_amd.fp16_gemm(half, half), lambda: llmmm_amd.fp16_mm(half, half, half, 256, 256, 256),
             lambda: llmmm_amd.fp8_gemm_add_rmsnorm_quant(a["A"], a["As"], a["Bt"], a["Bs"], h, h, w, 1e-6, M, N, K),
             lambda: llmmm_amd.fp8_gemm_qkv_rope(a["A"], a["As"], a["Bt"], a["Bs"], None, None, 1e-6, tab, tab, pos, 1, 0, M, N, K)]
    for call in calls:
        with pytest.raises(TypeError, match="must be a CUDA tensor"):
            call()
    for bad in (None, 5, [1.0]):
        with pytest.raises(TypeError):
            llmmm_amd.quantize_activation(bad)


@pytest.mark.gpu
@pytest.mark.parametrize("name,make,error,match", [
    ("A", lambda t: t[:, :K // 2], ValueError, "A must be contiguous"),
    ("A", lambda t: t.float(), RuntimeError, "T is not supported."),
    ("As", lambda t: t[:-1], ValueError, "A_scale_transposed holds 28 elements, 32 needed"),
    ("Bt", lambda t: t[:-1], ValueError, "B_transposed holds"),
    ("Bs", lambda t: t.half(), RuntimeError, "T is not supported."),
    ("C", lambda t: t.cpu(), TypeError, "C must be a CUDA tensor"),
    ("Cs", lambda t: None, TypeError, "C_scale_transposed must be a CUDA tensor"),
    ("C", lambda t: torch.zeros(M * N + 16, dtype=torch.uint8, device="cuda")[1:], RuntimeError, "16-byte aligned"),
])
def test_refusals_of_a_product(name, make, error, match):
    a = _fp8_args("cuda")
    with pytest.raises(error, match=match):
        _gemm(a, **{name: make(a[name])})


@pytest.mark.gpu
def test_streams_and_code_types():
    """The current stream, a named stream and a raw handle give the same bits; codes may be uint8 or float8_e4m3fn."""
    g = torch.Generator(device="cuda").manual_seed(5)
    x, wt = torch.randn((M, K), generator=g, device="cuda"), torch.randn((N, K), generator=g, device="cuda")
    (aq, as_), (bq, bs) = llmmm_amd.quantize_activation(x), llmmm_amd.quantize_weight(wt)
    side = torch.cuda.Stream()
    torch.cuda.synchronize()
    results = []
    for form in ("current", "context", "stream", "handle"):
        c = torch.zeros((M, N), dtype=torch.uint8, device="cuda").view(torch.float8_e4m3fn)
        cs = torch.zeros((N // 128, M), device="cuda")
        torch.cuda.synchronize()
        a = (aq.view(torch.float8_e4m3fn), as_, bq, bs, c, cs, M, N, K)
        ws = llmmm_amd.make_workspace(2, M, N, K)
        if form == "context":
            with torch.cuda.stream(side):
                llmmm_amd.fp8_gemm_blockwise_quant_A_1x128__B_128x128__C_1x128__output_fp8(*a, workspace=ws)
        else:
            s = {"current": None, "stream": side, "handle": side.cuda_stream}[form]
            llmmm_amd.fp8_gemm_blockwise_quant_A_1x128__B_128x128__C_1x128__output_fp8(*a, stream=s, workspace=ws)
        torch.cuda.synchronize()
        results.append((c.view(torch.uint8).clone(), cs.clone()))
    for c, cs in results[1:]:
        assert torch.equal(c, results[0][0]) and torch.equal(cs, results[0][1])
    assert results[0][0].any()
