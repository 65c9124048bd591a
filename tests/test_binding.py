"""The native side of the Python entry points (llmmm_amd/csrc/binding.cpp): what it refuses, how, and the streams it takes."""
import ctypes
import subprocess

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


def test_shapes_the_fp16_product_refuses():
    half = torch.zeros((256, 256), dtype=torch.float16)
    with pytest.raises(ValueError, match="two dimensions"):
        llmmm_amd.fp16_gemm(half[None], half)
    with pytest.raises(IndexError):
        llmmm_amd.fp16_gemm(half, half[0])
    with pytest.raises(ValueError, match="shape or dtype mismatch"):
        llmmm_amd.fp16_gemm(half, half[:128])
    with pytest.raises(TypeError, match="must be a CUDA tensor"):  # trailing dimensions of B are no reason
        llmmm_amd.fp16_gemm(half, half[:, :, None])


@pytest.mark.gpu
@pytest.mark.parametrize("bt", [False, True])
def test_trailing_dimensions_of_b(bt):
    g = torch.Generator(device="cuda").manual_seed(8)
    a, b = (torch.randn(s, generator=g, device="cuda").half() for s in ((128, 256), (256, 256)))
    assert torch.equal(llmmm_amd.fp16_gemm(a, b[:, :, None], b_transposed=bt), llmmm_amd.fp16_gemm(a, b, b_transposed=bt))


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


def _blocks(stream):
    """(bytes allocated, states of the blocks) of torch's allocator on one stream."""
    segments = [s for s in torch.cuda.memory_snapshot() if s["stream"] == stream]
    return sum(s["allocated_size"] for s in segments), [b["state"] for s in segments for b in s["blocks"]]


def _allocating_calls():
    """name -> call(stream) of every entry point that allocates a workspace or an output itself, on inputs that exist already."""
    M, N, K = 16, 2048, 4096
    g = torch.Generator(device="cuda").manual_seed(6)
    x, wt = torch.randn((M, K), generator=g, device="cuda"), torch.randn((N, K), generator=g, device="cuda") * 0.02
    (a, as_), (b, bs) = llmmm_amd.quantize_activation(x), llmmm_amd.quantize_weight(wt)
    residual, w, wk = torch.randn((M, N), generator=g, device="cuda").bfloat16(), torch.ones(N, device="cuda"), torch.ones(K, device="cuda")
    hidden = torch.empty_like(residual)
    tab, pos = torch.randn((M, 64), generator=g, device="cuda"), torch.arange(M, dtype=torch.int32, device="cuda")
    half, halfw = x[:1].expand(128, K).half().contiguous(), wt.half()
    streaming = llmmm_amd._lib.TILE_SKINNY
    return {
        "add_rmsnorm_quant": lambda s: llmmm_amd.fp8_gemm_add_rmsnorm_quant(a, as_, b, bs, residual, hidden, w, 1e-6, M, N, K, tile=streaming, split_k=8, stream=s),
        "qkv_rope": lambda s: (llmmm_amd.fp8_gemm_qkv_rope(a, as_, b, bs, None, None, 1e-6, tab, tab, pos, 8, 4, M, N, K, tile=streaming, split_k=8, stream=s),),
        "qkv_rope_fp8": lambda s: llmmm_amd.fp8_gemm_qkv_rope(a, as_, b, bs, None, None, 1e-6, tab, tab, pos, 8, 4, M, N, K, out_fp8=True, stream=s),
        "planes": lambda s: (llmmm_amd.fp8_gemm_planes(a, as_, b, bs, M, N, K, tile=streaming, split_k=4, stream=s)[0],),
        "quantize_activation": lambda s: llmmm_amd.quantize_activation(x, s),
        "quantize_weight": lambda s: llmmm_amd.quantize_weight(wt, s),
        "rmsnorm": lambda s: llmmm_amd.rmsnorm_quantize_activation(x, wk, 1e-6, s),
        "preshuffle": lambda s: (llmmm_amd.preshuffle_weight(b, s),),
        "fp16_gemm": lambda s: (llmmm_amd.fp16_gemm(half, halfw, b_transposed=True, stream=s),),
    }


@pytest.mark.gpu
@pytest.mark.parametrize("form", ["stream", "handle", "external", "default"])
def test_a_call_allocates_on_the_stream_it_runs_on(form):
    """Private workspaces and returned tensors come from the launch stream's blocks -- from the current stream's they could be handed
    on while the call still runs -- and a returned tensor dropped while the current stream still works is not given out again before."""
    side, here = torch.cuda.Stream(), torch.cuda.Stream()
    if form == "default":  # from a side stream onto the default one, named by its handle
        side = torch.cuda.default_stream()
    stream = {"stream": side, "handle": side.cuda_stream, "external": torch.cuda.ExternalStream(side.cuda_stream) if side.cuda_stream else side, "default": 0}[form]
    calls = _allocating_calls()
    torch.cuda.synchronize()
    with torch.cuda.stream(here):
        for name, call in calls.items():
            torch.cuda.synchronize()
            torch.cuda.empty_cache()
            before, before_here = _blocks(side.cuda_stream)[0], _blocks(here.cuda_stream)[0]
            out = call(stream)
            torch.cuda.synchronize()
            assert torch.cuda.current_stream() == here, name
            assert _blocks(here.cuda_stream)[0] == before_here, "%s took memory of the current stream" % name
            size = sum(-(-t.numel() * t.element_size() // 512) * 512 for t in out)
            assert _blocks(side.cuda_stream)[0] - before >= size, "%s: outputs are not the launch stream's" % name
            torch.cuda._sleep(20_000_000)  # about 10 ms of work on the current stream that may still read the outputs
            del out
            assert "active_pending_free" in _blocks(side.cuda_stream)[1], "%s: an output is free before the current stream is done" % name


@pytest.mark.gpu
def test_results_on_another_stream_while_the_current_one_reuses_its_memory():
    """The same bits as on the current stream, with the side stream busy at the call and every freed block of the current stream
    overwritten as soon as the call has returned."""
    calls = _allocating_calls()
    expect = {name: [t.clone() for t in call(None)] for name, call in calls.items()}
    side = torch.cuda.Stream()
    for name, call in calls.items():
        torch.cuda.synchronize()
        with torch.cuda.stream(side):
            torch.cuda._sleep(2_000_000)
        out = call(side)
        for n in (1 << 12, 1 << 17, 1 << 20, 1 << 22):
            torch.empty(n, dtype=torch.uint8, device="cuda").fill_(0x7f)
        torch.cuda.current_stream().wait_stream(side)
        n = 4 * 16 * 2048 if name == "planes" else None  # (rows beyond the splits are not written)
        for t, e in zip(out, expect[name]):
            assert torch.equal(t.view(torch.uint8).flatten()[:n and 4 * n], e.view(torch.uint8).flatten()[:n and 4 * n]), name


GIL_PROBE = r"""
#include <dlfcn.h>
#include <stddef.h>
int calls, held;  /* allocations, and those made with the interpreter lock held */
static void* hip(const char* name) { return dlsym(dlopen("libamdhip64.so.7", RTLD_NOW | RTLD_NOLOAD), name); }
void* probe_alloc(size_t n, int device, void* stream)
{
  void* p = NULL;
  ++calls;
  held += ((int (*)(void))dlsym(RTLD_DEFAULT, "PyGILState_Check"))();
  return ((int (*)(void**, size_t))hip("hipMalloc"))(&p, n) == 0 ? p : NULL;
}
void probe_free(void* p, size_t n, int device, void* stream) { ((int (*)(void*))hip("hipFree"))(p); }
"""


@pytest.mark.gpu
def test_the_interpreter_lock_is_free_while_memory_is_allocated(tmp_path):
    """An allocation that has to go to the device (here through an allocator of the test's own) does not hold up other Python threads."""
    src, so = tmp_path / "gil_probe.c", str(tmp_path / "gil_probe.so")
    src.write_text("#define _GNU_SOURCE\n" + GIL_PROBE)
    subprocess.run(["gcc", "-shared", "-fPIC", "-o", so, str(src), "-ldl"], check=True)
    probe = ctypes.CDLL(so)
    calls, held = ctypes.c_int.in_dll(probe, "calls"), ctypes.c_int.in_dll(probe, "held")
    allocator = torch.cuda.memory.CUDAPluggableAllocator(so, "probe_alloc", "probe_free")
    keep = test_the_interpreter_lock_is_free_while_memory_is_allocated.keep = [probe, allocator]  # (pools in use are not freed before the process ends)
    for name, call in _allocating_calls().items():
        torch.cuda.synchronize()
        before, pool = calls.value, torch.cuda.MemPool(allocator.allocator())
        with torch.cuda.use_mem_pool(pool):
            out = call(None)
        torch.cuda.synchronize()
        assert calls.value > before, name
        assert held.value == 0, "%s allocates with the interpreter lock held" % name
        keep += [pool, out]


@pytest.mark.gpu
def test_calls_on_a_stream_that_takes_part_in_a_capture():
    """Allocating calls on a forked side stream inside a capture: replayed results are the eager ones, every time."""
    calls = _allocating_calls()
    expect = {name: [t.clone() for t in call(None)] for name, call in calls.items()}
    torch.cuda.synchronize()
    side, outs = torch.cuda.Stream(), {}
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        side.wait_stream(torch.cuda.current_stream())
        for name, call in calls.items():
            outs[name] = call(side)
        torch.cuda.current_stream().wait_stream(side)
    for _ in range(3):
        for out in outs.values():
            for t in out:
                t.view(torch.uint8).fill_(0x11)
        graph.replay()
        torch.cuda.synchronize()
        for name, out in outs.items():
            n = 4 * 16 * 2048 if name == "planes" else None
            for t, e in zip(out, expect[name]):
                assert torch.equal(t.view(torch.uint8).flatten()[:n and 4 * n], e.view(torch.uint8).flatten()[:n and 4 * n]), name
        torch.empty(1 << 20, device="cuda").normal_()  # the program's own work between replays
