"""Host entry points of the matrix-multiplication path, mirroring the reference's launchers.

Same names, argument order and error behaviour as the reference's C++ functions
(``LLMMM::fp16_mm`` src/mm/fp16/mm.h:9-10; the FP8 launchers examples/005.fp8.mm.cu:217-225,
:547-549, :2467-2476), taking torch CUDA tensors where the reference takes raw device pointers.
Everything goes through the C ABI of ``libllmmm.so``; torch only owns the memory and the stream.  The calls of a
model's step check and marshal their arguments in ``_native.so`` (csrc/binding.cpp), the others through ctypes here.

``stream``: None (torch's current stream), a torch stream or a raw handle.  What a call allocates itself -- private workspaces, returned
tensors -- is allocated on that stream, and returned tensors are recorded on the current one; the caller orders the two streams where
inputs or results cross them.
"""
import contextlib
import ctypes

import torch

from . import _lib
from ._lib import GemmCfg, check, lib, native as _native

_FP8_DTYPES = (torch.uint8, torch.float8_e4m3fn)


def _stream(stream):
    if stream is None:
        return ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    if isinstance(stream, torch.cuda.Stream):
        return ctypes.c_void_p(stream.cuda_stream)
    return ctypes.c_void_p(int(stream))


def _launch_stream(stream):
    """A stream argument as the torch stream to allocate on: None (nothing to do) where it is the current stream."""
    if stream is None:
        return None
    handle = _stream(stream).value or 0
    if handle == torch.cuda.current_stream().cuda_stream:
        return None
    if isinstance(stream, torch.cuda.Stream):
        return stream
    return torch.cuda.ExternalStream(handle) if handle > 1 else torch.cuda.default_stream()  # 1: the legacy handle


def _ptr(t, what, dtypes=None, numel=None):
    if not isinstance(t, torch.Tensor) or not t.is_cuda:
        raise TypeError("%s must be a CUDA tensor" % what)
    if not t.is_contiguous():
        raise ValueError("%s must be contiguous" % what)
    if dtypes is not None and t.dtype not in dtypes:
        raise RuntimeError("T is not supported.")
    if numel is not None and t.numel() < numel:
        raise ValueError("%s holds %d elements, %d needed" % (what, t.numel(), numel))
    return ctypes.c_void_p(t.data_ptr())


# ------------------------------------------------------------------------------------- FP16 / BF16
def fp16_mm(A, B, C, M, N, K, stream=None):
    """``LLMMM::fp16_mm<T>(A, B, C, M, N, K, stream)`` (src/mm/fp16/mm.cu:6-42).

    A [M,K], B [K,N], C [M,N] row-major, T = float16 or bfloat16, fp32 accumulation.
    Raises RuntimeError("M or N or K are not aligned.") unless M % 256 == 0, N % 256 == 0 and
    K % 16 == 0 (the reference's rule, mm.cu:19-21) and RuntimeError("T is not supported.")
    for other element types.  Asynchronous on ``stream`` (default: torch's current stream)."""
    _native.fp16_mm(A, B, C, M, N, K, stream)


def fp16_gemm(A, B, C=None, b_transposed=False, tile=_lib.TILE_AUTO, stream=None):
    """C = A @ B (or A @ Bt.T when ``b_transposed``) through ``llmmm_fp16_gemm_ex``.

    The library's own (wider) shape rule applies: M, N multiples of 128, K of 16."""
    return _native.fp16_gemm(A, B, C, b_transposed, tile, stream)


# ------------------------------------------------------------------------------------- FP8 quantiser
def fp8_blockwise_symmetric_quantization(x, q, scale, M, N, quant_m, quant_n=128, scale_transpose=False, stream=None):
    """``fp8_blockwise_symmetric_quantization<QUANT_M, QUANT_N, SCALE_TRANSPOSE>(x, q, scale, M, N, stream)``
    (examples/005.fp8.mm.cu:547-563).  quant_m in {1, 128}, quant_n == 128 (its static_asserts)."""
    if quant_m not in (1, 128) or quant_n != 128:
        raise ValueError("QUANT_M must be 1 or 128 and QUANT_N 128")
    kind = {(1, True): _lib.QUANT_1x128_T, (128, False): _lib.QUANT_128x128, (1, False): _lib.QUANT_1x128,
            (128, True): _lib.QUANT_128x128_T}[(quant_m, bool(scale_transpose))]
    _native.quantize_into(x, q, scale, M, N, kind, stream)


def quantize_activation(x, stream=None):
    """1x128 quantisation with transposed scales: returns (codes uint8 [M,K], scales [K/128... ceil, M])."""
    return _native.quantize(x, _lib.QUANT_1x128_T, stream)


def quantize_weight(wt, stream=None):
    """128x128 quantisation of a transposed weight Wt [N,K]: (codes [N,K], scales [ceil(N/128), ceil(K/128)])."""
    return _native.quantize(wt, _lib.QUANT_128x128, stream)


def rmsnorm_quantize_activation(x, weight, eps, stream=None):
    """RMSNorm fused in front of the activation quantiser (the fusion the reference plans, README.md:16):
    x [M,K] float32 / bfloat16 / float16, weight [K] float32 -> (codes uint8 [M,K], scales float32 [K/128, M]) of
    ``x / sqrt(mean(x^2) + eps) * weight``, ready to be the A operand of the FP8 GEMM."""
    return _native.rmsnorm_quantize(x, weight, eps, stream)


# ------------------------------------------------------------------------------------- FP8 GEMM
def workspace_bytes(out_kind, M, N, K):
    return int(lib.llmmm_fp8_gemm_workspace(out_kind, M, N, K))


def make_workspace(out_kind, M, N, K, device="cuda", stream=None):
    """Allocate a split-K workspace for this shape (None when none is needed); plain scratch, no initialisation."""
    n = workspace_bytes(out_kind, M, N, K)
    if n == 0:
        return None
    return torch.empty(n, dtype=torch.uint8, device=device)


def query_config(out_kind, M, N, K):
    cfg = GemmCfg()
    check(lib.llmmm_fp8_gemm_query(out_kind, M, N, K, ctypes.byref(cfg)))
    return cfg.tile, cfg.split_k


class PlanesRmsnorm:
    """The A operand of a projection whose input is the RMSNorm of a hidden state still in pieces (llmmm_a_planes_rmsnorm):
    ``planes`` [splits, M, K] float32 from :func:`fp8_gemm_planes`, ``residual`` / ``hidden_out`` [M, K] (float32, bfloat16 or
    float16; different tensors for M <= 4), ``norm_weight`` [K] float32."""

    def __init__(self, planes, splits, residual, hidden_out, norm_weight, eps):
        self.planes, self.splits, self.residual, self.hidden_out, self.norm_weight, self.eps = planes, splits, residual, hidden_out, norm_weight, eps

    def c_struct(self, M, K):
        code = {torch.float32: _lib.DTYPE_F32, torch.bfloat16: _lib.DTYPE_BF16, torch.float16: _lib.DTYPE_F16}.get(self.residual.dtype)
        if code is None or self.hidden_out.dtype != self.residual.dtype:
            raise RuntimeError("T is not supported.")
        return _lib.APlanesRmsnorm(_ptr(self.planes, "planes", (torch.float32,), self.splits * M * K).value, self.splits, code,
                                   _ptr(self.residual, "residual", numel=M * K).value, _ptr(self.hidden_out, "hidden_out", numel=M * K).value,
                                   _ptr(self.norm_weight, "norm_weight", (torch.float32,), K).value, self.eps)


def _a_operand(A, As, M, K, a_swiglu):
    """(A pointer, As pointer, a_layout, keep-alive) of the A operand: quantised codes + transposed scales, the fp32 gate_up result
    [M, 2K] (a_swiglu), or a :class:`PlanesRmsnorm`."""
    kb = K // 128 if K % 128 == 0 else 0
    if isinstance(A, PlanesRmsnorm):
        st = A.c_struct(M, K)
        return ctypes.cast(ctypes.pointer(st), ctypes.c_void_p), None, _lib.FP8_A_PLANES_RMSNORM, st
    if a_swiglu:
        return _ptr(A, "A (fp32 gate_up result)", (torch.float32,), M * 2 * K), None, _lib.FP8_A_SWIGLU_F32, None
    return _ptr(A, "A", _FP8_DTYPES, M * K), _ptr(As, "A_scale_transposed", (torch.float32,), kb * M), _lib.FP8_A_QUANTISED, None


def _a_workspace_bytes(A, M, N, K, a_swiglu):
    """Workspace bytes the A operand adds to a call's own: 0 for quantised codes, the library's answer for an operand it makes."""
    if isinstance(A, PlanesRmsnorm):
        return int(lib.llmmm_fp8_planes_rmsnorm_a_workspace(M, N, K))
    return int(lib.llmmm_fp8_swiglu_a_workspace(M, N, K)) if a_swiglu else 0


def _a_argument(A, M, K, a_swiglu):
    """(A argument, a_layout, keep-alive) for the native entry points, which take a :class:`PlanesRmsnorm` as its structure's address."""
    if isinstance(A, PlanesRmsnorm):
        st = A.c_struct(M, K)
        return ctypes.addressof(st), _lib.FP8_A_PLANES_RMSNORM, st
    return A, _lib.FP8_A_SWIGLU_F32 if a_swiglu else _lib.FP8_A_QUANTISED, None


def _fp8_gemm(out_kind, A, As, Bt, Bs, C, Cs, M, N, K, workspace, tile, split_k, stream, b_preshuffled=False, a_swiglu=False):
    A, a_layout, _keep = _a_argument(A, M, K, a_swiglu)
    _native.fp8_gemm(out_kind, A, As, Bt, Bs, C, Cs, M, N, K, workspace, tile, split_k, b_preshuffled, a_layout, stream)


def fp8_gemm_blockwise_quant_A_1x128__B_128x128__output_fp32(A, A_scale_transposed, B_transposed, B_scale_transposed, C, M, N, K,
                                                             stream=None, workspace=None, tile=_lib.TILE_AUTO, split_k=0,
                                                             b_preshuffled=False, a_swiglu=False):
    """examples/005.fp8.mm.cu:217-246.  C [M,N] float32.  ``b_preshuffled``: B_transposed is the image written by
    :func:`construct_mfma_B_layout` instead of row-major [N,K] (same results, bit for bit).  ``a_swiglu``: A is the fp32
    result [M, 2K] of a gate_up projection and the GEMM runs on quantise(silu(gate) * up) (A_scale_transposed: None)."""
    _fp8_gemm(_lib.OUT_F32, A, A_scale_transposed, B_transposed, B_scale_transposed, C, None, M, N, K, workspace, tile, split_k, stream,
              b_preshuffled, a_swiglu)


def fp8_gemm_blockwise_quant_A_1x128__B_128x128__output_bf16(A, A_scale_transposed, B_transposed, B_scale_transposed, C, M, N, K,
                                                             stream=None, workspace=None, tile=_lib.TILE_AUTO, split_k=0,
                                                             b_preshuffled=False, a_swiglu=False):
    """The fp32 variant's result rounded to bfloat16 (no reference kernel; same signature)."""
    _fp8_gemm(_lib.OUT_BF16, A, A_scale_transposed, B_transposed, B_scale_transposed, C, None, M, N, K, workspace, tile, split_k, stream,
              b_preshuffled, a_swiglu)


def fp8_gemm_blockwise_quant_A_1x128__B_128x128__C_1x128__output_fp8(A, A_scale_transposed, B_transposed, B_scale_transposed, C,
                                                                     C_scale_transposed, M, N, K, stream=None, workspace=None,
                                                                     tile=_lib.TILE_AUTO, split_k=0, b_preshuffled=False, a_swiglu=False):
    """examples/005.fp8.mm.cu:2467-2500 / examples/005.fp8.mm.opt.cu:468-508.  C e4m3 codes [M,N],
    C_scale_transposed float32 [N/128, M]."""
    _fp8_gemm(_lib.OUT_FP8Q, A, A_scale_transposed, B_transposed, B_scale_transposed, C, C_scale_transposed, M, N, K, workspace, tile,
              split_k, stream, b_preshuffled, a_swiglu)


def fp8_gemm_blockwise_quant_A_1x128__B_128x128__swiglu__C_1x128__output_fp8(A, A_scale_transposed, B_transposed, B_scale_transposed, C,
                                                                             C_scale_transposed, M, N, K, stream=None, workspace=None,
                                                                             tile=_lib.TILE_AUTO, split_k=0, b_preshuffled=False):
    """The gate_up projection of a gated MLP with the activation fused in front of the C quantisation (the fusion
    the reference plans, README.md:16; no reference kernel).  B_transposed [N,K] holds the gate rows in [0, N/2) and
    the up rows in [N/2, N); C = e4m3 codes of silu(gate) * up [M, N/2], C_scale_transposed float32 [N/256, M].
    M <= 128 needs a workspace (``make_workspace(OUT_FP8Q_SWIGLU, ...)``).  (The other way to fuse the activation is on the
    consumer's side: run gate_up with fp32 output and pass it to the down projection with ``a_swiglu=True``.)"""
    _fp8_gemm(_lib.OUT_FP8Q_SWIGLU, A, A_scale_transposed, B_transposed, B_scale_transposed, C, C_scale_transposed, M, N, K, workspace,
              tile, split_k, stream, b_preshuffled)


def fp8_gemm_add_rmsnorm_quant(A, A_scale_transposed, B_transposed, B_scale_transposed, residual, hidden_out, norm_weight, eps, M, N, K,
                               stream=None, workspace=None, tile=_lib.TILE_AUTO, split_k=0, b_preshuffled=False, a_swiglu=False):
    """A projection back to the hidden size (O, down) with the decoder block's epilogue behind it (the fusion the reference
    plans, README.md:16): ``hidden_out = residual + A @ B`` (stored in the residual's dtype; may be the same tensor), then
    RMSNorm(hidden_out) * norm_weight quantised 1x128 with transposed scales.  Returns (codes uint8 [M,N], scales float32
    [N/128, M]): the A operand of the next projection, bit-identical to ``rmsnorm_quantize_activation(hidden_out, ...)``."""
    A, a_layout, _keep = _a_argument(A, M, K, a_swiglu)
    return _native.fp8_gemm_add_rmsnorm_quant(A, A_scale_transposed, B_transposed, B_scale_transposed, residual, hidden_out, norm_weight, eps, M, N, K,
                                              workspace, tile, split_k, b_preshuffled, a_layout, stream)


def fp8_gemm_planes(A, A_scale_transposed, B_transposed, B_scale_transposed, M, N, K, planes=None, stream=None, workspace=None, tile=_lib.TILE_AUTO,
                    split_k=0, b_preshuffled=False, a_swiglu=False):
    """A projection that stops at its fp32 partial sums: returns (planes float32 [>= splits, M, N], splits).  Feed them to the next
    projection as a :class:`PlanesRmsnorm` (residual add, RMSNorm and quantisation then happen in that projection's kernel)."""
    kb = K // 128 if K % 128 == 0 else 0
    own_planes, launch = planes is None, _launch_stream(stream)
    with contextlib.nullcontext() if launch is None else torch.cuda.stream(launch):  # the call's own tensors belong to the stream it runs on
        if own_planes:
            planes = torch.empty(max(int(lib.llmmm_fp8_gemm_planes_bytes(M, N, K)) // 4, max(split_k, 1) * M * N), dtype=torch.float32,
                                 device=B_transposed.device)
        if workspace is None and _a_workspace_bytes(A, M, N, K, a_swiglu):
            workspace = torch.empty(_a_workspace_bytes(A, M, N, K, a_swiglu), dtype=torch.uint8, device=B_transposed.device)
    if own_planes and launch is not None:
        planes.record_stream(torch.cuda.current_stream())
    a_p, as_p, a_layout, _keep = _a_operand(A, A_scale_transposed, M, K, a_swiglu)
    cfg = GemmCfg(tile, split_k, _lib.FP8_B_PRESHUFFLED if b_preshuffled else _lib.FP8_B_ROWS, a_layout)
    splits = ctypes.c_int(0)
    ws_p, ws_n = (ctypes.c_void_p(workspace.data_ptr()), workspace.numel() * workspace.element_size()) if workspace is not None else (None, 0)
    check(lib.llmmm_fp8_gemm_planes(a_p, as_p, _ptr(B_transposed, "B_transposed", _FP8_DTYPES, N * K),
                                    _ptr(B_scale_transposed, "B_scale_transposed", (torch.float32,), ((N + 127) // 128) * kb), M, N, K,
                                    _ptr(planes, "planes", (torch.float32,), M * N), planes.numel() * 4, ctypes.byref(splits), ws_p, ws_n, ctypes.byref(cfg),
                                    _stream(stream)))
    return planes, splits.value


def fp8_gemm_qkv_rope(A, A_scale_transposed, B_transposed, B_scale_transposed, q_norm_weight, k_norm_weight, eps, cos_table, sin_table, positions,
                      n_q_heads, n_kv_heads, M, N, K, out_fp8=False, stream=None, workspace=None, tile=_lib.TILE_AUTO, split_k=0,
                      b_preshuffled=False):
    """The QKV projection with per-head RMSNorm (weights [128] or None) and rotate-half RoPE of the query and key heads fused
    behind it (planned by the reference, README.md:16).  Heads are 128 wide; cos_table / sin_table [rows, 64] float32,
    positions [M] int32.  Returns the bf16 tensor [M,N], or (codes uint8 [M,N], scales float32 [N/128, M]) with out_fp8."""
    A, a_layout, _keep = _a_argument(A, M, K, False)
    return _native.fp8_gemm_qkv_rope(A, A_scale_transposed, B_transposed, B_scale_transposed, q_norm_weight, k_norm_weight, eps, cos_table, sin_table,
                                     positions, n_q_heads, n_kv_heads, M, N, K, out_fp8, workspace, tile, split_k, b_preshuffled, a_layout, stream)


# ------------------------------------------------------------------------------------- offline layout helpers
def construct_mfma_B_layout(dst, src_transposed, N, K, stream=None):
    """The role of ``LLMMM::construct_m16n8k32_B_layout(dst, src_transposed, N, K, stream)``
    (src/base/base.h:13, src/base/base.cu:222-271): the weights Bt [N,K] e4m3, permuted once into the order the
    matrix instructions read them in -- here the 16x16x128 MFMA operand image of gfx950, consumed by the FP8 GEMMs
    with ``b_preshuffled=True``.  Raises RuntimeError("K must be greater than 0 and divisible by 128.") like the
    reference (base.cu:265-267)."""
    check(lib.llmmm_fp8_preshuffle_b(_ptr(src_transposed, "src_transposed", _FP8_DTYPES, N * K), _ptr(dst, "dst", _FP8_DTYPES, N * K), N, K,
                                     _stream(stream)))


def restore_B_layout(dst_transposed, src, N, K, stream=None):
    """Exact inverse of :func:`construct_mfma_B_layout` (the reference checks its permutation the same way,
    examples/005.fp8.mm.opt.cu:710-765)."""
    check(lib.llmmm_fp8_unshuffle_b(_ptr(src, "src", _FP8_DTYPES, N * K), _ptr(dst_transposed, "dst_transposed", _FP8_DTYPES, N * K), N, K,
                                    _stream(stream)))


def preshuffle_weight(bq, stream=None):
    """Bt [N,K] e4m3 codes -> a new tensor holding the pre-shuffled image (same shape and dtype)."""
    return _native.preshuffle(bq, stream)


def transpose_matrix__aligned_128(dst, src, M, N, stream=None):
    """``LLMMM::transpose_matrix__aligned_128<T>(dst, src, M, N, stream)`` (src/base/base.cu:124-153): dst [N,M] =
    transpose of src [M,N] for 1-byte (e4m3) and 4-byte (float) elements.  Raises
    RuntimeError("M or N can't be divided 128.") unless both are multiples of 128 (base.cu:127-129)."""
    if src.dtype != dst.dtype or src.element_size() not in (1, 4):
        raise RuntimeError("T is not supported.")
    check(lib.llmmm_transpose(src.element_size(), _ptr(src, "src", numel=M * N), _ptr(dst, "dst", numel=M * N), M, N, _stream(stream)))
