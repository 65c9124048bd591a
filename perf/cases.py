"""The work that programs have this library do, as cases that a measuring program can prepare, run and compare.

Four kinds of case, over the sizes the library is used at:

  layer   the matrix-product side of one decoder layer, from the hidden state to the next layer's quantised operand: RMSNorm + quantiser,
          the QKV projection with per-head norm and rotary embedding, the attention result's quantiser, O with residual add + norm +
          quantiser, gate_up with SwiGLU, down with residual add + norm + quantiser (attention itself is not part of this library: its
          result is an input).  1 row: single-stream decode; tens of rows: batched decode; thousands: prefill
  fp8     one FP8 blockwise-scaled product by itself, with the fused 1x128 quantisation of C or with bf16 output
  fp16    one FP16 / BF16 product, B row-major or transposed
  weight  what loading a model does to every weight matrix: 128x128 quantisation, then the matrix-instruction image

Weights are N(0, 0.02), activations N(0, 1) with one channel in a hundred scaled by 20 (the outlier channels FP8 block scales exist for).
"""
import math

import torch

import llmmm_amd
from llmmm_amd import _lib

EPS = 1e-6
TABLE_ROWS = 4096

# (hidden, query heads, key/value heads, MLP width) of the model families the tune table lists; heads are 128 wide
FAMILIES = [(2048, 16, 8, 6144), (2560, 32, 8, 9728), (3072, 24, 8, 8192), (3584, 28, 4, 18944), (4096, 32, 8, 14336), (5120, 40, 8, 17408),
            (5120, 64, 8, 25600), (8192, 64, 8, 28672)]


def _layer(name, M, family, preshuffled):
    hidden, n_q, n_kv, inter = family
    return {"name": name, "kind": "layer", "M": M, "hidden": hidden, "n_q": n_q, "n_kv": n_kv, "inter": inter, "preshuffled": preshuffled}


def listed():
    return [
        # the smallest call: one token through one projection with the fused quantisation of C
        {"name": "fp8_qkv_m1", "kind": "fp8", "M": 1, "N": 6144, "K": 2560, "out": "fp8", "preshuffled": False},
        # single-stream decode
        _layer("layer_decode_m1", 1, FAMILIES[1], True),
        # batched decode on a larger model, weights kept as they were quantised
        _layer("layer_decode_m16", 16, FAMILIES[4], False),
        # a server's ragged decode batch
        _layer("layer_decode_m100", 100, FAMILIES[1], True),
        # prefill of a 2048-token chunk
        _layer("layer_prefill_m2048", 2048, FAMILIES[1], True),
        # prefill on the largest model
        _layer("layer_prefill_wide", 4096, FAMILIES[7], False),
        # the headline FP8 product
        {"name": "fp8_4096", "kind": "fp8", "M": 4096, "N": 4096, "K": 4096, "out": "fp8", "preshuffled": False},
        # the rest of a prompt: a few hundred rows, long K
        {"name": "fp8_chunk_m384", "kind": "fp8", "M": 384, "N": 3584, "K": 18944, "out": "bf16", "preshuffled": False},
        # the FP16 product: the small and the headline size
        {"name": "fp16_1024", "kind": "fp16", "M": 1024, "N": 1024, "K": 1024, "dtype": "float16", "b_transposed": False},
        {"name": "fp16_4096", "kind": "fp16", "M": 4096, "N": 4096, "K": 4096, "dtype": "float16", "b_transposed": False},
        # sizes that divide no tile but the smallest, K no multiple of a stage, nn.Linear's weight layout
        {"name": "bf16_ragged", "kind": "fp16", "M": 1152, "N": 3456, "K": 2000, "dtype": "bfloat16", "b_transposed": True},
        # loading a model: the largest matrix of a small one
        {"name": "weight_load", "kind": "weight", "N": 19456, "K": 2560},
    ]


def _spread(rng, lo, hi, step):
    """A multiple of step in lo .. hi, even over the logarithm."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return max(lo, min(hi, int(round(v / step)) * step))


def _rows(rng):
    """Token counts the FP8 products take: any number up to 128, multiples of 128 beyond."""
    return _spread(rng, 1, 128, 1) if rng.random() < 0.5 else _spread(rng, 128, 4096, 128)


def draw(rng):
    kind = rng.choice(["layer", "layer", "fp8", "fp8", "fp16", "fp16", "weight"])
    if kind == "layer":
        c = _layer("", _rows(rng), rng.choice(FAMILIES), rng.random() < 0.5)
        del c["name"]
        return c
    if kind == "fp8":
        return {"kind": "fp8", "M": _rows(rng), "N": _spread(rng, 1024, 32768, 128), "K": _spread(rng, 1024, 28672, 128), "out": rng.choice(["fp8", "bf16"]),
                "preshuffled": rng.random() < 0.5}
    if kind == "fp16":
        return {"kind": "fp16", "M": _spread(rng, 256, 8192, 128), "N": _spread(rng, 256, 8192, 128), "K": _spread(rng, 256, 8192, 16),
                "dtype": rng.choice(["float16", "bfloat16"]), "b_transposed": rng.random() < 0.5}
    return {"kind": "weight", "N": _spread(rng, 1024, 32768, 128), "K": _spread(rng, 1024, 28672, 128)}


# ---------------------------------------------------------------------------------------------------------- prepare
def _activations(g, M, K):
    x = torch.randn((M, K), generator=g, device="cuda")
    x[:, torch.randperm(K, generator=g, device="cuda")[: max(1, K // 100)]] *= 20.0
    return x


def _fp8_weight(g, N, K, preshuffled):
    q, s = llmmm_amd.quantize_weight(torch.randn((N, K), generator=g, device="cuda") * 0.02)
    return (llmmm_amd.preshuffle_weight(q) if preshuffled else q), s


def prepare(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return {"layer": _prepare_layer, "fp8": _prepare_fp8, "fp16": _prepare_fp16, "weight": _prepare_weight}[case["kind"]](case, g)


def _prepare_layer(case, g):
    M, H, I = case["M"], case["hidden"], case["inter"]
    n_q, n_kv, pre = case["n_q"], case["n_kv"], case["preshuffled"]
    n_qkv = (n_q + 2 * n_kv) * 128
    angle = torch.arange(TABLE_ROWS, device="cuda", dtype=torch.float64)[:, None] * 1e6 ** (-torch.arange(64, device="cuda", dtype=torch.float64) / 64)[None, :]

    def norm_weight(n):
        return 1.0 + 0.1 * torch.randn(n, generator=g, device="cuda")

    return {
        "case": case, "n_qkv": n_qkv,
        "hidden": _activations(g, M, H).to(torch.bfloat16),
        "attention": _activations(g, M, n_q * 128),
        "qkv": _fp8_weight(g, n_qkv, H, pre), "o": _fp8_weight(g, H, n_q * 128, pre),
        "gate_up": _fp8_weight(g, 2 * I, H, pre), "down": _fp8_weight(g, H, I, pre),
        "norm_in": norm_weight(H), "norm_mlp": norm_weight(H), "norm_next": norm_weight(H), "norm_q": norm_weight(128), "norm_k": norm_weight(128),
        "cos": torch.cos(angle).float().contiguous(), "sin": torch.sin(angle).float().contiguous(),
        # prefill: one sequence's consecutive positions; decode: every row a sequence of its own
        "positions": (torch.arange(M, device="cuda", dtype=torch.int32) if M > 128
                      else torch.randint(0, TABLE_ROWS, (M,), generator=g, device="cuda", dtype=torch.int32)),
        "hidden_mid": torch.empty((M, H), dtype=torch.bfloat16, device="cuda"), "hidden_out": torch.empty((M, H), dtype=torch.bfloat16, device="cuda"),
        "act": torch.empty((M, I), dtype=torch.uint8, device="cuda"), "act_scale": torch.empty((I // 128, M), dtype=torch.float32, device="cuda"),
        "workspace": llmmm_amd.make_workspace(_lib.OUT_FP8Q_SWIGLU, M, 2 * I, H),
    }


def _prepare_fp8(case, g):
    M, N, K = case["M"], case["N"], case["K"]
    fp8 = case["out"] == "fp8"
    return {
        "case": case, "a": llmmm_amd.quantize_activation(_activations(g, M, K)), "b": _fp8_weight(g, N, K, case["preshuffled"]),
        "c": torch.empty((M, N), dtype=torch.uint8 if fp8 else torch.bfloat16, device="cuda"),
        "c_scale": torch.empty((N // 128, M), dtype=torch.float32, device="cuda") if fp8 else None,
        "workspace": llmmm_amd.make_workspace(_lib.OUT_FP8Q if fp8 else _lib.OUT_BF16, M, N, K),
    }


def _prepare_fp16(case, g):
    M, N, K, t = case["M"], case["N"], case["K"], getattr(torch, case["dtype"])
    return {"case": case, "a": torch.randn((M, K), generator=g, device="cuda").to(t),
            "b": (torch.randn((N, K) if case["b_transposed"] else (K, N), generator=g, device="cuda") * 0.02).to(t),
            "c": torch.empty((M, N), dtype=t, device="cuda")}


def _prepare_weight(case, g):
    return {"case": case, "w": torch.randn((case["N"], case["K"]), generator=g, device="cuda") * 0.02}


# -------------------------------------------------------------------------------------------------------------- run
def run(state):
    return {"layer": _run_layer, "fp8": _run_fp8, "fp16": _run_fp16, "weight": _run_weight}[state["case"]["kind"]](state)


def _run_layer(s):
    c = s["case"]
    M, H, I, n_q, n_kv, pre = c["M"], c["hidden"], c["inter"], c["n_q"], c["n_kv"], c["preshuffled"]
    a, a_scale = llmmm_amd.rmsnorm_quantize_activation(s["hidden"], s["norm_in"], EPS)
    qkv = llmmm_amd.fp8_gemm_qkv_rope(a, a_scale, s["qkv"][0], s["qkv"][1], s["norm_q"], s["norm_k"], EPS, s["cos"], s["sin"], s["positions"], n_q, n_kv,
                                      M, s["n_qkv"], H, b_preshuffled=pre)
    a, a_scale = llmmm_amd.quantize_activation(s["attention"])
    a, a_scale = llmmm_amd.fp8_gemm_add_rmsnorm_quant(a, a_scale, s["o"][0], s["o"][1], s["hidden"], s["hidden_mid"], s["norm_mlp"], EPS, M, H, n_q * 128,
                                                      b_preshuffled=pre)
    llmmm_amd.fp8_gemm_blockwise_quant_A_1x128__B_128x128__swiglu__C_1x128__output_fp8(
        a, a_scale, s["gate_up"][0], s["gate_up"][1], s["act"], s["act_scale"], M, 2 * I, H, workspace=s["workspace"], b_preshuffled=pre)
    a, a_scale = llmmm_amd.fp8_gemm_add_rmsnorm_quant(s["act"], s["act_scale"], s["down"][0], s["down"][1], s["hidden_mid"], s["hidden_out"], s["norm_next"],
                                                      EPS, M, H, I, b_preshuffled=pre)
    return {"qkv": qkv, "hidden_mid": s["hidden_mid"], "act": s["act"], "act_scale": s["act_scale"], "hidden_out": s["hidden_out"], "next": a,
            "next_scale": a_scale}


def _run_fp8(s):
    c = s["case"]
    if c["out"] == "fp8":
        llmmm_amd.fp8_gemm_blockwise_quant_A_1x128__B_128x128__C_1x128__output_fp8(
            s["a"][0], s["a"][1], s["b"][0], s["b"][1], s["c"], s["c_scale"], c["M"], c["N"], c["K"], workspace=s["workspace"], b_preshuffled=c["preshuffled"])
        return s["c"], s["c_scale"]
    llmmm_amd.fp8_gemm_blockwise_quant_A_1x128__B_128x128__output_bf16(
        s["a"][0], s["a"][1], s["b"][0], s["b"][1], s["c"], c["M"], c["N"], c["K"], workspace=s["workspace"], b_preshuffled=c["preshuffled"])
    return s["c"]


def _run_fp16(s):
    return llmmm_amd.fp16_gemm(s["a"], s["b"], s["c"], b_transposed=s["case"]["b_transposed"])


def _run_weight(s):
    q, scale = llmmm_amd.quantize_weight(s["w"])
    return llmmm_amd.preshuffle_weight(q), scale


# --------------------------------------------------------------------------------------------------- work, tolerance
def _fp8_product(M, N, K):
    """Operand bytes (codes and scales) and operations of one blockwise product, without its output."""
    return M * K + N * K + 4 * (M * K // 128 + (N // 128) * (K // 128)), 2 * M * N * K


def work(case):
    if case["kind"] == "layer":
        M, H, I, heads = case["M"], case["hidden"], case["inter"], case["n_q"] + 2 * case["n_kv"]
        nq = case["n_q"] * 128
        weights = heads * 128 * H + H * nq + 2 * I * H + H * I
        # the hidden state in and out twice, attention's fp32 result in, q/k/v out, the MLP's codes and the next operand out, the angles
        rows = M * (2 * H + 2 * 2 * H + 4 * nq + 2 * heads * 128 + (I + I // 32) + (H + H // 32) + 512)
        return {"bytes": weights + weights // 4096 + rows, "flops": 2 * M * weights}
    if case["kind"] == "fp8":
        M, N = case["M"], case["N"]
        operands, flops = _fp8_product(M, N, case["K"])
        return {"bytes": operands + (M * N + M * N // 32 if case["out"] == "fp8" else 2 * M * N), "flops": flops}
    if case["kind"] == "fp16":
        M, N, K = case["M"], case["N"], case["K"]
        return {"bytes": 2 * (M * K + K * N + M * N), "flops": 2 * M * N * K}
    return {"bytes": 5 * case["N"] * case["K"] + case["N"] * case["K"] // 4096, "flops": 0}


def tolerance(case):
    """About four times what was measured: layers with K of every product split in another way (outputs differ where a sum that moved by an fp32
    ulp crosses a bf16 or e4m3 rounding boundary; the widest layer: rel 1e-3, max 0.06, 0.4 % of the last codes), single products against
    float64 sums (FP8: 0.24 % of codes, bf16 rel 3.4e-4, max one bf16 step; FP16 / BF16 rel 1.5e-5 / 3.8e-5, max one step of the type)."""
    if case["kind"] == "layer":
        return {"rel": 4e-3, "max": 0.2, "differ": 0.01}
    if case["kind"] == "fp8":
        return {"rel": 1.5e-3, "max": 0.03, "differ": 0.01}
    if case["kind"] == "fp16":
        return {"rel": 1.5e-4, "max": 0.03} if case["dtype"] == "bfloat16" else {"rel": 6e-5, "max": 0.004}
    return "exact"
