"""Timed cases: what a program that uses this package has it do on the GPU.

Every case is one pass through public entry points:

  kind "gemm"      one linear layer.  entry "drop-in": linear_forward_eXmY_cuda on reference-layout weights; "native":
                   linear_forward_native on native-layout weights (with group exponents or without); "module": FPxLinear
                   (with a bias or without), as an inference program holds it.
  kind "layer"     the four linear layers of a decoder layer as FPxLinear modules: fused Q/K/V, output projection, fused
                   gate + up, down (examples/decode_layer.py holds the same four).
  kind "quantize"  float weights -> native codes and scales (loading a checkpoint onto the GPU).
  kind "relayout"  reference-layout weights -> native layout (what the first drop-in call on a weight tensor does).
  kind "dequant"   native weights -> fp16 (merging, exporting, checking).

Sizes: M = output features (multiples of 256), K = input features (multiples of 64, so K need not fill the last 256-column
block), N = tokens.  Formats are (exponent, mantissa) bits.
"""
import math

import torch

import fp6_llm_amd as fp6
from fp6_llm_amd.module import FPxLinear

DEVICE = "cuda:0"
MAX_WEIGHTS = 28672 * 8192          # the largest single matrix of the listed cases
MAX_MACS = MAX_WEIGHTS * 2048       # and the largest GEMM
MAX_LAYER_WEIGHTS = 8192 * (8192 + 2 * 1024) + 8192 * 8192 + 3 * 28672 * 8192


def _gemm(name, entry, E, M, OC, IC, B, groups=False, bias=False):
    return {"name": name, "kind": "gemm", "entry": entry, "E": E, "Mb": M, "M": OC, "K": IC, "N": B, "groups": groups, "bias": bias}


def _layer(name, E, M, hidden, kv, mlp, B):
    return {"name": name, "kind": "layer", "E": E, "Mb": M, "hidden": hidden, "kv": kv, "mlp": mlp, "N": B}


def listed():
    return [
        # one token through an attention projection by way of the reference's own entry point: the smallest call there is
        _gemm("drop_in_4096x4096_n1", "drop-in", 3, 2, 4096, 4096, 1),
        # decode steps: a small model at a small batch, a large one (grouped-query attention, 5-bit weights) at a serving batch
        _layer("layer_4096_11008_n8", 3, 2, 4096, 4096, 11008, 8),
        _layer("layer_8192_28672_n32", 2, 2, 8192, 1024, 28672, 32),
        # 4-bit weights with group exponents at the largest batch of the small-batch range
        _gemm("native_8192x8192_n16_e2m1_groups", "native", 2, 1, 8192, 8192, 16, groups=True),
        # a scheduler's odd batch on a fused Q/K/V matrix
        _gemm("native_10240x8192_n72", "native", 3, 2, 10240, 8192, 72),
        # few rows (a grouped-query key projection), speculative or chunked decoding
        _gemm("native_1024x8192_n200_e2m3", "native", 2, 3, 1024, 8192, 200),
        # a prefill chunk
        _gemm("prefill_8192x8192_n512", "native", 3, 2, 8192, 8192, 512),
        # a ragged prompt on a ragged matrix: K cuts the last block, N cuts the last tile
        _gemm("prefill_4608x4544_n777_e2m2_groups", "native", 2, 2, 4608, 4544, 777, groups=True),
        # the widest projection of a large model over a long prompt: the largest case
        _gemm("prefill_28672x8192_n2048", "module", 3, 2, 28672, 8192, 2048),
        # a longer prompt still, through a module with a bias
        _gemm("prefill_8192x8192_n4096_bias", "module", 3, 2, 8192, 8192, 4096, bias=True),
        # loading weights: a bf16 checkpoint quantized on the GPU, reference-layout weights turned into the native layout
        {"name": "quantize_8192x8192_bf16", "kind": "quantize", "E": 3, "Mb": 2, "M": 8192, "K": 8192, "dtype": "bf16", "groups": False},
        {"name": "relayout_11008x4096", "kind": "relayout", "E": 3, "Mb": 2, "M": 11008, "K": 4096},
    ]


def _log_size(rng, lo, hi, step):
    """A multiple of `step` between lo and hi, spread evenly over the logarithm."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return min(hi, max(lo, int(v / step + 0.5) * step))


def draw(rng):
    E, Mb = rng.choice(((3, 2), (3, 2), (2, 2), (2, 3), (2, 1)))
    kind = rng.choice(("gemm",) * 7 + ("layer", "quantize", "relayout", "dequant"))
    if kind == "layer":
        while True:
            hidden, mlp = _log_size(rng, 2048, 8192, 256), _log_size(rng, 5632, 28672, 256)
            kv = max(256, hidden // rng.choice((1, 4, 8)) // 256 * 256)
            if hidden * (2 * hidden + 2 * kv + 3 * mlp) <= MAX_LAYER_WEIGHTS:
                return {"kind": kind, "E": E, "Mb": Mb, "hidden": hidden, "kv": kv, "mlp": mlp, "N": _log_size(rng, 1, 64, 1)}
    while True:
        M, K = _log_size(rng, 1024, 28672, 256), _log_size(rng, 1024, 28672, 64)
        if M * K <= MAX_WEIGHTS:
            break
    if kind == "gemm":
        entry = rng.choice(("drop-in", "native", "module"))
        N = _log_size(rng, 1, min(4096, MAX_MACS // (M * K)), 1)
        return {"kind": kind, "entry": entry, "E": E, "Mb": Mb, "M": M, "K": K, "N": N,
                "groups": entry != "drop-in" and rng.random() < 0.3, "bias": entry == "module" and rng.random() < 0.3}
    if kind == "quantize":
        return {"kind": kind, "E": E, "Mb": Mb, "M": M, "K": K, "dtype": rng.choice(("fp16", "bf16", "fp32")), "groups": rng.random() < 0.3}
    case = {"kind": kind, "E": E, "Mb": Mb, "M": M, "K": K}
    if kind == "dequant":
        case["groups"] = rng.random() < 0.3
    return case


DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16, "fp32": torch.float32}


def _weight(gen, M, K, dtype=torch.float16):
    return torch.randn(M, K, generator=gen, device=DEVICE, dtype=dtype) * 0.02


def _activations(gen, N, K):
    return torch.randn(N, K, generator=gen, device=DEVICE, dtype=torch.float16)


def _reference_layout(gen, M, K, bits):
    """Weights in the reference's prepacked layout: a permutation of the code bits, so every bit pattern is a weight matrix."""
    return torch.randint(-2 ** 31, 2 ** 31 - 1, (M, K // 32 * bits), generator=gen, device=DEVICE, dtype=torch.int64).to(torch.int32)


def _scales(gen, M):
    return (torch.rand(M, generator=gen, device=DEVICE) * 9e-3 + 1e-3).half()


def prepare(case, seed):
    gen = torch.Generator(device=DEVICE).manual_seed(seed)
    E, Mb, kind = case["E"], case["Mb"], case["kind"]
    state = {"case": case}
    if kind == "layer":
        H, KV, F, N = case["hidden"], case["kv"], case["mlp"], case["N"]
        layer = lambda M, K: FPxLinear.from_float(_weight(gen, M, K), E, Mb)   # noqa: E731
        state["qkv"] = FPxLinear.fused([layer(H, H), layer(KV, H), layer(KV, H)])
        state["o"], state["gate_up"], state["down"] = layer(H, H), FPxLinear.fused([layer(F, H), layer(F, H)]), layer(H, F)
        state["x"], state["x_mlp"] = _activations(gen, N, H), _activations(gen, N, F)
        return state
    M, K = case["M"], case["K"]
    if kind == "quantize":
        state["w"] = _weight(gen, M, K, DTYPES[case["dtype"]])
    elif kind == "relayout":
        state["packed"] = _reference_layout(gen, M, K, 1 + E + Mb)
    elif kind == "dequant":
        state["native"], state["scales"], *rest = fp6.weight_quantize_native_cuda(E, Mb, _weight(gen, M, K), case["groups"])
        state["exps"] = rest[0] if rest else None
    else:
        N = case["N"]
        state["x"] = _activations(gen, N, K)
        state["split"] = fp6.heuristic_splitk_mi355x(M, N, K, EXPONENT=E, MANTISSA=Mb)
        if case["entry"] == "drop-in":
            state["packed"], state["scales"] = _reference_layout(gen, M, K, 1 + E + Mb), _scales(gen, M)
        elif case["entry"] == "native":
            state["native"], state["scales"], *rest = fp6.weight_quantize_native_cuda(E, Mb, _weight(gen, M, K), case["groups"])
            state["exps"] = rest[0] if rest else None
        else:
            bias = torch.randn(M, generator=gen, device=DEVICE, dtype=torch.float16) if case["bias"] else None
            state["layer"] = FPxLinear.from_float(_weight(gen, M, K), E, Mb, bias=bias, group_scales=case["groups"])
    return state


def run(state):
    case = state["case"]
    E, Mb, kind = case["E"], case["Mb"], case["kind"]
    if kind == "layer":
        return [state["qkv"](state["x"]), state["o"](state["x"]), state["gate_up"](state["x"]), state["down"](state["x_mlp"])]
    M, K = case["M"], case["K"]
    if kind == "quantize":
        return fp6.weight_quantize_native_cuda(E, Mb, state["w"], case["groups"])
    if kind == "relayout":
        return fp6.to_native(state["packed"], E, Mb)
    if kind == "dequant":
        return fp6.weight_dequant_native_cuda(E, Mb, state["native"], state["scales"], M, K, state["exps"])
    if case["entry"] == "drop-in":
        return fp6.linear_forward_eXmY_cuda(E, Mb, state["x"], state["packed"], state["scales"], state["split"])
    if case["entry"] == "native":
        return fp6.linear_forward_native(E, Mb, state["x"], state["native"], state["scales"], M, state["split"], group_exps=state["exps"])
    return state["layer"](state["x"])


def _gemm_work(M, K, N, bits, groups=False, bias=False):
    extra = M * math.ceil(K / 128) if groups else 0
    return M * K * bits / 8 + extra + 2 * M * (2 if bias else 1) + 2 * N * K + 2 * N * M, 2 * M * N * K


def work(case):
    bits, kind = 1 + case["E"] + case["Mb"], case["kind"]
    if kind == "layer":
        H, KV, F, N = case["hidden"], case["kv"], case["mlp"], case["N"]
        parts = [_gemm_work(m, k, N, bits) for m, k in ((H + 2 * KV, H), (H, H), (2 * F, H), (H, F))]
        return {"bytes": sum(b for b, _ in parts), "flops": sum(f for _, f in parts)}
    M, K = case["M"], case["K"]
    if kind == "gemm":
        b, f = _gemm_work(M, K, case["N"], bits, case["groups"], case["bias"])
        return {"bytes": b, "flops": f}
    codes, exps = M * K * bits / 8, M * math.ceil(K / 128) if case.get("groups") else 0
    if kind == "quantize":
        return {"bytes": M * K * DTYPES[case["dtype"]].itemsize + codes + exps + 2 * M, "flops": 0}
    if kind == "relayout":
        return {"bytes": 2 * codes, "flops": 0}
    return {"bytes": codes + exps + 2 * M + 2 * M * K, "flops": 0}


def tolerance(case):
    if case["kind"] in ("quantize", "relayout", "dequant"):
        return "exact"
    # Four times what one rounding of an exact sum to fp16 gives (measured against float64: rel 2.1e-4, max 4.9e-4 on every
    # size and format).  A bias is a second rounding, and long prompts through a module may round scaled weights to fp16
    # first (measured: rel 3.3e-4, max 1.9e-3).
    if case["kind"] == "gemm" and case["entry"] == "module" and (case["bias"] or case["N"] >= FPxLinear.PREFILL_CROSSOVER):
        return {"rel": 1.4e-3, "max": 8e-3}
    return {"rel": 8.5e-4, "max": 2e-3}
