"""Performance cases of the quantized-matmul framework.

Each case is one call (or the short run of calls a program makes for one layer) through the
public entry points: the packed int4 linear layer (``quant_linear.QuantLinear``), the drop-in
int4 matmul (``gemm_int4.int4_gemm``), the fp8 path (``gemm_fp8``), the dense matmuls
(``gemm.triton_gemm``, ``gemm_splitk.triton_gemm_splitk``), split-KV decode attention
(``flash_decoding``) and the packing of a layer's weights (``gemm_int4.quantize_int4_group``).
GPTQ is not among them: a rounding decided the other way in one column changes every later
column, so two correct fp32 implementations differ by a large part of a quantization step.

Layer sizes are those of the benchmark (the decode GEMV's 4096 x 11008, the Llama-3-8B
projections, 4096 x 4096 prefill) and of the reference's own benchmark tables; drawn cases
spread over the same ranges with odd sizes among them.
"""

from __future__ import annotations

import math
import os
import sys

import torch

# the package directory's name is no Python identifier: its modules are imported by their own
# names, as the reference's callers import them
sys.path.insert(1, os.path.join(os.getcwd(), "pico-kernels_amd"))

import flash_decoding  # noqa: E402
import gemm  # noqa: E402
import gemm_fp8  # noqa: E402
import gemm_int4  # noqa: E402
import gemm_splitk  # noqa: E402
from quant_linear import QuantLinear  # noqa: E402

GROUP = 128
DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16, "fp32": torch.float32}


def listed() -> list[dict]:
    return [
        # one token of one sequence through the widest layer of the decode benchmark
        dict(name="decode_1", kind="linear", M=1, K=4096, N=11008, dtype="fp16", bias=False,
             scheme="group"),
        # a decode step of eight sequences in a bf16 model, the MLP's down projection
        dict(name="decode_8_bf16", kind="linear", M=8, K=14336, N=4096, dtype="bf16", bias=False,
             scheme="group"),
        # a decode step of a serving batch, the MLP's gate / up projection
        dict(name="batch_32", kind="linear", M=32, K=4096, N=14336, dtype="fp16", bias=False,
             scheme="group"),
        # a short prompt of odd length through a biased projection of a bf16 model that was
        # quantized the reference's way (one scale per input feature)
        dict(name="prompt_333_per_input", kind="linear", M=333, K=4096, N=6144, dtype="bf16",
             bias=True, scheme="per_input"),
        # prefill of a 2048-token prompt
        dict(name="prefill_2048", kind="linear", M=2048, K=4096, N=4096, dtype="fp16", bias=False,
             scheme="group"),
        # the drop-in per-tensor matmul on pack_int4_n's bytes, the reference's decode row
        dict(name="int4_gemm_16", kind="int4", M=16, K=4096, N=4096, dtype="fp16"),
        # fp8 matmul on operands cast beforehand, the reference's largest row
        dict(name="fp8_precast_4096", kind="fp8", M=4096, K=4096, N=4096, dtype="fp16", cast=False),
        # an fp8 layer in use: weights cast once, activations quantized on every call
        dict(name="fp8_layer_1000", kind="fp8", M=1000, K=4096, N=6144, dtype="bf16", cast=True),
        # dense 16-bit matmul
        dict(name="dense_2048_bf16", kind="dense", M=2048, K=4096, N=4096, dtype="bf16", split=1),
        # one decode step over a short cache: the reference's smallest row, a launch's latency
        dict(name="attention_1k", kind="attention", B=2, H=4, N=1024, D=64, split=256, room=4096),
        # one decode step of a batch over long caches
        dict(name="attention_8k", kind="attention", B=8, H=32, N=8192, D=128, split=256, room=8192),
        # loading a model: the MLP's gate / up projection quantized to int4 groups and packed
        dict(name="pack_4096x14336", kind="pack", K=4096, N=14336, dtype="fp16"),
    ]


def _log(rng, lo: float, hi: float) -> int:
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng) -> dict:
    kind = rng.choice(["linear", "linear", "linear", "linear", "int4", "fp8", "dense", "attention",
                       "pack"])
    if kind == "linear":
        scheme = rng.choice(["group", "group", "per_input"])
        # in % 128 (the group), out % 16; half of them whole 256-column tiles
        n = 256 * rng.randint(4, 56) if rng.random() < 0.5 else 16 * rng.randint(64, 896)
        return dict(kind=kind, M=_log(rng, 1, 2048), K=128 * rng.randint(8, 64), N=n,
                    dtype=rng.choice(["fp16", "bf16"]), bias=rng.random() < 0.3, scheme=scheme)
    if kind == "int4":
        return dict(kind=kind, M=_log(rng, 1, 2048), K=32 * rng.randint(32, 256),
                    N=8 * rng.randint(128, 1024), dtype=rng.choice(["fp16", "fp16", "bf16"]))
    if kind == "fp8":
        return dict(kind=kind, M=_log(rng, 16, 4096), K=16 * rng.randint(32, 256),
                    N=16 * rng.randint(32, 384), dtype=rng.choice(["fp16", "bf16", "fp32"]),
                    cast=rng.random() < 0.5)
    if kind == "dense":
        split = rng.choice([1, 1, 4, 8])
        if split > 1:  # few output tiles and a long K, where a split is asked for
            return dict(kind=kind, M=256 * rng.randint(1, 4), K=64 * split * rng.randint(8, 32),
                        N=256 * rng.randint(1, 4), dtype=rng.choice(["fp16", "bf16"]), split=split)
        return dict(kind=kind, M=256 * rng.randint(1, 16), K=64 * rng.randint(8, 64),
                    N=256 * rng.randint(1, 16), dtype=rng.choice(["fp16", "bf16"]), split=1)
    if kind == "attention":
        split = rng.choice([64, 128, 256, 256])
        n = split * max(1, _log(rng, 256, 8192) // split)
        return dict(kind=kind, B=rng.randint(1, 8), H=rng.choice([4, 8, 12, 16, 32]), N=n,
                    D=rng.choice([64, 128]), split=split, room=n + 64 * rng.randint(0, 16))
    return dict(kind=kind, K=128 * rng.randint(4, 64), N=8 * rng.randint(64, 1792),
                dtype=rng.choice(["fp16", "bf16", "fp32"]))


# ---------------------------------------------------------------------------------------
# inputs (made from the seed alone)
# ---------------------------------------------------------------------------------------
def _gen(seed: int) -> torch.Generator:
    return torch.Generator(device="cuda").manual_seed(seed)


def _randn(g, *shape, scale: float = 1.0, dtype=torch.float16) -> torch.Tensor:
    return (torch.randn(*shape, generator=g, device="cuda") * scale).to(dtype)


def _inputs(case: dict, seed: int) -> dict:
    g, kind = _gen(seed), case["kind"]
    if kind == "linear":
        dt = DTYPES[case["dtype"]]
        return {"x": _randn(g, case["M"], case["K"], dtype=dt),
                "w": _randn(g, case["N"], case["K"], scale=0.02, dtype=dt),
                "b": _randn(g, case["N"], scale=0.1, dtype=dt) if case["bias"] else None}
    if kind == "int4":
        return {"a": _randn(g, case["M"], case["K"], dtype=DTYPES[case["dtype"]]),
                "w": _randn(g, case["K"], case["N"], scale=0.02)}
    if kind == "fp8":
        dt = DTYPES[case["dtype"]]
        return {"a": _randn(g, case["M"], case["K"], dtype=dt),
                "b": _randn(g, case["K"], case["N"], scale=0.02, dtype=dt)}
    if kind == "dense":
        dt = DTYPES[case["dtype"]]
        return {"a": _randn(g, case["M"], case["K"], dtype=dt),
                "b": _randn(g, case["K"], case["N"], dtype=dt)}
    if kind == "attention":
        B, H, N, D = case["B"], case["H"], case["N"], case["D"]
        return {"q": _randn(g, B, H, 1, D), "k": _randn(g, B, H, N, D), "v": _randn(g, B, H, N, D)}
    return {"w": _randn(g, case["K"], case["N"], scale=0.02, dtype=DTYPES[case["dtype"]])}


# ---------------------------------------------------------------------------------------
# what a program holds before the call, and the call
# ---------------------------------------------------------------------------------------
def prepare(case: dict, seed: int) -> dict:
    t, kind = _inputs(case, seed), case["kind"]
    if kind == "linear":
        lin = torch.nn.Linear(case["K"], case["N"], bias=case["bias"], device="meta")
        lin.weight = torch.nn.Parameter(t["w"], requires_grad=False)
        if case["bias"]:
            lin.bias = torch.nn.Parameter(t["b"], requires_grad=False)
        method = "rtn" if case["scheme"] == "per_input" else None
        return {"kind": kind, "layer": QuantLinear.from_linear(lin, GROUP, method), "x": t["x"]}
    if kind == "int4":
        codes, scale = gemm_int4.quantize_int4(t["w"])
        return {"kind": kind, "a": t["a"], "w": gemm_int4.pack_int4_n(codes), "scale": scale}
    if kind == "fp8":
        b8, sb = gemm_fp8.quantize(t["b"])
        if case["cast"]:
            return {"kind": kind, "a": t["a"], "b8": b8, "sb": sb}
        a8, sa = gemm_fp8.quantize(t["a"])
        return {"kind": kind, "a8": a8, "sa": sa, "b8": b8, "sb": sb}
    if kind == "dense":
        return {"kind": kind, "split": case["split"], **t}
    if kind == "attention":
        cache = flash_decoding.KVCache(case["B"], case["H"], case["D"], case["room"], "cuda")
        cache.k.zero_()
        cache.v.zero_()
        n = case["N"]
        cache.k[:, :, :n] = t["k"]
        cache.v[:, :, :n] = t["v"]
        cache.pos = n
        return {"kind": kind, "q": t["q"], "cache": cache, "split": case["split"]}
    return {"kind": kind, **t}


def run(s: dict):
    kind = s["kind"]
    if kind == "linear":
        return s["layer"](s["x"])
    if kind == "int4":
        return gemm_int4.int4_gemm(s["a"], s["w"], s["scale"])
    if kind == "fp8":
        a8, sa = gemm_fp8.quantize(s["a"]) if "a" in s else (s["a8"], s["sa"])
        return gemm_fp8.fp8_gemm_precast(a8, sa, s["b8"], s["sb"])
    if kind == "dense":
        if s["split"] == 1:
            return gemm.triton_gemm(s["a"], s["b"])
        return gemm_splitk.triton_gemm_splitk(s["a"], s["b"], split_k=s["split"])
    if kind == "attention":
        cache = s["cache"]
        return flash_decoding.flash_decoding(s["q"], cache.k[:, :, :cache.pos],
                                             cache.v[:, :, :cache.pos], split_size=s["split"])
    return gemm_int4.quantize_int4_group(s["w"], GROUP)


# ---------------------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------------------
def work(case: dict) -> dict:
    kind = case["kind"]
    if kind == "attention":
        B, H, N, D = case["B"], case["H"], case["N"], case["D"]
        return {"bytes": 4 * B * H * N * D + 6 * B * H * D, "flops": 4 * B * H * N * D}
    if kind == "pack":  # the weights in, codes and fp16 scales out; a divide and a round each
        K, N = case["K"], case["N"]
        es = 4 if case["dtype"] == "fp32" else 2
        return {"bytes": es * K * N + K * N // 2 + 2 * (K // GROUP) * N, "flops": 3 * K * N}
    M, K, N = case["M"], case["K"], case["N"]
    flops = 2 * M * K * N
    if kind == "linear":  # activations and outputs in 16 bits, codes, scales
        scales = 2 * (K // GROUP) * N if case["scheme"] == "group" else 4 * K
        return {"bytes": 2 * M * (K + N) + K * N // 2 + scales + 2 * N * case["bias"], "flops": flops}
    if kind == "int4":
        return {"bytes": 2 * M * K + K * N // 2 + 4 * M * N, "flops": flops}
    es = 4 if case["dtype"] == "fp32" else 2
    if kind == "fp8":
        return {"bytes": (es if case["cast"] else 1) * M * K + K * N + 4 * M * N, "flops": flops}
    return {"bytes": 2 * K * (M + N) + 4 * M * N, "flops": flops}


def tolerance(case: dict):
    kind = case["kind"]
    if kind == "pack":
        return "exact"
    if kind == "linear":  # one rounding to the 16-bit output; fp16 dequantized weights in prefill
        return {"rel": 1e-3 if case["dtype"] == "fp16" else 6e-3}
    # fp32 sums of exact products; 1.4e-5 from the 64-bit result is seen for int4 and fp8 operands
    return {"rel": 6e-5 if kind in ("int4", "fp8") else 1e-5}


# ---------------------------------------------------------------------------------------
# the same results in 64 bits
# ---------------------------------------------------------------------------------------
def _rtn(w: torch.Tensor, group: int) -> tuple[torch.Tensor, torch.Tensor]:
    """int4 codes of (K, N) fp32 weights and their (groups, N) fp32 scales, groups along K."""
    K, N = w.shape
    wg = w.view(K // group, group, N)
    a = wg.abs().amax(1).clamp_min(1e-12)
    s = a / torch.full_like(a, 7)  # tensor by tensor: a true division
    return torch.clamp(torch.round(wg / s[:, None]), -7, 7).view(K, N), s


def _cast_fp8(x: torch.Tensor) -> tuple[torch.Tensor, float]:
    scale = torch.finfo(torch.float8_e4m3fn).max / x.abs().max().item()
    return (x * scale).to(torch.float8_e4m3fn).double(), scale


def exact(case: dict, seed: int):
    t, kind = _inputs(case, seed), case["kind"]
    if kind == "linear":
        w = t["w"].float()
        if case["scheme"] == "group":
            q, s = _rtn(w.t().contiguous(), GROUP)
            wd = (q.view(-1, GROUP, case["N"]).double() * s.half().double()[:, None]).view(-1, case["N"])
        else:
            # the layer is packed from the quantized weight in the model's own dtype: each
            # input feature's scale is read back from that
            q, s = _rtn(w, case["N"])
            s = (q * s).to(t["w"].dtype).double().abs().amax(0, keepdim=True) / 7
            wd = (q.double() * s).t()
        y = t["x"].double() @ wd
        return y if t["b"] is None else y + t["b"].half().double()
    if kind == "int4":
        w = t["w"]
        scale = w.abs().max().item() / 7.0
        div = torch.full((), scale, dtype=torch.float32, device="cuda").expand_as(w)
        q = torch.round((w.float() / div).to(w.dtype)).clamp(-8, 7)
        return t["a"].double() @ q.double() * scale
    if kind == "fp8":
        (a, sa), (b, sb) = _cast_fp8(t["a"]), _cast_fp8(t["b"])
        return a @ b / (sa * sb)
    if kind == "dense":
        return t["a"].double() @ t["b"].double()
    if kind == "attention":
        outs = []
        for q, k, v in zip(t["q"].double(), t["k"], t["v"]):  # one sequence at a time
            p = torch.softmax((k.double() * q).sum(-1) / math.sqrt(case["D"]), -1)
            outs.append((p[..., None] * v.double()).sum(1, keepdim=True))
        return torch.stack(outs)
    q, s = _rtn(t["w"].float(), GROUP)
    nib = (q.to(torch.int32) & 15).view(case["K"], case["N"] // 8, 8)
    words = torch.zeros_like(nib[..., 0])
    for i in range(8):  # column 8j + i in nibble i of word j
        words |= nib[..., i] << (4 * i)
    return words, s.half()
