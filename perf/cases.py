"""The quantized linears a diffusion transformer runs, as cases to time: each
is one pass through the public entry points, on inputs made from a seed.

A case's ``kind`` says which part of a model it stands for:

  modulation    ``linear(silu(temb))``: the adaLN call of a block, one row per
                image of the batch.  Hundreds per denoising step, each as short
                as its launch.
  text_stream   the linears of a joint block's text stream: q, k, v and out as
                the reference calls them, then the GELU feed-forward with its
                gated residual.  As many rows as the prompt has tokens.
  encoder_mlp   the SwiGLU feed-forward of a text encoder's layer (gate and up
                stacked, then down), run once per prompt.
  projection    one linear by itself over everything a caller may choose: any
                number of rows, every bit width and group size, 16-bit and
                float32 activations (the attention output after rotary
                embeddings in float32), wide and narrow outputs.
  single_block  a single-stream block: LayerNorm and modulation, the stacked
                q/k/v/mlp linear with GELU on its mlp part, and the output
                linear with gate and residual, over image and text tokens.
  swiglu_block  the feed-forward of a Z-Image block over image tokens.
  lora          inference through a linear with LoRA adapters on it.
  training      forward and backward of a trainable LoRA on a quantized base.
  quantize      packing a weight at load time.

Sizes are those of the model families the tests and the benchmark use, and for
the drawn cases anything between.
"""
from __future__ import annotations

import math

import torch

from mflux_amd import core, lora, nn

_DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}


def listed():
    return [
        # Z-Image's adaLN, two per block: a row of 256 against 15360 features, the smallest call there is
        {"name": "modulation_256_w8", "kind": "modulation", "M": 1, "K": 256, "N": 15360, "bits": 8, "dtype": "bf16"},
        # FLUX.1's and Qwen-Image's adaLN of a joint block at -q 8
        {"name": "modulation_3072_w8", "kind": "modulation", "M": 1, "K": 3072, "N": 18432, "bits": 8, "dtype": "bf16"},
        # the same of a single-stream block at -q 4, for a batch of five images
        {"name": "modulation_batch_w4", "kind": "modulation", "M": 5, "K": 3072, "N": 9216, "bits": 4, "dtype": "bf16"},
        # Qwen-Image's text stream, 256 prompt tokens
        {"name": "text_stream_w4", "kind": "text_stream", "M": 256, "K": 3072, "bits": 4},
        # Qwen2.5-VL's MLP on a prompt of 320 tokens
        {"name": "encoder_mlp_w4", "kind": "encoder_mlp", "M": 320, "K": 3584, "N": 18944, "bits": 4},
        # Qwen3's q projection at -q 6 on 300 tokens
        {"name": "projection_w6", "kind": "projection", "M": 300, "K": 2560, "N": 4096, "bits": 6, "group_size": 64,
         "dtype": "bf16", "x_dtype": "bf16", "bias": False},
        # FLUX.1's to_out over 4096 image tokens that left attention in float32
        {"name": "projection_f32_w4", "kind": "projection", "M": 4096, "K": 3072, "N": 3072, "bits": 4, "group_size": 64,
         "dtype": "bf16", "x_dtype": "f32", "bias": True},
        # FLUX.1's single-stream block at 1024 x 1024: 4096 image and 512 text tokens; the largest
        {"name": "single_block_w4", "kind": "single_block", "M": 4608, "K": 3072, "bits": 4},
        # Z-Image's feed-forward at 1024 x 1024: 4096 image and 256 caption tokens
        {"name": "swiglu_block_w8", "kind": "swiglu_block", "M": 4352, "K": 3840, "N": 10240, "bits": 8},
        # a rank-16 adapter on a projection of Qwen-Image's image stream at 1328 x 1328
        {"name": "lora_w4", "kind": "lora", "M": 6889, "K": 3072, "N": 3072, "bits": 4, "rank": 16, "adapters": 1},
        # LoRA training on the MLP's first linear at 512 x 512: 1024 image and 512 text tokens
        {"name": "training_w4", "kind": "training", "M": 1536, "K": 3072, "N": 12288, "bits": 4, "rank": 16},
        # loading a bfloat16 checkpoint at -q 4: the stacked q/k/v/mlp weight of a single-stream block
        {"name": "quantize_w4", "kind": "quantize", "N": 21504, "K": 3072, "bits": 4, "group_size": 64, "dtype": "bf16"},
    ]


_MOST_FLOPS = 1.0e12   # of a drawn case; the largest listed one has 1.04e12
_HIDDEN = (2560, 3072, 3584, 3840, 4096)


def _log_int(rng, lo, hi):
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng):
    kind = rng.choice(("modulation", "modulation", "text_stream", "encoder_mlp", "projection", "projection",
                       "single_block", "swiglu_block", "lora", "training", "quantize"))
    bits = rng.choice((4, 8))
    if kind == "modulation":
        K = rng.choice((256, 2560, 3072, 3072, 3840, 4096, 6144))
        N = rng.choice((15360, 12288)) if K == 256 else K * rng.choice((2, 3, 6))
        return {"kind": kind, "M": rng.choice((1, 1, 1, rng.randint(2, 16))), "K": K, "N": N, "bits": bits,
                "dtype": rng.choice(("bf16", "bf16", "f16"))}
    if kind == "text_stream":
        return {"kind": kind, "M": _log_int(rng, 17, 1024), "K": rng.choice((2560, 3072, 3840)), "bits": bits}
    if kind == "encoder_mlp":
        K, N = rng.choice(((3584, 18944), (2560, 9728), (4096, 10240), (4096, 12288)))
        return {"kind": kind, "M": _log_int(rng, 17, 1024), "K": K, "N": N, "bits": bits}
    if kind == "projection":
        K = rng.choice((768, 1152, *_HIDDEN, 6144, 9728, 12288, 15360))
        # 512: grouped-query k/v; 4304: SigLIP's MLP; 64: the projection back to latents
        N = rng.choice((64, 512, 1024, 4304, *_HIDDEN, 9216, 12288, 21504))
        M = min(_log_int(rng, 17, 8192), int(_MOST_FLOPS / (2 * K * N)))
        return {"kind": kind, "M": M, "K": K, "N": N, "bits": rng.choice((3, 4, 4, 5, 6, 8, 8)),
                "group_size": rng.choice((64, 64, 64, 32, 128)), "dtype": rng.choice(("bf16", "bf16", "bf16", "f16")),
                "x_dtype": rng.choice(("16", "16", "f32")), "bias": rng.random() < 0.5}
    if kind == "single_block":
        return {"kind": kind, "M": _log_int(rng, 768, 4416), "K": 3072, "bits": bits}
    if kind == "swiglu_block":
        return {"kind": kind, "M": _log_int(rng, 768, 4224), "K": 3840, "N": 10240, "bits": bits}
    if kind == "lora":
        K, N = rng.choice(((3072, 3072), (3840, 3840), (3072, 12288), (12288, 3072), (3840, 10240)))
        M = min(_log_int(rng, 256, 8192), int(_MOST_FLOPS / (2 * K * N)))
        return {"kind": kind, "M": M, "K": K, "N": N, "bits": bits, "rank": rng.choice((4, 8, 16, 32, 64)),
                "adapters": rng.choice((1, 1, 2, 3))}
    if kind == "training":
        K, N = rng.choice(((3072, 3072), (3840, 3840), (3072, 12288), (12288, 3072)))
        return {"kind": kind, "M": _log_int(rng, 256, 2304), "K": K, "N": N, "bits": bits, "rank": rng.choice((4, 8, 16, 32))}
    group_size = rng.choice((32, 64, 64, 64, 128))
    return {"kind": "quantize", "N": _log_int(rng, 500, 24000), "K": group_size * rng.randint(1536 // group_size, 12288 // group_size),
            "bits": rng.choice((3, 4, 4, 5, 6, 8, 8)), "group_size": group_size, "dtype": rng.choice(("bf16", "bf16", "bf16", "f16", "f32"))}


class _Maker:
    """Seeded operands: activations N(0, 1), weights and biases N(0, 0.02), rounded once to the 16-bit type."""

    def __init__(self, seed, dtype=torch.bfloat16):
        self.gen = torch.Generator(device="cuda").manual_seed(seed)
        self.dtype = dtype

    def normal(self, *shape, std=1.0, dtype=None):
        t = torch.randn(shape, generator=self.gen, device="cuda", dtype=torch.float32)
        return t.mul_(std).to(dtype or self.dtype)

    def linear(self, K, N, bits, bias=True, group_size=64):
        layer = nn.Linear(K, N, bias=bias, device="meta", dtype=self.dtype)
        layer.weight = torch.nn.Parameter(self.normal(N, K, std=0.02), requires_grad=False)
        if bias:
            layer.bias = torch.nn.Parameter(self.normal(N, std=0.02), requires_grad=False)
        return layer.to_quantized(group_size, bits)

    def adapter(self, base, rank, scale):
        layer = lora.LoRALinear.from_linear(base, r=rank, scale=scale)
        for p in (layer.lora_A, layer.lora_B):  # trained adapters: both factors away from zero
            p.data.copy_(self.normal(*p.shape, std=0.02))
        return layer


def _x_dtype(case):
    return _DTYPES[case["dtype"] if case["x_dtype"] == "16" else case["x_dtype"]]


def prepare(case, seed):
    kind = case["kind"]
    make = _Maker(seed, _DTYPES[case.get("dtype", "bf16")])
    K, N, M, bits = case["K"], case.get("N"), case.get("M"), case["bits"]
    state = dict(case)
    if kind == "quantize":
        state["w"] = make.normal(N, K, std=0.02)
        return state
    state["x"] = make.normal(M, K)
    if kind == "modulation":
        state["layer"] = make.linear(K, N, bits)
    elif kind == "text_stream":
        state["qkvo"] = [make.linear(K, K, bits) for _ in range(4)]
        state["up"], state["down"] = make.linear(K, 4 * K, bits), make.linear(4 * K, K, bits)
        state["attended"], state["residual"], state["gate"] = make.normal(M, K), make.normal(M, K), make.normal(K)
    elif kind in ("encoder_mlp", "swiglu_block"):
        state["gate_up"] = nn.stack_gate_up(make.linear(K, N, bits, bias=False), make.linear(K, N, bits, bias=False))
        state["down"] = make.linear(N, K, bits, bias=False)
        if kind == "swiglu_block":
            state["residual"], state["gate"] = make.normal(M, K), make.normal(K)
    elif kind == "projection":
        state["x"] = make.normal(M, K, dtype=_x_dtype(case))
        state["layer"] = make.linear(K, N, bits, bias=case["bias"], group_size=case["group_size"])
    elif kind == "single_block":
        state["qkv_mlp"], state["out"] = make.linear(K, 7 * K, bits), make.linear(5 * K, K, bits)
        state["scale"], state["shift"], state["gate"] = make.normal(K, std=0.1), make.normal(K, std=0.1), make.normal(K)
        state["attended"] = make.normal(M, 5 * K)
    elif kind == "lora":
        base = make.linear(K, N, bits)
        adapters = [make.adapter(base, case["rank"], 1.0 / (1 + i)) for i in range(case["adapters"])]
        state["layer"] = adapters[0] if len(adapters) == 1 else lora.FusedLoRALinear(base, adapters)
    elif kind == "training":
        state["layer"] = make.adapter(make.linear(K, N, bits), case["rank"], 1.0)
        state["x"].requires_grad_(True)
        state["grad"] = make.normal(M, N)
    else:
        raise ValueError(f"unknown kind {kind}")
    return state


def run(state):
    kind = state["kind"]
    if kind == "quantize":
        codes, scales, biases = core.quantize(state["w"], state["group_size"], state["bits"])
        return codes.view(torch.int32), scales, biases
    if kind == "training":
        layer, x = state["layer"], state["x"]
        y = layer(x)
        return (y, *torch.autograd.grad(y, (x, layer.lora_A, layer.lora_B), state["grad"]))
    with torch.no_grad():
        x = state["x"]
        if kind == "modulation":
            return nn.silu_linear(state["layer"], x)
        if kind in ("projection", "lora"):
            return state["layer"](x)
        if kind == "text_stream":
            to_q, to_k, to_v, to_out = state["qkvo"]
            q, k, v = to_q(x), to_k(x), to_v(x)
            h = nn.gate_residual_linear(to_out, state["attended"], state["gate"], state["residual"])
            return q, k, v, h, nn.gate_residual_linear(state["down"], nn.gelu_linear(state["up"], x), state["gate"], h)
        if kind == "encoder_mlp":
            return state["down"](nn.swiglu_linear(state["gate_up"], x))
        if kind == "swiglu_block":
            return nn.gate_residual_linear(state["down"], nn.swiglu_linear(state["gate_up"], x), state["gate"],
                                           state["residual"])
        # single_block: attention between the two linears is not this package's; its result stands ready
        h = nn.layer_norm_modulate(x, state["scale"], state["shift"])
        y = nn.gelu_linear(state["qkv_mlp"], h, act_from=3 * x.shape[1])
        return y, nn.gate_residual_linear(state["out"], state["attended"], state["gate"], x)


def _weight_bytes(K, N, bits, group_size=64):
    return N * K * bits / 8 + 4 * N * K / group_size + 2 * N


def work(case):
    """Every input read once, every output written once; what passes between the calls of a case not at all."""
    kind, K, N, bits = case["kind"], case["K"], case.get("N"), case["bits"]
    gs = case.get("group_size", 64)
    if kind == "quantize":
        size = 4 if case["dtype"] == "f32" else 2
        return {"bytes": N * K * (size + bits / 8) + 2 * size * N * K / gs, "flops": 0}
    M = case["M"]
    if kind in ("modulation", "projection"):
        size = 4 if case.get("x_dtype") == "f32" else 2
        return {"bytes": _weight_bytes(K, N, bits, gs) + size * M * (K + N), "flops": 2 * M * K * N}
    if kind == "text_stream":
        return {"bytes": 12 * _weight_bytes(K, K, bits) + 2 * M * 8 * K, "flops": 2 * M * 12 * K * K}
    if kind == "encoder_mlp":
        return {"bytes": 3 * _weight_bytes(K, N, bits) + 2 * M * 2 * K, "flops": 2 * M * 3 * K * N}
    if kind == "swiglu_block":
        return {"bytes": 3 * _weight_bytes(K, N, bits) + 2 * M * 3 * K, "flops": 2 * M * 3 * K * N}
    if kind == "single_block":
        return {"bytes": 12 * _weight_bytes(K, K, bits) + 2 * M * (K + 7 * K + 5 * K + K), "flops": 2 * M * 12 * K * K}
    rank = case["rank"] * case.get("adapters", 1)
    update = 2 * rank * (K + N)
    if kind == "lora":
        return {"bytes": _weight_bytes(K, N, bits) + update + 2 * M * (K + N), "flops": 2 * M * (K * N + rank * (K + N))}
    # training: y = x W + (x A) B, dx = g W^T + (g B^T) A^T, dA = x^T (g B^T), dB = (x A)^T g
    return {"bytes": _weight_bytes(K, N, bits) + 2 * update + 2 * M * (2 * K + 2 * N),
            "flops": 2 * M * (2 * K * N + 3 * rank * (K + N))}


def tolerance(case):
    """Packing is exact.  Products: an implementation may round the dequantised
    weights to 16 bits or keep them, and rounds its result (and, where calls
    follow one another, what passes between them) to 16 bits: 2^-9 per rounding
    in bfloat16, 2^-12 in float16, relative to the value rounded."""
    if case["kind"] == "quantize":
        return "exact"
    return {"rel": 2e-3 if case.get("dtype") == "f16" else 1e-2}
