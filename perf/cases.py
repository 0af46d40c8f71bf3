"""The performance cases of this framework: the calls a diffusion transformer makes of the INT8 convrot linear and of
the low-rank linear, from a few conditioning rows to a whole clip's tokens.

A case names one call (``kind``) and its sizes:

* ``layer``: one `Int8RotLinear` forward on tokens [1, M, K] (rotation + quantization, low-rank projection, INT8 GEMM
  with its epilogue); ``rank``, ``bias`` and ``activation`` are the module's own options.
* ``qkv``: three `Int8RotLinear` projections of one input that share its quantized form (`keep_input`).
* ``ffn``: an up projection with its fused activation, then the down projection back.
* ``lowrank``: one standalone `LowRankLinear` forward.
* ``rotate``: the rotation and quantization of an activation by itself, in either arithmetic.

Activations are N(0, 1) with 0.5 % outlier channels 30 times as large, the shape of a transformer block's inputs;
weights are N(0, 1/K) rows quantized by their absmax, as a checkpoint's are. Everything lies in HBM in the layouts
that the modules keep.
"""

from __future__ import annotations

import math

import torch

from hyperflow_h3_flash_amd import Int8RotLinear, LowRankLinear
from hyperflow_h3_flash_amd.int8 import rotate_quant

#: The Hadamard group of the released checkpoints.
GROUP = 256
#: The most int8 operations of a listed case (the gated up-projection); a drawn case stays below.
MOST_OPS = 2.0 * 32768 * 28672 * 5376


def _layer(name, M, K, N, rank, bias=False, activation="none"):
    return {"name": name, "kind": "layer", "M": M, "K": K, "N": N, "rank": rank, "bias": bias,
            "activation": activation, "group": GROUP}


def listed():
    return [
        # Conditioning rows (timestep and text embeddings): the smallest calls, where launches and latency count.
        _layer("rows64_5120", 64, 5120, 5120, 32),
        # A few hundred rows against a wide modulation projection: the weight stream is the work.
        _layer("rows256_wide", 256, 5120, 30720, 32),
        # A small model's square projection with every option of the epilogue.
        _layer("rows1024_3072_bias", 1024, 3072, 3072, 32, bias=True),
        # A low-resolution image's tokens, none of the sizes a multiple of a tile.
        _layer("rows1000_ragged", 1000, 5120, 5000, 64, bias=True),
        # The q, k and v projections of one block on a short token window, sharing one quantized input; no low-rank
        # term, as the released INT8 layers are.
        {"name": "qkv_shared_2048", "kind": "qkv", "M": 2048, "K": 5376, "N": 7168, "rank": 0, "group": GROUP},
        # One GPU's share of a clip's tokens under an 8-way sequence split: the attention output projection ...
        _layer("shard5168_out", 5168, 5120, 5120, 64),
        # ... and the feed-forward, tanh-GELU fused, both projections.
        {"name": "shard5168_ffn", "kind": "ffn", "M": 5168, "K": 5120, "F": 13824, "rank": 64,
         "activation": "gelu_tanh", "group": GROUP},
        # The fused q/k/v projection on a long clip: the framework's headline workload.
        _layer("clip32768_qkv", 32768, 5120, 15360, 64),
        # The model's gated up projection, SwiGLU fused: the largest call.
        _layer("clip32768_swiglu", 32768, 5376, 28672, 64, activation="swiglu"),
        # The model's down projection on a 5.2 s clip: deep K, ragged rows.
        _layer("clip37710_down", 37710, 14336, 5376, 64),
        # A projection kept in low-rank form on the same clip.
        {"name": "clip37710_lowrank", "kind": "lowrank", "M": 37710, "K": 5376, "N": 7168, "rank": 256},
        # The rotation and quantization by itself, in the arithmetic of the reference's GPU pipeline.
        {"name": "clip32768_rotate", "kind": "rotate", "M": 32768, "K": 5120, "arithmetic": "bf16_div",
         "group": GROUP},
    ]


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(["layer"] * 5 + ["qkv", "ffn", "lowrank", "rotate"])
    while True:
        # Rows: half the draws below a few thousand, odd numbers as likely as even ones.
        M = _log_int(rng, 1 if kind == "layer" else 16, 41344)
        K = 256 * rng.randint(12, 56)  # 3072 .. 14336
        rank = rng.choice([0, 16, 32, 64, 64, 64])
        if kind == "layer":
            N = _log_int(rng, 2048, 30720)
            activation = rng.choice(["none", "none", "none", "gelu_tanh", "swiglu"])
            N -= N % (32 if activation == "swiglu" else 8)
            case = {"kind": kind, "M": M, "K": K, "N": N, "rank": rank, "bias": rng.random() < 0.3,
                    "activation": activation, "group": rng.choice([64, 256, 256, 256])}
            ops = 2.0 * M * K * N
        elif kind == "qkv":
            N = _log_int(rng, 2048, 8192)
            N -= N % 8
            case = {"kind": kind, "M": M, "K": K, "N": N, "rank": rank, "group": GROUP}
            ops = 6.0 * M * K * N
        elif kind == "ffn":
            K = 256 * rng.randint(12, 24)
            F = 256 * rng.randint(32, 56)
            case = {"kind": kind, "M": M, "K": K, "F": F, "rank": rank,
                    "activation": rng.choice(["gelu_tanh", "swiglu"]), "group": GROUP}
            ops = (6.0 if case["activation"] == "swiglu" else 4.0) * M * K * F
        elif kind == "lowrank":
            N = _log_int(rng, 2048, 28672)
            N -= N % 8
            case = {"kind": kind, "M": M, "K": K, "N": N, "rank": 8 * rng.randint(8, 80)}
            ops = 2.0 * M * case["rank"] * (K + N)
        else:
            case = {"kind": kind, "M": M, "K": K, "arithmetic": rng.choice(["bf16_div", "f32_recip"]),
                    "group": rng.choice([64, 256, 256, 1024])}
            if K % case["group"]:
                continue
            ops = 1.0
        if ops <= MOST_OPS:
            return case


def _tokens(M, K, gen):
    x = torch.randn(M, K, device="cuda", generator=gen)
    cols = torch.randperm(K, device="cuda", generator=gen)[: -(-K * 5 // 1000)]
    x[:, cols] *= 30.0
    return x.to(torch.bfloat16)


def _weights(K, N, rank, bias, gen):
    """{qweight, wscale[, down, up][, bias]} of one layer."""
    w = torch.randn(N, K, device="cuda", generator=gen) / math.sqrt(K)
    wscale = w.abs().amax(1) / 127
    t = {"qweight": (w / wscale[:, None]).round_().to(torch.int8), "wscale": wscale}
    if rank:
        t["down"] = (torch.randn(rank, K, device="cuda", generator=gen) / math.sqrt(K)).to(torch.bfloat16)
        t["up"] = (torch.randn(N, rank, device="cuda", generator=gen) * (0.3 / math.sqrt(rank))).to(torch.bfloat16)
    if bias:
        t["bias"] = (torch.randn(N, device="cuda", generator=gen) * 0.1).to(torch.bfloat16)
    return t


def _layers(case):
    """(K, N, bias, activation) of each INT8 layer of a case, in the order of their calls."""
    kind = case["kind"]
    if kind == "layer":
        return [(case["K"], case["N"], case["bias"], case["activation"])]
    if kind == "qkv":
        return [(case["K"], case["N"], False, "none")] * 3
    if kind == "ffn":
        wide = case["F"] * (2 if case["activation"] == "swiglu" else 1)
        return [(case["K"], wide, False, case["activation"]), (case["F"], case["K"], False, "none")]
    return []


def _inputs(case, seed):
    """The tensors of a case, from the seed alone: (tokens [M, K], one dict of weights for each layer)."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    x = _tokens(case["M"], case["K"], gen)
    if case["kind"] == "lowrank":
        K, N, r = case["K"], case["N"], case["rank"]
        down = (torch.randn(r, K, device="cuda", generator=gen) / math.sqrt(K)).to(torch.bfloat16)
        up = (torch.randn(N, r, device="cuda", generator=gen) / math.sqrt(r)).to(torch.bfloat16)
        return x, [{"down": down, "up": up}]
    return x, [_weights(K, N, case["rank"], bias, gen) for K, N, bias, _ in _layers(case)]


def prepare(case, seed):
    x, tensors = _inputs(case, seed)
    kind = case["kind"]
    if kind == "rotate":
        return {"kind": kind, "x": x, "group": case["group"], "arithmetic": case["arithmetic"]}
    if kind == "lowrank":
        with torch.device("cuda"):
            layer = LowRankLinear(case["K"], case["N"], case["rank"]).to(torch.bfloat16)
        layer.requires_grad_(False)
        layer.down.weight.copy_(tensors[0]["down"])
        layer.up.weight.copy_(tensors[0]["up"])
        return {"kind": kind, "x": x[None], "layers": [layer]}
    layers = []
    for (K, N, bias, activation), t in zip(_layers(case), tensors):
        with torch.device("cuda"):
            layer = Int8RotLinear(K, N, case["group"], rank=case["rank"], bias=bias,
                                  activation=None if activation == "none" else activation)
        with torch.no_grad():
            layer.qweight.copy_(t["qweight"])
            layer.wscale.copy_(t["wscale"])
            if case["rank"]:
                layer.down.weight.copy_(t["down"])
                layer.up.weight.copy_(t["up"])
            if bias:
                layer.bias.copy_(t["bias"])
        layers.append(layer)
    if kind == "qkv":  # the last reader of the input leaves nothing behind
        layers[0].keep_input = layers[1].keep_input = True
    return {"kind": kind, "x": x[None], "layers": layers}


def run(state):
    kind, x = state["kind"], state["x"]
    if kind == "rotate":
        return rotate_quant(x, state["group"], state["arithmetic"])
    layers = state["layers"]
    if kind == "qkv":
        return [layer(x) for layer in layers]
    if kind == "ffn":
        return layers[1](layers[0](x))
    return layers[0](x)


def _glu(activation):
    return activation in ("swiglu", "swiglu_gate_first")


def work(case):
    """Every tensor a call reads or writes once: tokens, weights, scales, low-rank factors and outputs (the codes only
    where they are the output); 2 operations for each multiply-add of the GEMM and the low-rank products."""
    M, K = case["M"], case["K"]
    if case["kind"] == "rotate":
        return {"bytes": 3 * M * K + 4 * M, "flops": 2 * M * K * int(math.log(case["group"], 4) + 0.5)}
    r = case["rank"]
    if case["kind"] == "lowrank":
        N = case["N"]
        return {"bytes": 2 * (M * K + r * (K + N) + M * N), "flops": 2 * M * r * (K + N)}
    layers = _layers(case)
    nbytes, flops = 2 * M * K, 0
    for k, n, bias, activation in layers:
        nbytes += n * k + 4 * n + 2 * r * (k + n) + (2 * n if bias else 0)
        flops += 2 * M * n * k + 2 * M * r * (k + n)
        if case["kind"] != "ffn" or n == K:
            nbytes += 2 * M * (n // 2 if _glu(activation) else n)
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    if case["kind"] == "rotate":
        # Codes and scales are defined to the bit: exact sums, one rounding, true divisions.
        return "exact"
    # One bf16 rounding of each output (2^-9 of it at most): 1.7e-3 in the mean from exact(); 2.3e-3 with the low-rank
    # linear's bf16 intermediate, 3.4e-3 for a gated output (three roundings), 7.3e-3 for a chained layer, whose input
    # codes move with the roundings before it. About four times that each.
    if case["kind"] == "ffn":
        return {"rel": 2.5e-2, "max": 0.15}
    if case["kind"] == "lowrank":
        return {"rel": 1e-2, "max": 5e-2}
    if case.get("activation", "none") != "none":
        return {"rel": 1.4e-2, "max": 6e-2}
    return {"rel": 7e-3, "max": 2e-2}


# ---- exact(): the layers' definition in torch float64 ----


def _round_bits(v, bits):
    """v (float64, no subnormals) rounded once to `bits` significant bits, ties to even."""
    power = (v.view(torch.int64) & 0x7FF0000000000000).view(torch.float64)  # 2^exponent: every product here is exact
    r = torch.round(v / power * 2.0 ** (bits - 1)).mul_(2.0 ** (1 - bits)).mul_(power)
    return torch.where(v == 0, v, r)


def _hadamard(group):
    h4 = torch.tensor([[1, 1, 1, -1], [1, 1, -1, 1], [1, -1, 1, 1], [-1, 1, 1, 1]], dtype=torch.float64) / 2
    h = torch.ones(1, 1, dtype=torch.float64)
    while h.shape[0] < group:
        h = torch.kron(h, h4)
    return h.cuda()


def _codes(x, group, arithmetic="bf16_div"):
    """Codes (float64, whole) and scales (float64, fp32 values) of x [M, K] float64."""
    rot = (x.reshape(-1, group) @ _hadamard(group)).reshape(x.shape)
    rot = _round_bits(rot, 8 if arithmetic == "bf16_div" else 24)
    # A quotient rounded to float64 and then to fp32 is the fp32 quotient: 53 bits are more than twice 24 and two.
    sx = _round_bits(rot.abs().amax(1, keepdim=True).clamp_min(torch.tensor(1e-12).double().item()) / 127.0, 24)
    if arithmetic == "bf16_div":
        q = _round_bits(rot / sx, 24)
    else:
        q = _round_bits(rot * _round_bits(1.0 / sx, 24), 24)
    return q.round_().clamp_(-127, 127), sx


def _exact_layer(x, t, case, activation, codes=None):
    """One layer's output in float64 for x float64 [M, K] (rows in parts)."""
    w = t["qweight"].double()
    out = []
    step = max(64, (1 << 28) // max(w.shape))
    for i in range(0, x.shape[0], step):
        part = x[i:i + step].double()
        q, sx = _codes(part, case["group"])
        y = (q @ w.t()).mul_(sx).mul_(t["wscale"].double())
        if "down" in t:
            y += (part @ t["down"].double().t()) @ t["up"].double().t()
        if "bias" in t:
            y += t["bias"].double()
        if activation == "gelu_tanh":
            y = torch.nn.functional.gelu(y, approximate="tanh")
        elif activation == "swiglu":
            h, g = y.chunk(2, -1)
            y = h * torch.nn.functional.silu(g)
        out.append(y)
    return torch.cat(out)


def exact(case, seed):
    x, tensors = _inputs(case, seed)
    kind = case["kind"]
    if kind == "rotate":
        parts = [_codes(x[i:i + 4096].double(), case["group"], case["arithmetic"]) for i in range(0, x.shape[0], 4096)]
        return torch.cat([q for q, _ in parts]).to(torch.int8), torch.cat([s for _, s in parts]).reshape(-1)
    if kind == "lowrank":
        t = tensors[0]
        down, up = t["down"].double(), t["up"].double()
        y = torch.cat([(x[i:i + 4096].double() @ down.t()) @ up.t() for i in range(0, x.shape[0], 4096)])
        return y[None]
    acts = [activation for _, _, _, activation in _layers(case)]
    if kind == "qkv":
        return [_exact_layer(x, t, case, "none")[None] for t in tensors]
    y = _exact_layer(x, tensors[0], case, acts[0])
    if kind == "ffn":  # the layers hand bf16 tokens on
        y = _exact_layer(_round_bits(y, 8), tensors[1], case, acts[1])
    return y[None]
