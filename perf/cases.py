"""The calls whose speed is measured: the FP8 block-scaled linear and its fused producers as an
engine makes them, from one decode row to a 16384-row prefill.

Every case runs public entry points of ``minillm_amd`` on synthetic tensors of the Qwen3-4B
projection sizes (or generic odd ones): weights N(0, 0.02) block-quantized to e4m3fn with fp32
128x128 scales, activations N(0, 1) with 1 % of the channels 20 times larger.

Kinds of case (``kind``):

* ``linear``  one ``mi355x_fp8_linear`` call.
* ``qkv``     the merged q/k/v projection through ``project_qkv`` on installed modules.
* ``norm``    ``rmsnorm_linear_mi355x_fp8`` with a residual: a layer's input side.
* ``mlp``     ``mlp_forward_mi355x_fp8``: gate/up, SiLU*up, down.
* ``stack``   the four projections of several layers, each on its own input: the linears of one
              continuous-batching step, weights streamed from HBM.
* ``decode``  the projections and norms of two layers as a decode step runs them, captured in a
              HIP graph that each pass replays, as serving engines do.  Each norm and o_proj has
              its own input, so that one layer's rounding does not travel through the next.
* ``quant``   ``quantize_mi355x_fp8_activation`` alone.
"""

from __future__ import annotations

import os
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "mini-inference-engine_amd"))

from minillm_amd import merged_projections, mi355x_fp8 as fp8  # noqa: E402

DEVICE = "cuda"
BLOCK = [128, 128]
EPS = 1e-6
HIDDEN, INTER, Q_WIDTH, KV_WIDTH = 2560, 9728, 4096, 1024
# (N, K) of the four merged projections, and of the ones a model without merging calls.
PROJECTIONS = ((6144, 2560), (2560, 4096), (19456, 2560), (2560, 9728))
SEPARATE = ((4096, 2560), (1024, 2560), (9728, 2560))


def listed():
    return [
        # One token through o_proj, eager: the smallest call, all latency.
        {"name": "linear_o_1", "kind": "linear", "m": 1, "n": 2560, "k": 4096, "dtype": "bf16"},
        # A decode batch through down_proj, eager: the longest K.
        {"name": "linear_down_32", "kind": "linear", "m": 32, "n": 2560, "k": 9728, "dtype": "bf16"},
        # 16 tokens through the merged q/k/v projection as the attention module calls it.
        {"name": "merged_qkv_16", "kind": "qkv", "m": 16},
        # Two layers of a decode step at a small and at a larger batch, from a captured graph.
        {"name": "decode_layers_8", "kind": "decode", "m": 8},
        {"name": "decode_layers_32", "kind": "decode", "m": 32},
        # A mixed step: a 512-token prefill chunk and 24 decode tokens, eight layers of linears.
        {"name": "stack_536", "kind": "stack", "m": 536, "layers": 8},
        # The MLP block on a prefill chunk, middle-sized and full.
        {"name": "mlp_512", "kind": "mlp", "m": 512},
        {"name": "mlp_2048", "kind": "mlp", "m": 2048},
        # Residual add, RMSNorm and the merged q/k/v projection of a full prefill chunk.
        {"name": "norm_qkv_2048", "kind": "norm", "m": 2048, "n": 6144, "k": 2560},
        # The widest projection on the longest prompt of the benchmark sweep.
        {"name": "linear_gate_up_16384", "kind": "linear", "m": 16384, "n": 19456, "k": 2560, "dtype": "bf16"},
        # A generic fp16 linear whose rows, width and depth all end inside a 128-block.
        {"name": "linear_f16_ragged", "kind": "linear", "m": 333, "n": 2880, "k": 2880, "dtype": "f16"},
        # The activation quantizer alone on a prefill chunk of the down projection's input.
        {"name": "quant_2048", "kind": "quant", "m": 2048, "k": 9728, "dtype": "bf16"},
    ]


def _log(rng, low, high):
    return int(round(low * (high / low) ** rng.random()))


def draw(rng):
    kind = rng.choice(("linear", "linear", "linear", "qkv", "norm", "mlp", "mlp", "stack", "decode", "decode", "quant"))
    if kind == "linear":
        how = rng.random()
        dtype = "bf16" if rng.random() < 0.75 else "f16"
        if how < 0.75:
            n, k = rng.choice(PROJECTIONS + PROJECTIONS + SEPARATE)
            return {"kind": kind, "m": _log(rng, 1, 16384), "n": n, "k": k, "dtype": dtype}
        if how < 0.95:  # whole 16-element pieces, not whole 128-blocks
            return {"kind": kind, "m": _log(rng, 1, 4096), "n": 16 * _log(rng, 8, 600), "k": 16 * _log(rng, 8, 500), "dtype": dtype}
        return {"kind": kind, "m": _log(rng, 1, 1024), "n": _log(rng, 129, 1500), "k": _log(rng, 127, 1500), "dtype": dtype}
    if kind == "norm":
        return {"kind": kind, "m": _log(rng, 1, 8192), "n": rng.choice((6144, 19456)), "k": 2560}
    if kind == "stack":
        return {"kind": kind, "m": _log(rng, 64, 1500), "layers": rng.randint(2, 6)}
    if kind == "decode":
        return {"kind": kind, "m": _log(rng, 1, 64)}
    if kind == "quant":
        return {"kind": kind, "m": _log(rng, 1, 8192), "k": rng.choice((2560, 4096, 9728, 16 * _log(rng, 8, 600))), "dtype": rng.choice(("bf16", "f16"))}
    return {"kind": kind, "m": _log(rng, 1, 4096)}


# --------------------------------------------------------------------------------------
# Inputs
# --------------------------------------------------------------------------------------
def _generator(seed):
    return torch.Generator(device=DEVICE).manual_seed(seed)


def _activations(gen, m, k, dtype=torch.bfloat16):
    x = torch.randn((m, k), generator=gen, device=DEVICE)
    x[:, torch.randperm(k, generator=gen, device=DEVICE)[: max(1, k // 100)]] *= 20
    return x.to(dtype)


def _weights(gen, n, k):
    """e4m3fn codes [n, k] and fp32 block scales (amax / 448 per 128x128 block)."""

    gn, gk = -(-n // 128), -(-k // 128)
    padded = torch.zeros((gn * 128, gk * 128), device=DEVICE)
    padded[:n, :k] = (torch.randn((n, k), generator=gen, device=DEVICE) * 0.02).bfloat16()
    blocks = padded.view(gn, 128, gk, 128)
    scale = blocks.abs().amax(dim=(1, 3)) / 448.0
    codes = (blocks / scale[:, None, :, None]).view(gn * 128, gk * 128)[:n, :k]
    return codes.contiguous().to(torch.float8_e4m3fn), scale


def _norm_weight(gen, k):
    return (1.0 + 0.1 * torch.randn(k, generator=gen, device=DEVICE)).bfloat16()


class _Projection(torch.nn.Module):
    """A linear as the checkpoint holds it: e4m3fn weight and block scales."""

    def __init__(self, weight, scale):
        super().__init__()
        self.weight = torch.nn.Parameter(weight, requires_grad=False)
        self.weight_scale_inv = torch.nn.Parameter(scale, requires_grad=False)
        self.block_size = (128, 128)
        self.bias = None
        self.activation_scale = None


def _dtype(case):
    return torch.float16 if case.get("dtype") == "f16" else torch.bfloat16


def _inputs(case, seed):
    """The tensors of a case, from the seed alone (what prepare and exact both start from)."""

    gen = _generator(seed)
    kind, m = case["kind"], case["m"]
    if kind == "linear":
        return {"x": _activations(gen, m, case["k"], _dtype(case)), "w": _weights(gen, case["n"], case["k"])}
    if kind == "quant":
        return {"x": _activations(gen, m, case["k"], _dtype(case))}
    if kind == "qkv":
        return {"x": _activations(gen, m, HIDDEN),
                "w": [_weights(gen, n, HIDDEN) for n in (Q_WIDTH, KV_WIDTH, KV_WIDTH)]}
    if kind == "norm":
        return {"x": _activations(gen, m, case["k"]), "residual": _activations(gen, m, case["k"]),
                "norm": _norm_weight(gen, case["k"]), "w": _weights(gen, case["n"], case["k"])}
    if kind == "mlp":
        return {"x": _activations(gen, m, HIDDEN), "gate_up": _weights(gen, 2 * INTER, HIDDEN),
                "down": _weights(gen, HIDDEN, INTER)}
    if kind == "stack":
        x = {k: _activations(gen, m, k) for k in (2560, 4096, 9728)}
        return {"x": x, "w": [[_weights(gen, n, k) for n, k in PROJECTIONS] for _ in range(case["layers"])]}
    layers = [{"norms": [_norm_weight(gen, HIDDEN) for _ in range(2)], "w": [_weights(gen, n, k) for n, k in PROJECTIONS],
               "x": _activations(gen, m, HIDDEN), "residual": _activations(gen, m, HIDDEN),
               "attn": _activations(gen, m, Q_WIDTH), "o": _activations(gen, m, HIDDEN)} for _ in range(2)]
    return {"layers": layers}


def _decode_step(state):
    """Per layer: norm + q/k/v, o_proj, norm + gate/up + SiLU*up, down."""

    outs = []
    for layer in state["layers"]:
        qkv_w, o_w, gate_up_w, down_w = layer["w"]
        qkv, residual = fp8.rmsnorm_linear_mi355x_fp8(layer["x"], layer["norms"][0], EPS, *qkv_w, residual=layer["residual"])
        o = fp8.mi355x_fp8_linear(layer["attn"], *o_w, BLOCK)
        h, residual = fp8.rmsnorm_gate_up_silu_mi355x_fp8(layer["o"], layer["norms"][1], EPS, *gate_up_w, residual=residual)
        outs += [qkv, o, h, fp8.mi355x_fp8_linear(h, *down_w, BLOCK), residual]
    return outs


def prepare(case, seed):
    state = _inputs(case, seed)
    state["kind"] = case["kind"]
    if case["kind"] == "qkv":
        attention = torch.nn.Module()
        for name, (w, s) in zip(("q_proj", "k_proj", "v_proj"), state.pop("w")):
            setattr(attention, name, _Projection(w, s))
        merged_projections.install_merged_projections(attention)
        state["attention"] = attention
    elif case["kind"] == "decode":
        stream = torch.cuda.Stream()
        stream.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(stream):
            _decode_step(state)
        torch.cuda.current_stream().wait_stream(stream)
        state["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(state["graph"], stream=stream):
            state["outs"] = _decode_step(state)
    return state


def run(state):
    kind = state["kind"]
    if kind == "linear":
        return fp8.mi355x_fp8_linear(state["x"], *state["w"], BLOCK)
    if kind == "quant":
        codes, scales = fp8.quantize_mi355x_fp8_activation(state["x"])
        return codes.view(torch.uint8), scales
    if kind == "qkv":
        return merged_projections.project_qkv(state["attention"], state["x"])
    if kind == "norm":
        return fp8.rmsnorm_linear_mi355x_fp8(state["x"], state["norm"], EPS, *state["w"], residual=state["residual"])
    if kind == "mlp":
        return fp8.mlp_forward_mi355x_fp8(state["x"], *state["gate_up"], *state["down"])
    if kind == "stack":
        return [fp8.mi355x_fp8_linear(state["x"][w.shape[1]], w, s, BLOCK) for layer in state["w"] for w, s in layer]
    state["graph"].replay()
    return state["outs"]


# --------------------------------------------------------------------------------------
# What a pass cannot do without
# --------------------------------------------------------------------------------------
def _linear_work(m, n, k):
    """Codes and scales of the weight, 16-bit input and output, each once."""

    return {"bytes": n * k + 4 * -(-n // 128) * -(-k // 128) + 2 * m * k + 2 * m * n, "flops": 2 * m * n * k}


def work(case):
    kind, m = case["kind"], case["m"]
    if kind == "linear":
        return _linear_work(m, case["n"], case["k"])
    if kind == "quant":
        return {"bytes": 3 * m * case["k"] + 4 * m * -(-case["k"] // 128), "flops": 3 * m * case["k"]}
    if kind == "qkv":
        return _linear_work(m, Q_WIDTH + 2 * KV_WIDTH, HIDDEN)
    if kind == "norm":
        w = _linear_work(m, case["n"], case["k"])
        return {"bytes": w["bytes"] + 4 * m * case["k"] + 2 * case["k"], "flops": w["flops"]}
    if kind == "mlp":  # x in, out out; the product between the two projections stays on the way
        up, down = _linear_work(m, 2 * INTER, HIDDEN), _linear_work(m, HIDDEN, INTER)
        between = 2 * m * 2 * INTER + 2 * m * INTER
        return {"bytes": up["bytes"] + down["bytes"] - between, "flops": up["flops"] + down["flops"]}
    each = [_linear_work(m, n, k) for n, k in PROJECTIONS]
    total = {key: sum(w[key] for w in each) for key in ("bytes", "flops")}
    if kind == "stack":  # the layers' three inputs are the same tensors
        x = 2 * m * sum(k for _, k in PROJECTIONS)
        return {"bytes": case["layers"] * (total["bytes"] - x) + 2 * m * (2560 + 4096 + 9728),
                "flops": case["layers"] * total["flops"]}
    # decode: per layer the weights, four inputs, four outputs (gate/up's after SiLU*up) and the residual.
    layer = sum(n * k + 4 * (n // 128) * (k // 128) for n, k in PROJECTIONS) + 2 * 2 * HIDDEN
    layer += 2 * m * (3 * HIDDEN + Q_WIDTH + 6144 + HIDDEN + INTER + HIDDEN + HIDDEN)
    return {"bytes": 2 * layer, "flops": 2 * total["flops"]}


def tolerance(case):
    """About four times the distance from exact(): the output's rounding (bf16 1.7e-3, fp16
    2.1e-4, both 2-norm) and, behind a SiLU*up or a norm, codes that a rounding of the bf16
    product moves to their neighbour (2.9e-3)."""

    if case["kind"] == "quant":
        return "exact"
    if case["kind"] in ("mlp", "decode"):
        return {"rel": 1.2e-2, "max": 0.06}
    if case.get("dtype") == "f16":
        return {"rel": 9e-4, "max": 4e-3}
    return {"rel": 7e-3, "max": 0.03}


# --------------------------------------------------------------------------------------
# The same in 64 bits, in plain torch
# --------------------------------------------------------------------------------------
def _quantized(x):
    """Codes and scales per row and 128 columns: s = amax / 448, code = e4m3(x / max(s, 1e-12)).
    The codes are decided by fp32 divisions, so both are divisions by a tensor (torch multiplies
    by the reciprocal of a scalar divisor)."""

    m, k = x.shape
    groups = -(-k // 128)
    padded = torch.zeros((m, groups * 128), device=x.device)
    padded[:, :k] = x.float()
    padded = padded.view(m, groups, 128)
    amax = padded.abs().amax(dim=2)
    scale = amax / torch.full_like(amax, 448.0)
    codes = (padded / scale.clamp_min(1e-12)[:, :, None]).to(torch.float8_e4m3fn)
    return codes.view(m, groups * 128)[:, :k], scale


def _wide(scale, block, size):
    return scale.double().repeat_interleave(block, dim=1)[:, :size]


def _linear64(x, w, s):
    """The linear in fp64 on the quantized operands (rows in pieces: the largest case is 16384 rows)."""

    n, k = w.shape
    weight = w.double() * _wide(s, 128, k).repeat_interleave(128, dim=0)[:n]
    parts = []
    for rows in x.split(4096):
        codes, scale = _quantized(rows)
        parts.append((codes.double() * _wide(scale, 128, k)) @ weight.t())
    return torch.cat(parts)


def _norm64(x, weight):
    v = x.double()
    normed = (v * torch.rsqrt(v.square().mean(dim=1, keepdim=True) + EPS)).bfloat16()
    return (weight.double() * normed.double()).bfloat16()


def _silu_mul64(gate_up):
    gate, up = gate_up.bfloat16().double().chunk(2, dim=1)
    return torch.nn.functional.silu(gate).bfloat16().double() * up


def exact(case, seed):
    t = _inputs(case, seed)
    kind = case["kind"]
    if kind == "linear":
        return _linear64(t["x"], *t["w"])
    if kind == "quant":
        codes, scales = _quantized(t["x"])
        return codes.contiguous().view(torch.uint8), scales
    if kind == "qkv":
        return tuple(_linear64(t["x"], w, s) for w, s in t["w"])
    if kind == "norm":
        summed = (t["x"].double() + t["residual"].double())
        return _linear64(_norm64(summed.bfloat16(), t["norm"]), *t["w"]), summed
    if kind == "mlp":
        return _linear64(_silu_mul64(_linear64(t["x"], *t["gate_up"])).bfloat16(), *t["down"])
    if kind == "stack":
        return [_linear64(t["x"][w.shape[1]], w, s) for layer in t["w"] for w, s in layer]
    outs = []
    for layer in t["layers"]:
        qkv_w, o_w, gate_up_w, down_w = layer["w"]
        after_x = layer["x"].double() + layer["residual"].double()
        qkv = _linear64(_norm64(after_x.bfloat16(), layer["norms"][0]), *qkv_w)
        after_o = after_x.bfloat16().double() + layer["o"].double()
        h = _silu_mul64(_linear64(_norm64(after_o.bfloat16(), layer["norms"][1]), *gate_up_w))
        outs += [qkv, _linear64(layer["attn"], *o_w), h, _linear64(h.bfloat16(), *down_w), after_o]
    return outs
