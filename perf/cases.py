"""The calls that this framework is used for, at sizes from the smallest to the largest, for timing them.

A case is a dict of plain values.  ``listed()`` names the standing ones, ``draw(rng)`` gives one more of the
same ranges, ``prepare(case, seed)`` builds what a program holds before the call (layers with their weights
loaded, activations on the GPU), ``run(state)`` makes one pass through the public entry points and returns
what it computes, ``work(case)`` counts the bytes and operations that pass cannot do without and
``tolerance(case)`` says how far another correct implementation may be off.

Kinds of case:

``linear``  one quantized linear layer called as a module (``ColumnParallelLinear``), eager; per-channel weights
            with per-token activations, or per-tensor scales on both sides
``mlp``     one ``DenseMLP`` called as a module, eager; gated or plain, with or without the gated residual behind it
``layer``   one decoder layer of the action expert (``ExpertLayer``), eager, attention left out
``prefix``  the norms and linears of one prefix (prefill) layer, eager, attention left out
``dit``     the linears of one diffusion-transformer block, eager, attention and norms left out
``loop``    the whole flow-matching denoise loop as one recorded graph (``ExpertDenoiseLoop``), attention left out
``load``    a bf16 weight matrix quantized into a layer and laid out for serving, as after reading a checkpoint

Attention is not part of this framework: where a layer has one, its callback hands on the query part of the
fused projection, which has the shape of an attention output.
"""

from __future__ import annotations

import math

import torch

import phyai_amd.linear as L
from phyai_amd.cache_plan import plan_weight_streaming
from phyai_amd.mlp import DenseMLP
from phyai_amd.norm import GemmaRMSNorm
from phyai_amd.runtime.expert_loop import ExpertDenoiseLoop, ExpertLayer, ExpertLayerModulation

ACTION_DIM = 32
MAX_FLOPS = 2.0 * 13056 * 2048 * 3 * 16384      # the largest listed pass; no drawn one asks for more


def listed() -> list[dict]:
    return [
        # The smallest call there is: the modulation linear of a diffusion block, one conditioning row per batch.
        dict(name="adaln_m1", kind="linear", scheme="per_channel", m=1, n=12288, k=2048, bias=True, operand=True),
        # One chunk of 50 action tokens through a single layer whose weights stay as the checkpoint holds them.
        dict(name="linear_m50_bias", kind="linear", scheme="per_channel", m=50, n=4096, k=1024, bias=True, operand=False),
        # A checkpoint with static per-tensor scales, at a batch of 8 action chunks.
        dict(name="per_tensor_m400", kind="linear", scheme="per_tensor", m=400, n=2560, k=1024, bias=False, operand=False),
        # Widths that are multiples of 16 and of nothing larger, and an odd number of tokens.
        dict(name="mlp_ragged_m777", kind="mlp", m=777, h=1168, i=4304, act="gelu_tanh", gated=False, bias=True,
             operand=True, residual=False),
        # The action expert's MLP for one chunk, called eagerly.
        dict(name="mlp_expert_m50", kind="mlp", m=50, h=1024, i=4096, act="gelu_tanh", gated=True, bias=False,
             operand=True, residual=True),
        # A whole decoder layer of the expert for a batch of 8 chunks: the mid-sized calls of a serving engine.
        dict(name="expert_layer_m400", kind="layer", m=400, h=1024, heads=8, head_dim=256, i=4096, operand=True),
        # What an engine launches per action chunk: 10 Euler steps x 18 layers, one graph.
        dict(name="denoise_loop_m50", kind="loop", m=50, h=1024, heads=8, head_dim=256, i=4096, layers=18, steps=10),
        # Prefill of one sample (3 images x 256 patches + 48 text tokens), one backbone layer.
        dict(name="prefix_layer_m816", kind="prefix", m=816, h=2048, heads=8, head_dim=256, i=16384, operand=True),
        # Prefill of four samples, weights as loaded.
        dict(name="prefix_layer_m3264", kind="prefix", m=3264, h=2048, heads=8, head_dim=256, i=16384, operand=False),
        # One video diffusion block: 4800 latent tokens, every linear with bias, plain GELU.
        dict(name="dit_block_m4800", kind="dit", m=4800, h=2048, i=8192, operand=True),
        # The largest: the backbone's MLP for a batch of 16 samples.
        dict(name="mlp_prefix_m13056", kind="mlp", m=13056, h=2048, i=16384, act="gelu_tanh", gated=True, bias=False,
             operand=True, residual=False),
        # Loading: one gate | up matrix of the backbone from bf16.
        dict(name="load_gate_up", kind="load", n=32768, k=2048, gated=True, operand=True),
    ]


def _log_int(rng, lo: int, hi: int) -> int:
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def _width(rng, lo: int, hi: int, step: int = 16) -> int:
    """A multiple of ``step``, spread over the logarithm; two of three are multiples of 128 as models have them."""
    step = max(step, 128) if rng.random() < 0.67 else step
    return max(step, round(_log_int(rng, lo, hi) / step) * step)


def draw(rng) -> dict:
    kind = rng.choice(["linear", "linear", "linear", "mlp", "mlp", "mlp", "layer", "prefix", "dit", "loop", "load"])
    operand = rng.random() < 0.6
    if kind == "linear":
        case = dict(kind=kind, scheme=rng.choice(["per_channel", "per_channel", "per_tensor"]), m=_log_int(rng, 1, 13056),
                    n=_width(rng, 256, 12288), k=_width(rng, 512, 16384), bias=rng.random() < 0.5, operand=operand)
    elif kind == "mlp":
        gated = rng.random() < 0.67
        case = dict(kind=kind, m=_log_int(rng, 1, 13056), h=_width(rng, 512, 2048), i=_width(rng, 1024, 16384), gated=gated,
                    act=rng.choice(["silu", "gelu", "gelu_tanh"] if gated else ["gelu", "gelu_tanh"]),
                    bias=rng.random() < 0.5, operand=operand, residual=rng.random() < 0.5)
    elif kind == "layer":
        case = dict(kind=kind, m=_log_int(rng, 8, 1600), h=_width(rng, 512, 2048), heads=rng.choice([4, 8]),
                    head_dim=rng.choice([128, 256]), i=_width(rng, 2048, 8192), operand=operand)
    elif kind == "prefix":
        case = dict(kind=kind, m=_log_int(rng, 128, 6528), h=_width(rng, 1024, 2048), heads=8, head_dim=rng.choice([128, 256]),
                    i=_width(rng, 4096, 16384), operand=operand)
    elif kind == "dit":
        case = dict(kind=kind, m=_log_int(rng, 512, 9600), h=_width(rng, 1024, 2048, 128), i=_width(rng, 4096, 8192), operand=operand)
    elif kind == "loop":
        case = dict(kind=kind, m=_log_int(rng, 8, 100), h=_width(rng, 512, 1024, 128), heads=8, head_dim=rng.choice([128, 256]),
                    i=_width(rng, 2048, 4096, 128), layers=rng.randint(2, 18), steps=rng.randint(2, 10))
    else:
        case = dict(kind=kind, n=_width(rng, 1024, 32768, 32), k=_width(rng, 512, 16384), gated=rng.random() < 0.5, operand=operand)
        case["n"] = max(1024, min(case["n"], (1 << 26) // case["k"] // 32 * 32))
    if "m" in case and work(case)["flops"] > MAX_FLOPS:
        case["m"] = max(1, int(case["m"] * MAX_FLOPS / work(case)["flops"]))
    return case


# ---- building what a program holds ---------------------------------------------------------------------------

class _Maker:
    """Seeded tensors on the GPU: weights ~N(0, 0.02), activations ~N(0, 1) with one channel in a hundred x 20."""

    def __init__(self, seed: int) -> None:
        self.dev = torch.device("cuda", torch.cuda.current_device())
        self.gen = torch.Generator(device=self.dev).manual_seed(int(seed))

    def normal(self, *shape, scale: float = 1.0) -> torch.Tensor:
        t = torch.empty(*shape, dtype=torch.bfloat16, device=self.dev)
        return t.normal_(0.0, scale, generator=self.gen)

    def activations(self, m: int, k: int) -> torch.Tensor:
        x = self.normal(m, k)
        channels = torch.rand(k, generator=self.gen, device=self.dev) < 0.01
        return torch.where(channels, x * 20.0, x)


def _init() -> None:
    try:
        L.get_linear_dispatcher()
    except RuntimeError:
        L.init()


def _spec(scheme: str, operand: bool) -> L.Fp8Spec:
    g = L.Granularity.PER_TENSOR if scheme == "per_tensor" else L.Granularity.PER_CHANNEL
    return L.Fp8Spec(granularity=g, operand_order=operand)


def _load(mk: _Maker, lin) -> None:
    """Give a freshly built layer its weights, as a loader does, and let it lay them out."""
    n, k = lin.weight.shape
    w = mk.normal(n, k, scale=0.02)
    if lin.spec.granularity is L.Granularity.PER_TENSOR:
        s = w.abs().amax().float() / 448.0
        lin.weight.data.copy_((w.float() / s).clamp(-448.0, 448.0).to(torch.float8_e4m3fn))
        lin.weight_scale.data.fill_(s)
        lin.input_scale.data.fill_(16.0 / 448.0)      # a calibrated range that a few outliers exceed
    else:
        lin.spec.quantize_weight_(lin, w)
    if lin.bias is not None:
        lin.bias.data.copy_(mk.normal(n, scale=0.01))
    lin.post_load()


def _mlp(mk: _Maker, case: dict, *, gated: bool, act: str, bias: bool) -> DenseMLP:
    mlp = DenseMLP(case["h"], case["i"], activation=act, gated=gated, bias=bias, params_dtype=torch.bfloat16,
                   spec_in=_spec("per_channel", case["operand"]), spec_out=_spec("per_channel", case["operand"]))
    for lin in ((mlp.gate_up_proj, mlp.down_proj) if gated else (mlp.fc1, mlp.fc2)):
        _load(mk, lin)
    return mlp


def _expert_layer(mk: _Maker, case: dict, index: int) -> ExpertLayer:
    layer = ExpertLayer(case["h"], case["head_dim"], case["heads"], 1, case["i"], case["h"],
                        spec=_spec("per_channel", case.get("operand", True)), prefix=f"model.layers.{index}")
    for lin in (layer.qkv_proj, layer.o_proj, layer.mlp.gate_up_proj, layer.mlp.down_proj):
        _load(mk, lin)
    for norm in (layer.input_layernorm, layer.post_attention_layernorm):
        norm.dense.weight.data.copy_(mk.normal(3 * case["h"], case["h"], scale=0.003))
        norm.dense.bias.data.copy_(mk.normal(3 * case["h"], scale=0.03))
    return layer


def _query_part(width: int):
    """Stands where attention does: the query columns of the fused projection, as they lie."""
    return lambda fused, index: fused[:, :width]


def prepare(case: dict, seed: int) -> dict:
    _init()
    mk = _Maker(seed)
    kind = case["kind"]
    st: dict = {"kind": kind}
    with torch.no_grad():
        if kind == "linear":
            st["lin"] = L.ColumnParallelLinear(case["k"], case["n"], bias=case["bias"], params_dtype=torch.bfloat16,
                                               spec=_spec(case["scheme"], case["operand"]))
            _load(mk, st["lin"])
            st["x"] = mk.activations(case["m"], case["k"])
        elif kind == "mlp":
            st["mlp"] = _mlp(mk, case, gated=case["gated"], act=case["act"], bias=case["bias"])
            st["x"] = mk.activations(case["m"], case["h"])
            st["residual"] = mk.normal(case["m"], case["h"]) if case["residual"] else None
            st["gate"] = mk.normal(1, case["h"], scale=0.3) if case["residual"] else None
        elif kind == "layer":
            st["layer"] = _expert_layer(mk, case, 0)
            st["attend"] = _query_part(case["heads"] * case["head_dim"])
            st["mod"] = ExpertLayerModulation(mk.normal(1, 3 * case["h"], scale=0.1), mk.normal(1, 3 * case["h"], scale=0.1))
            st["x"] = mk.activations(case["m"], case["h"])
        elif kind == "prefix":
            h, width = case["h"], case["heads"] * case["head_dim"]
            spec = _spec("per_channel", case["operand"])
            st["norm1"], st["norm2"] = GemmaRMSNorm(h), GemmaRMSNorm(h)
            for norm in (st["norm1"], st["norm2"]):
                norm.weight.data.copy_(mk.normal(h, scale=0.1))
            st["qkv"] = L.QKVParallelLinear(h, case["head_dim"], case["heads"], 1, bias=False, params_dtype=torch.bfloat16, spec=spec)
            st["o"] = L.RowParallelLinear(width, h, bias=False, params_dtype=torch.bfloat16, spec=spec)
            for lin in (st["qkv"], st["o"]):
                _load(mk, lin)
            st["mlp"] = _mlp(mk, case, gated=True, act="gelu_tanh", bias=False)
            st["attend"] = _query_part(width)
            st["x"] = mk.activations(case["m"], h)
        elif kind == "dit":
            h = case["h"]
            spec = _spec("per_channel", case["operand"])
            st["qkv"] = L.QKVParallelLinear(h, 128, h // 128, bias=True, params_dtype=torch.bfloat16, spec=spec)
            st["out"] = L.RowParallelLinear(h, h, bias=True, params_dtype=torch.bfloat16, spec=spec)
            for lin in (st["qkv"], st["out"]):
                _load(mk, lin)
            st["mlp"] = _mlp(mk, case, gated=False, act="gelu", bias=True)
            st["attend"] = _query_part(h)
            st["x"], st["y"] = mk.activations(case["m"], h), mk.activations(case["m"], h)
        elif kind == "loop":
            h, steps = case["h"], case["steps"]
            layers = [_expert_layer(mk, case, i) for i in range(case["layers"])]
            plan_weight_streaming([lin for lay in layers for lin in (lay.qkv_proj, lay.o_proj, lay.mlp.gate_up_proj, lay.mlp.down_proj)])
            loop = ExpertDenoiseLoop(layers, _query_part(case["heads"] * case["head_dim"]), chunk_size=case["m"],
                                     action_dim=ACTION_DIM, hidden_size=h, cond_dim=h)
            loop.embed_action.weight.data.copy_(mk.normal(h, ACTION_DIM, scale=0.3))
            loop.project_action.weight.data.copy_(mk.normal(ACTION_DIM, h, scale=0.03))
            loop.embed_action.bias.data.zero_()
            loop.project_action.bias.data.zero_()
            loop.final_norm.dense.weight.data.copy_(mk.normal(3 * h, h, scale=0.01))
            loop.bind_euler_schedule(mk.normal(steps, h), -1.0 / steps, steps)
            loop.setup()
            st["loop"], st["noise"] = loop, mk.normal(case["m"], ACTION_DIM)
        elif kind == "load":
            st["lin"] = L.ColumnParallelLinear(case["k"], case["n"], bias=False, params_dtype=torch.bfloat16,
                                               spec=_spec("per_channel", case["operand"]))
            st["lin"].gated_pairs = case["gated"]
            st["w"] = mk.normal(case["n"], case["k"], scale=0.02)
        else:
            raise ValueError(f"unknown kind {kind!r}")
    return st


# ---- one pass --------------------------------------------------------------------------------------------------

@torch.no_grad()
def run(st: dict):
    kind = st["kind"]
    if kind == "linear":
        return st["lin"](st["x"])[0]
    if kind == "mlp":
        return st["mlp"](st["x"], residual=st["residual"], gate=st["gate"])
    if kind == "layer":
        return st["layer"](st["x"], st["attend"], 0, st["mod"])
    if kind == "prefix":
        x = st["x"]
        fused, _ = st["qkv"](st["norm1"].forward_fp8(x))
        h = x + st["o"](st["attend"](fused, 0))[0]
        return {"qkv": fused, "out": h + st["mlp"](st["norm2"](h))}
    if kind == "dit":
        fused, _ = st["qkv"](st["x"])
        return {"qkv": fused, "attn_out": st["out"](st["attend"](fused, 0))[0], "mlp_out": st["mlp"](st["y"])}
    if kind == "loop":
        return st["loop"].run(st["noise"])
    lin = st["lin"]
    lin.spec.quantize_weight_(lin, st["w"])
    lin.post_load()
    return {"codes": lin.weight.data.view(torch.uint8), "scale": lin.weight_scale.data}


# ---- what a pass cannot do without -------------------------------------------------------------------------------

def _mlp_counts(m: int, h: int, i: int, gated: bool) -> tuple[float, float]:
    """(weight bytes, flops) of both projections."""
    rows = (2 if gated else 1) * i
    return float(rows * h + 4 * rows + h * i + 4 * h), 2.0 * m * h * (rows + i)


def _qkv_o_counts(m: int, h: int, qkv: int, width: int) -> tuple[float, float]:
    return float(qkv * h + 4 * qkv + h * width + 4 * h), 2.0 * m * h * (qkv + width)


def work(case: dict) -> dict:
    kind, m = case["kind"], case.get("m", 0)
    if kind == "load":
        n, k = case["n"], case["k"]
        return {"bytes": 3.0 * n * k + 4.0 * n, "flops": 0.0}
    if kind == "linear":
        n, k = case["n"], case["k"]
        return {"bytes": 2.0 * m * k + n * k + 4.0 * n + (2.0 * n if case["bias"] else 0.0) + 2.0 * m * n, "flops": 2.0 * m * n * k}
    h, i = case["h"], case["i"]
    if kind == "mlp":
        w, flops = _mlp_counts(m, h, i, case["gated"])
        bias = 2.0 * ((2 if case["gated"] else 1) * i + h) if case["bias"] else 0.0
        return {"bytes": w + bias + 4.0 * m * h + (2.0 * m * h + 2.0 * h if case["residual"] else 0.0), "flops": flops}
    if kind == "dit":
        w1, f1 = _mlp_counts(m, h, i, False)
        w2, f2 = _qkv_o_counts(m, h, 3 * h, h)
        return {"bytes": w1 + w2 + 2.0 * (5 * h + i) + 2.0 * m * (2 * h + 3 * h + 2 * h), "flops": f1 + f2}
    width = case["heads"] * case["head_dim"]
    w1, f1 = _mlp_counts(m, h, i, True)
    w2, f2 = _qkv_o_counts(m, h, width + 2 * case["head_dim"], width)
    if kind == "layer":
        return {"bytes": w1 + w2 + 12.0 * h + 4.0 * m * h, "flops": f1 + f2}
    if kind == "prefix":
        return {"bytes": w1 + w2 + 4.0 * h + 4.0 * m * h + 2.0 * m * (width + 2 * case["head_dim"]), "flops": f1 + f2}
    # loop: every step needs every layer's weights again (a step depends on the whole one before it, and
    # the weights are larger than the registers, LDS and L2 of the chip together)
    times = case["layers"] * case["steps"]
    return {"bytes": times * (w1 + w2 + 12.0 * h) + 4.0 * m * ACTION_DIM, "flops": times * (f1 + f2)}


def tolerance(case: dict):
    """bf16 results of fp8 products summed in fp32.  One linear rounds once (2^-9 relative); behind a second
    quantizer a sum that lands on the other side of a bf16 step can move a code by one e4m3 step (2^-4) of one
    value in many; a loop chains this through all its layers and steps.  Quantized weights are exact."""
    if case["kind"] == "load":
        return "exact"
    if case["kind"] == "linear":
        return {"rel": 5e-3, "max": 0.05}
    if case["kind"] == "loop":
        return {"rel": 2e-2}
    return {"rel": 1e-2}
