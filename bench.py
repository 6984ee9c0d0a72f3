#!/usr/bin/env python3
"""Benchmark of the W8A8 fp8 linear hot path on one MI355X.

Workload (the configuration the metric is quoted on): the Pi0.5 action-expert
linear set.  18 layers x {qkv 1024->2560, o 2048->1024, gate_up 1024->8192 with
fused GeGLU-tanh, down 4096->1024}, M = 50 action tokens, bf16 activations
~N(0,1), fp8 e4m3fn weights ~N(0,0.02) with per-output-channel scales, every
layer with its own weight tensors (311 MB of fp8 weights per denoise step), and
10 flow-matching steps recorded in ONE hipGraph.  A bench "step" is one replay of
that graph (what the engine launches per action chunk); `value` is the p50 time
of one denoise step (replay time / 10) in microseconds.

How the linears are called is what a model built on this library does (phyai_amd.linear layers with
Fp8Spec(operand_order=True), phyai_amd.mlp.DenseMLP): weights re-laid in MFMA operand order once after
loading, qkv and o as one phyai_fp8_linear each, gate_up + GeGLU and down as one phyai_fp8_mlp call (down
consumes gate_up's output, as in the model; its own random input tensor is used only by the variants that
run the four linears separately).  --row-major / --separate-linears switch either back for A/B runs.

Printed JSON (one line):
  value / ms_per_step  whole-path numbers (quantization + GEMM + epilogue, graph replay)
  roofline             the kernels that read the weights: algorithmic bytes of one layer's four
                       linears / the measured duration of the launches that read their weights (the
                       whole linear where it is one kernel that quantizes its own rows, else the GEMM
                       behind the quantizer), HIP events around replays of a graph that holds only
                       those launches and walks all 18 layers' distinct weights
  roofline_prefill     the MFMA-bound regime (M = 816), per shape and for the layer
  launch_floor         what the kernel nodes of a layer cost before any byte moves
  cpu_baseline         torch CPU dequantize + matmul form of the same layer set on
                       this box's host cores (a reported baseline, not the target)
  extra                neighbouring measurements (prefill layer, decoder layer with norms, ...)

Inputs are resident in HBM before the timed region starts.
"""

from __future__ import annotations

import argparse
import json
import os
import statistics
import sys
import time

import torch

ROOT = os.path.dirname(os.path.abspath(__file__))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)

HBM_PEAK_GBS = 8000.0       # MI355X HBM3E
FP8_PEAK_TFLOPS = 5000.0    # MI355X dense fp8 MFMA

# (name, N, K, epilogue) per layer
EXPERT_SET = [("qkv", 2560, 1024, None), ("o", 1024, 2048, None),
              ("gate_up", 8192, 1024, "geglu_tanh"), ("down", 1024, 4096, None)]
PREFILL_SET = [("qkv", 2560, 2048, None), ("o", 2048, 2048, None),
               ("gate_up", 32768, 2048, "geglu_tanh"), ("down", 2048, 16384, None)]
# DiT block (benchmark configuration 5): M = 4800 video-latent tokens, every linear with bias; the
# adaLN modulation linear runs at M = batch = 1.  (name, N, K, epilogue, M)
DIT_SET = [("qkv", 6144, 2048, None, 4800), ("out", 2048, 2048, None, 4800),
           ("fc1", 8192, 2048, "gelu", 4800), ("fc2", 2048, 8192, None, 4800),
           ("adaLN", 12288, 2048, None, 1)]


def profiled_layer_traffic():
    """HBM bytes moved by one layer's four GEMM launches at M = 50, as measured with rocprofv3 --pmc
    FETCH_SIZE / WRITE_SIZE on `bench.py --probe` and calibrated against a 64 MiB copy: read from the
    committed counter summary (its `traffic_bytes_per_layer` line), so that the figure in the JSON
    line is the one the profile holds.  None when the summary is missing."""
    import re

    path = os.path.join(ROOT, "profiles", "expert_m50_hbm_traffic.md")
    try:
        m = re.search(r"^\s*traffic_bytes_per_layer\s*=\s*(\d+)", open(path, encoding="utf-8").read(), flags=re.M)
    except OSError:
        return None
    return int(m.group(1)) if m else None


def algorithmic_bytes(M: int, N: int, K: int, epilogue, bias: bool = False) -> int:
    """bf16 X in + fp8 W + fp32 weight scales (+ bf16 bias) + bf16 out (half width if gated)."""
    n_out = N // 2 if epilogue in ("geglu_tanh", "geglu_erf", "swiglu") else N
    return 2 * M * K + N * K + 4 * N + (2 * N if bias else 0) + 2 * M * n_out


# How the benchmark calls the library (switched by --row-major / --separate-linears for A/B runs)
OPTS = {"operand": True, "mlp": True}


def make_layers(dev, shapes, M, n_layers, seed0=0):
    """Seeded synthetic tensors, generated on the CPU and copied to the device so that
    the CPU baseline sees the same bits.  Weights are quantized on the device by the
    library's own weight quantizer (bit-exact with the oracle's) and, as Fp8Spec(operand_order=True)
    does in process_after_loading, re-laid in MFMA operand order (`wo`; `w` stays row-major for the
    torch and CPU paths)."""
    from phyai_amd import ops

    layers = []
    seed = seed0
    for li in range(n_layers):
        layer = {}
        for name, N, K, epi in shapes:
            g = torch.Generator().manual_seed(seed)
            seed += 1
            w = (torch.randn(N, K, generator=g) * 0.02).to(torch.bfloat16)
            x = torch.randn(M, K, generator=g).to(torch.bfloat16)
            wq, ws = ops.fp8_weight_quant(w.to(dev))
            n_out = N // 2 if epi else N
            layer[name] = dict(w=wq, ws=ws, x=x.to(dev), epi=epi, N=N, K=K,
                               out=torch.empty(M, n_out, dtype=torch.bfloat16, device=dev),
                               w_bf16_cpu=w if li == 0 else None, x_cpu=x if li == 0 else None)
            if K % 128 == 0:
                layer[name]["wo"] = ops.fp8_weight_to_operand_order(wq, gated=bool(epi))
                layer[name]["lay"] = ("operand_gated" if epi in ("geglu_tanh", "geglu_erf", "swiglu") else "operand")
        layers.append(layer)
    return layers


def weight_of(t):
    """(weight tensor, weight_layout) the benchmark passes for this linear."""
    if OPTS["operand"] and "wo" in t:
        return t["wo"], t["lay"]
    return t["w"], None


def linear(t, x=None, out=None):
    from phyai_amd import ops

    w, lay = weight_of(t)
    return ops.fp8_linear(t["x"] if x is None else x, w, t["ws"], None, epilogue=t["epi"],
                          out=t["out"] if out is None else out, stream_weights=t.get("stream", False), weight_layout=lay)


def is_mlp_pair(a, b) -> bool:
    """gate_up (an activation epilogue) followed by the projection that consumes its output."""
    return bool(a["epi"]) and b["epi"] is None and b["K"] == a["out"].shape[-1] and a["out"].shape[0] == b["out"].shape[0]


def mlp(a, b):
    from phyai_amd import ops

    (w1, l1), (w2, l2) = weight_of(a), weight_of(b)
    return ops.fp8_mlp(a["x"], w1, a["ws"], None, w2, b["ws"], None, epilogue=a["epi"], out=b["out"],
                       stream_weights1=a.get("stream", False), stream_weights2=b.get("stream", False),
                       weight1_layout=l1, weight2_layout=l2)


def run_layer(layer, shapes):
    """One layer's linears as a model calls them: an MLP's two projections as one phyai_fp8_mlp call."""
    names = [name for name, _, _, _ in shapes]
    i = 0
    while i < len(names):
        t = layer[names[i]]
        if OPTS["mlp"] and i + 1 < len(names) and is_mlp_pair(t, layer[names[i + 1]]):
            mlp(t, layer[names[i + 1]])
            i += 2
        else:
            linear(t)
            i += 1


def run_layers(layers, shapes):
    for layer in layers:
        run_layer(layer, shapes)


def torch_reference_times(dev, layers, shapes, denoise_steps, steps, warmup):
    """The reference's own GPU path for the same linears, as far as this image can run it: the
    quantizer's torch expressions (layers/quant/fp8.py:152-154) and torch._scaled_mm
    (layers/linear/backends/torch.py:166-175; hipBLASLt underneath on ROCm), the gated activation as
    torch ops because flashinfer is not installed.  Same tensors, same graph shape.  Returns us per
    denoise step, or a reason string when torch._scaled_mm does not run here."""
    import torch.nn.functional as F

    from phyai_amd.runtime import HipGraph

    def linear(t):
        x = t["x"]
        a = x.abs().amax(dim=-1, keepdim=True).clamp_min(1e-12)
        s = (a / 448.0).to(torch.float32)
        xq = (x / s).to(torch.float8_e4m3fn)
        y = torch._scaled_mm(xq, t["w"].t(), scale_a=s, scale_b=t["ws"].reshape(1, -1), out_dtype=torch.bfloat16)
        if t["epi"]:
            half = y.shape[-1] // 2
            y = F.gelu(y[:, :half], approximate="tanh") * y[:, half:]
        return y

    try:
        linear(layers[0][shapes[0][0]])
        torch.cuda.synchronize()
    except Exception as e:  # noqa: BLE001 - any failure means "not runnable on this image"
        return f"torch._scaled_mm unavailable: {str(e)[:120]}"

    def chunk():
        for _ in range(denoise_steps):
            for layer in layers:
                for name, _, _, _ in shapes:
                    linear(layer[name])

    g = HipGraph()
    g.capture(chunk, {})
    ts, _ = time_replays(g, steps, warmup)
    return round(statistics.median(ts) * 1e3 / denoise_steps, 2)


def decoder_layer_times(dev, layers, M, denoise_steps, steps, warmup):
    """The expert layer's linear path WITH its neighbours (adaptive norms before qkv / gate_up, gated
    residuals after o / down; reference models/pi05/modeling_pi05.py:812-835), two ways on the same
    tensors: `separate` = norm, quantizer, GEMM and addcmul as their own kernels (12 per layer, the
    reference's structure), `fused` = norm+quantizer in one kernel, addcmul in the GEMM epilogue
    (8 per layer).  Attention and RoPE are not part of either."""
    from phyai_amd import ops
    from phyai_amd.runtime import HipGraph

    D = 1024
    g = torch.Generator().manual_seed(777)
    h = torch.randn(M, D, generator=g).to(torch.bfloat16).to(dev)
    mods = [(torch.randn(1, 3 * D, generator=g) * 0.1).to(torch.bfloat16).to(dev) for _ in range(2)]
    attn = torch.randn(M, 2048, generator=g).to(torch.bfloat16).to(dev)
    h1 = torch.empty_like(h)
    h2 = torch.empty_like(h)

    def separate():
        for _ in range(denoise_steps):
            for layer in layers:
                q, o, gu, dn = layer["qkv"], layer["o"], layer["gate_up"], layer["down"]
                n, gate = ops.adarmsnorm(h, mods[0], 1e-6)
                ops.fp8_linear(n, q["w"], q["ws"], None, out=q["out"])
                y = ops.fp8_linear(attn, o["w"], o["ws"], None, out=o["out"])
                torch.addcmul(h, y, gate, out=h1)
                m, gate2 = ops.adarmsnorm(h1, mods[1], 1e-6)
                a = ops.fp8_linear(m, gu["w"], gu["ws"], None, epilogue="geglu_tanh", out=gu["out"],
                                   stream_weights=gu.get("stream", False))
                y2 = ops.fp8_linear(a, dn["w"], dn["ws"], None, out=dn["out"])
                torch.addcmul(h1, y2, gate2, out=h2)

    def fused():
        for _ in range(denoise_steps):
            for layer in layers:
                q, o, gu, dn = layer["qkv"], layer["o"], layer["gate_up"], layer["down"]
                (wq_, lq), (wo_, lo), (wg_, lg), (wd_, ld) = weight_of(q), weight_of(o), weight_of(gu), weight_of(dn)
                nq, ns, gate = ops.adarmsnorm_fp8(h, mods[0], 1e-6)
                ops.fp8_gemm(nq, ns, wq_, q["ws"], None, out=q["out"], weight_layout=lq)
                ops.fp8_linear(attn, wo_, o["ws"], None, residual=h, gate=gate, out=h1, weight_layout=lo)
                mq, ms, gate2 = ops.adarmsnorm_fp8(h1, mods[1], 1e-6)
                a = ops.fp8_gemm(mq, ms, wg_, gu["ws"], None, epilogue="geglu_tanh", out=gu["out"],
                                 stream_weights=gu.get("stream", False), weight_layout=lg)
                ops.fp8_linear(a, wd_, dn["ws"], None, residual=h1, gate=gate2, out=h2, weight_layout=ld)

    def one_launch_linears():
        for _ in range(denoise_steps):
            for layer in layers:
                q, o, gu, dn = layer["qkv"], layer["o"], layer["gate_up"], layer["down"]
                (wq_, lq), (wo_, lo), (wg_, lg), (wd_, ld) = weight_of(q), weight_of(o), weight_of(gu), weight_of(dn)
                n, gate = ops.adarmsnorm(h, mods[0], 1e-6)
                ops.fp8_linear(n, wq_, q["ws"], None, out=q["out"], weight_layout=lq)
                ops.fp8_linear(attn, wo_, o["ws"], None, residual=h, gate=gate, out=h1, weight_layout=lo)
                m, gate2 = ops.adarmsnorm(h1, mods[1], 1e-6)
                ops.fp8_mlp(m, wg_, gu["ws"], None, wd_, dn["ws"], None, epilogue="geglu_tanh", residual=h1, gate=gate2,
                            out=h2, stream_weights1=gu.get("stream", False), weight1_layout=lg, weight2_layout=ld)

    res = {}
    for name, fn in (("separate", separate), ("fused", fused), ("one_launch_linears", one_launch_linears)):
        gr = HipGraph()
        gr.capture(fn, {})
        ts, _ = time_replays(gr, steps, warmup)
        res[name] = round(statistics.median(ts) * 1e3 / denoise_steps, 2)
        del gr
    return res


def whole_step_times(dev, layers, M, prefix_len, denoise_steps, steps, warmup):
    """The whole flow-matching loop as ONE hipGraph - phyai_amd.runtime.expert_loop.ExpertDenoiseLoop,
    the mirror of the reference's runner loop (models/pi05/model_runner_pi05.py:689-738) and decoder
    layer (models/pi05/modeling_pi05.py:801-835) - on this benchmark's weights.  Attention (RoPE +
    torch SDPA over the prefix KV plus the chunk's own keys and values), embedding and projection
    are plain torch ops in BOTH variants: stand-ins for the reference's attention back end, which
    this library does not replace.  The variants differ in the linear path only: `library` = the
    fused layer (norm+quantizer, GEMM, GEMM+gated residual), `torch_path` = the reference's
    structure on torch ops (norm, quantizer expressions, torch._scaled_mm, gelu*mul, addcmul).
    Data chains through the layers.  Returns us per denoise step for each, or a reason string."""
    import phyai_amd.linear as L
    from phyai_amd.runtime.expert_loop import ExpertDenoiseLoop, ExpertLayer, PrefixAttentionStandIn

    D, ADIM = 1024, 32
    g = torch.Generator().manual_seed(4242)

    def rnd(*shape, scale=1.0):
        return (torch.randn(*shape, generator=g) * scale).to(torch.bfloat16).to(dev)

    L.init()
    try:
        mods = []
        for li, layer in enumerate(layers):
            lay = ExpertLayer(prefix=f"model.layers.{li}")
            for lin, name in ((lay.qkv_proj, "qkv"), (lay.o_proj, "o"), (lay.mlp.gate_up_proj, "gate_up"),
                              (lay.mlp.down_proj, "down")):
                lin.weight.data, lin.weight_scale.data = layer[name]["w"], layer[name]["ws"]
                lin.stream_weights = bool(layer[name].get("stream", False))
            for norm in (lay.input_layernorm, lay.post_attention_layernorm):
                norm.dense.weight.data.copy_(rnd(3 * D, D, scale=0.003))
                norm.dense.bias.data.copy_(rnd(3 * D, scale=0.03))
            mods.append(lay)
        attend = PrefixAttentionStandIn(len(layers), M, prefix_len, device=dev)
        time_emb = rnd(denoise_steps, D)
        noise = rnd(M, ADIM)
        res = {}
        for name, variant in (("library", "fused"), ("torch_path", "torch")):
            try:
                loop = ExpertDenoiseLoop(mods, attend, chunk_size=M, action_dim=ADIM, variant=variant, use_graph=False)
                loop.embed_action.weight.data.copy_(rnd(D, ADIM, scale=0.1))
                loop.project_action.weight.data.copy_(rnd(ADIM, D, scale=0.02))
                loop.embed_action.bias.data.zero_()
                loop.project_action.bias.data.zero_()
                loop.bind_euler_schedule(time_emb, -1.0 / denoise_steps, denoise_steps)
                out = loop.run(noise)    # eager first: anything this image cannot run shows up here, not inside a capture
                torch.cuda.synchronize()
                if not bool(torch.isfinite(out.float()).all()):
                    res[name] = "non-finite result"
                    continue
                loop.use_graph = True
                loop.setup()
                ts, _ = time_replays(loop.graph, steps, warmup)
                res[name] = round(statistics.median(ts) * 1e3 / denoise_steps, 2)
                del loop
            except Exception as e:  # noqa: BLE001 - report, do not fail the bench line
                res[name] = f"unavailable: {str(e)[:160]}"
        return res
    finally:
        L._reset_for_test()


def separate_qkv_times(dev, M, n_layers, denoise_steps, steps, warmup):
    """The expert layer with q, k and v as three linears (1024 -> 2048 / 256 / 256), the way the
    benchmark definition lists them, instead of the reference's fused qkv projection
    (layers/linear/layers.py:447-449): `three_linears` = three whole quantized linears (the
    activations are quantized three times), `shared_quantizer` = one quantizer launch and three
    GEMMs on its codes.  o, gate_up + GeGLU and down as in the headline.  us per denoise step."""
    from phyai_amd import ops
    from phyai_amd.runtime import HipGraph

    shapes = [("q", 2048, 1024, None), ("k", 256, 1024, None), ("v", 256, 1024, None)] + EXPERT_SET[1:]
    layers = make_layers(dev, shapes, M, n_layers, seed0=50_000)

    def rest(layer):
        for name, _, _, _ in EXPERT_SET[1:]:
            t = layer[name]
            ops.fp8_linear(t["x"], t["w"], t["ws"], None, epilogue=t["epi"], out=t["out"])

    def three_linears():
        for _ in range(denoise_steps):
            for layer in layers:
                for name in ("q", "k", "v"):
                    t = layer[name]
                    ops.fp8_linear(layer["q"]["x"], t["w"], t["ws"], None, out=t["out"])
                rest(layer)

    def shared_quantizer():
        for _ in range(denoise_steps):
            for layer in layers:
                xq, xs = ops.fp8_quant_rowwise(layer["q"]["x"])
                for name in ("q", "k", "v"):
                    t = layer[name]
                    ops.fp8_gemm(xq, xs, t["w"], t["ws"], None, out=t["out"])
                rest(layer)

    res = {}
    for name, fn in (("three_linears", three_linears), ("shared_quantizer", shared_quantizer)):
        gr = HipGraph()
        gr.capture(fn, {})
        ts, _ = time_replays(gr, steps, warmup)
        res[name] = round(statistics.median(ts) * 1e3 / denoise_steps, 2)
        del gr
    return res


def hardware_probe(dev):
    """Peaks re-measured on this box in the manner of the reference's probe
    (benchmark/pi05/hardware_probe.py:36-131): a large device-to-device copy counted as 2 x bytes, best
    of the runs; a large square GEMM at the path's precision (fp8 x fp8, 8192^3), best of the runs,
    through this library and through torch._scaled_mm (hipBLASLt); and the bare fp8 MFMA issue rate
    with the shader clock held under that load, which is the ceiling `fp8_TFLOPs` reports."""
    from phyai_amd import ops

    res = {}
    src = torch.empty(1 << 30, dtype=torch.uint8, device=dev).fill_(1)
    dst = torch.empty_like(src)
    for _ in range(3):
        dst.copy_(src)
    torch.cuda.synchronize()
    best = float("inf")
    for _ in range(12):
        a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        a.record()
        dst.copy_(src)
        b.record()
        torch.cuda.synchronize()
        best = min(best, a.elapsed_time(b))
    res["copy_GBps"] = round(2.0 * src.numel() / (best * 1e-3) / 1e9, 1)
    del src, dst
    n = 8192
    g = torch.Generator(device=dev).manual_seed(1)
    xq, xs = ops.fp8_quant_rowwise(torch.randn(n, n, generator=g, device=dev).to(torch.bfloat16))
    wq, ws = ops.fp8_weight_quant((torch.randn(n, n, generator=g, device=dev) * 0.02).to(torch.bfloat16))
    out = torch.empty(n, n, dtype=torch.bfloat16, device=dev)

    def best_of(fn, iters=10):
        for _ in range(3):
            fn()
        torch.cuda.synchronize()
        best = float("inf")
        for _ in range(iters):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            fn()
            b.record()
            torch.cuda.synchronize()
            best = min(best, a.elapsed_time(b))
        return round(2.0 * n ** 3 / (best * 1e-3) / 1e12, 1)

    res["fp8_gemm_8192_TFLOPs_this_library"] = best_of(lambda: ops.fp8_gemm(xq, xs, wq, ws, None, out=out))
    try:
        res["fp8_gemm_8192_TFLOPs_scaled_mm"] = best_of(
            lambda: torch._scaled_mm(xq, wq.t(), scale_a=xs, scale_b=ws.reshape(1, -1), out_dtype=torch.bfloat16, out=out))
    except Exception as e:  # noqa: BLE001 - torch._scaled_mm may not run on every image
        res["fp8_gemm_8192_TFLOPs_scaled_mm"] = f"unavailable: {str(e)[:80]}"
    # the instruction the path is bound by, with nothing else going on: issue rate and the clock the
    # chip holds under a chip-wide MFMA load (the vendor figure assumes the peak engine clock)
    probe = ops.mfma_rate_probe(workgroups=1024, iters=1000)
    res["fp8_mfma_issue_TFLOPs"] = probe["TFLOPs"]
    res["clock_GHz_under_mfma_load"] = probe["clock_GHz"]
    res["cycles_per_mfma_32x32x64"] = probe["cycles_per_mfma"]
    res["fp8_TFLOPs"] = probe["TFLOPs"]
    return res


def launch_floor_us(dev, nodes=2000):
    """Duration of one kernel node that does next to nothing (the quantizer on a single 8-element
    row: one wavefront), from a graph of `nodes` such launches in a row: what every kernel node of
    a replayed graph costs on this stack before it moves a byte."""
    from phyai_amd import ops
    from phyai_amd.runtime import HipGraph

    x = torch.zeros(1, 8, dtype=torch.bfloat16, device=dev)
    q = torch.empty(1, 8, dtype=torch.float8_e4m3fn, device=dev)
    sc = torch.empty(1, 1, dtype=torch.float32, device=dev)

    def fn():
        for _ in range(nodes):
            ops.fp8_quant_rowwise(x, out=q, scale_out=sc)

    g = HipGraph()
    g.capture(fn, {})
    ts, _ = time_replays(g, 10, 2)
    return statistics.median(ts) * 1e3 / nodes


def ops_plan(M, N, K, epi):
    """What the whole linear is launched as, for weights in the layout the benchmark passes."""
    from phyai_amd import ops

    lay = None
    if OPTS["operand"] and K % 128 == 0:
        lay = "operand_gated" if (epi is not None and "glu" in str(epi)) else "operand"
    return ops.describe_linear_plan(M, N, K, epi, weight_layout=lay)


def layer_plans(layer, shapes, M):
    """What each linear of a layer is launched as, by name (the second projection of an MLP that takes the
    first's row maxima: the part of phyai_fp8_describe_mlp_plan behind the bar)."""
    from phyai_amd import ops

    names = [name for name, _, _, _ in shapes]
    plans = {name: ops_plan(M, N, K, epi) for name, N, K, epi in shapes}
    for i in range(len(names) - 1):
        a, b = layer[names[i]], layer[names[i + 1]]
        if mlp_hands_over(a, b):
            first, second = ops.describe_mlp_plan(M, a["K"], b["K"], b["N"], a["epi"]).split(": ", 1)[1].split(" | ")
            plans[names[i]] = first + " (leaves its output's row maxima)"
            plans[names[i + 1]] = second + " (takes them)"
    return plans


def time_replays(graph, n, warmup):
    """HIP events around each replay, on the stream the replays are launched on."""
    for _ in range(warmup):
        graph.replay()
    torch.cuda.synchronize()
    evs = [(torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)) for _ in range(n)]
    t0 = time.perf_counter()
    for a, b in evs:
        a.record()
        graph.replay()
        b.record()
    torch.cuda.synchronize()
    wall = time.perf_counter() - t0
    return [a.elapsed_time(b) for a, b in evs], wall


def one_launch(M, N, K, epi) -> bool:
    """Does the whole linear run as one kernel (the GEMM that quantizes its own token rows)?"""
    from phyai_amd import ops

    return ops.describe_linear_plan(M, N, K, epi).startswith("one launch")


def weight_kernel_launch(xq, xs, t):
    """The kernel of a linear that reads its weights: the whole linear where that is one kernel,
    else the GEMM on codes and scales the quantizer left (its launch is not part of this figure)."""
    from phyai_amd import ops

    if one_launch(t["x"].shape[0], t["N"], t["K"], t["epi"]):
        linear(t)
    else:
        w, lay = weight_of(t)
        ops.fp8_gemm(xq, xs, w, t["ws"], None, epilogue=t["epi"], out=t["out"], stream_weights=t.get("stream", False),
                     weight_layout=lay)


def mlp_hands_over(a, b) -> bool:
    """Do both projections of this MLP run as one kernel each, the second on the first's row maxima?"""
    from phyai_amd import ops

    M = a["x"].shape[0]
    return OPTS["mlp"] and is_mlp_pair(a, b) and \
        ops.describe_mlp_plan(M, a["K"], b["K"], b["N"], a["epi"]).startswith("row maxima handed over")


def layer_weight_kernels(layer, shapes, codes):
    """The launches of one layer that read its weights, as the benchmark runs them: an MLP whose second
    projection takes the first's row maxima is one call of two kernels; a linear that is one kernel is that
    kernel; any other is the GEMM on the codes the quantizer left (`codes[name]`)."""
    names = [name for name, _, _, _ in shapes]
    i = 0
    while i < len(names):
        t = layer[names[i]]
        if i + 1 < len(names) and mlp_hands_over(t, layer[names[i + 1]]):
            mlp(t, layer[names[i + 1]])
            i += 2
        else:
            weight_kernel_launch(*codes[names[i]], t)
            i += 1


def gemm_only_times(dev, layers, shapes, M, reps=8, iters=30):
    """Average launch duration of the weight-reading kernel per shape: a graph holding only those
    launches (reps passes over the distinct per-layer weights)."""
    from phyai_amd import ops
    from phyai_amd.runtime import HipGraph

    out = {}
    for name, N, K, epi in shapes:
        pre = []
        for layer in layers:
            t = layer[name]
            xq, xs = ops.fp8_quant_rowwise(t["x"])
            pre.append((xq, xs, t))

        def fn():
            for _ in range(reps):
                for xq, xs, t in pre:
                    weight_kernel_launch(xq, xs, t)

        g = HipGraph()
        g.capture(fn, {})
        ts, _ = time_replays(g, iters, 3)
        launches = reps * len(pre)
        out[name] = statistics.median(ts) * 1e3 / launches  # us per launch
    # an MLP whose second projection takes the first's row maxima: the pair is timed as the one call it is,
    # and the second projection's kernel is that minus the first projection alone
    names = [name for name, _, _, _ in shapes]
    for i in range(len(names) - 1):
        if mlp_hands_over(layers[0][names[i]], layers[0][names[i + 1]]):
            def fn(a=names[i], b=names[i + 1]):
                for _ in range(reps):
                    for layer in layers:
                        mlp(layer[a], layer[b])

            g = HipGraph()
            g.capture(fn, {})
            ts, _ = time_replays(g, iters, 3)
            pair = statistics.median(ts) * 1e3 / (reps * len(layers))
            out[names[i] + "+" + names[i + 1]] = pair
            out[names[i + 1]] = pair - out[names[i]]
    return out


def gemm_only_layer_time(dev, layers, shapes, reps=8, iters=30, ready_codes=False):
    """Average duration of one layer's weight-reading kernels in the order and under the cache conditions
    of the benchmark: a graph holding only those launches, all shapes of a layer, layer
    after layer (the whole 311 MB of weights per pass, so no matrix is cache-warm by accident; a
    graph of one shape alone holds 47-151 MB, which fits the 256 MB Infinity Cache).
    ready_codes: every shape as the GEMM on codes the quantizer left (what this figure measured
    before a linear could be one kernel)."""
    from phyai_amd import ops
    from phyai_amd.runtime import HipGraph

    pre = [{name: ops.fp8_quant_rowwise(layer[name]["x"]) for name, _, _, _ in shapes} for layer in layers]

    def fn():
        for _ in range(reps):
            for layer, codes in zip(layers, pre):
                if ready_codes:
                    for name, _, _, _ in shapes:
                        t = layer[name]
                        w, lay = weight_of(t)
                        ops.fp8_gemm(*codes[name], w, t["ws"], None, epilogue=t["epi"], out=t["out"],
                                     stream_weights=t.get("stream", False), weight_layout=lay)
                else:
                    layer_weight_kernels(layer, shapes, codes)

    g = HipGraph()
    g.capture(fn, {})
    ts, _ = time_replays(g, iters, 3)
    return statistics.median(ts) * 1e3 / (reps * len(layers))   # us per layer (its four launches)


def sweep(dev):
    """Batched serving sweep (benchmark configuration 4): per (B, shape) the latency of the whole
    quantized linear (quantizer + GEMM + epilogue, graph replay over 6 distinct weight sets) and
    its fraction of the roofline that bounds it (HBM bytes or fp8 MFMA flops, whichever is slower)."""
    from phyai_amd import ops
    from phyai_amd.runtime import HipGraph

    rows = []
    cases = [(set_name, B, m1 * B, name, N, K, epi, False)
             for set_name, shapes, m1 in (("expert", EXPERT_SET, 50), ("prefill", PREFILL_SET, 816))
             for B in (1, 2, 4, 8, 16) for name, N, K, epi in shapes]
    cases += [("dit_block", 1, M, name, N, K, epi, True) for name, N, K, epi, M in DIT_SET]
    for set_name, B, M, name, N, K, epi, with_bias in cases:
        g = torch.Generator(device=dev).manual_seed(B * 1000 + N)
        gated = epi in ("geglu_tanh", "geglu_erf", "swiglu")
        items = []
        for _ in range(6):
            x = torch.randn(M, K, generator=g, device=dev)
            if set_name != "dit_block":
                idx = torch.randperm(K, generator=g, device=dev)[: K // 100]
                x[:, idx] *= 20.0                  # 1 % outlier channels
            w = (torch.randn(N, K, generator=g, device=dev) * 0.02).to(torch.bfloat16)
            wq, ws = ops.fp8_weight_quant(w)
            b = (torch.randn(N, generator=g, device=dev) * 0.01).to(torch.bfloat16) if with_bias else None
            n_out = N // 2 if gated else N
            # the layout the layers install after loading (Fp8Spec(operand_order=True)); `wp`: plain operand order
            # for the GEMM without the activation
            wl, lay, wp, play = wq, None, wq, None
            if OPTS["operand"] and K % 128 == 0:
                wp, play = ops.fp8_weight_to_operand_order(wq), "operand"
                wl, lay = (ops.fp8_weight_to_operand_order(wq, gated=True), "operand_gated") if gated else (wp, play)
            items.append((x.to(torch.bfloat16), wq, ws, b, torch.empty(M, n_out, dtype=torch.bfloat16, device=dev), wl, lay, wp, play))
            del w

        def fn():
            for x, _, ws, b, o, wl, lay, _, _ in items:
                ops.fp8_linear(x, wl, ws, b, epilogue=epi, out=o, weight_layout=lay)

        gr = HipGraph()
        gr.capture(fn, {})
        ts, _ = time_replays(gr, 15, 3)
        us = statistics.median(ts) * 1e3 / len(items)
        t_hbm = algorithmic_bytes(M, N, K, epi, with_bias) / (HBM_PEAK_GBS * 1e9) * 1e6
        t_mfma = 2.0 * M * N * K / (FP8_PEAK_TFLOPS * 1e12) * 1e6
        row = {"set": set_name, "B": B, "M": M, "shape": name, "us": round(us, 2),
               "bound": "hbm" if t_hbm >= t_mfma else "mfma",
               "roofline_us": round(max(t_hbm, t_mfma), 3),
               "frac": round(max(t_hbm, t_mfma) / us, 4)}
        del gr
        # the GEMM alone (codes ready, no activation) beside torch._scaled_mm - the call the
        # reference makes (layers/linear/backends/torch.py:168-175), hipBLASLt underneath
        pre = [(ops.fp8_quant_rowwise(x), wq, ws, b, torch.empty(M, N, dtype=torch.bfloat16, device=dev), wp, play)
               for x, wq, ws, b, _, _, _, wp, play in items]

        def ours():
            for (xq, xs), _, ws, b, o, wp, play in pre:
                ops.fp8_gemm(xq, xs, wp, ws, b, out=o, weight_layout=play)

        def blaslt():
            for (xq, xs), wq, ws, b, o, _, _ in pre:
                torch._scaled_mm(xq, wq.t(), scale_a=xs, scale_b=ws.reshape(1, -1), bias=b, out_dtype=torch.bfloat16, out=o)

        for key, f in (("gemm_us", ours), ("scaled_mm_us", blaslt)):
            try:
                f()
                torch.cuda.synchronize()
                gr = HipGraph()
                gr.capture(f, {})
                ts, _ = time_replays(gr, 10, 3)
                row[key] = round(statistics.median(ts) * 1e3 / len(pre), 2)
                del gr
            except Exception as e:  # noqa: BLE001 - torch._scaled_mm may not run on every image
                row[key] = f"unavailable: {str(e)[:80]}"
        rows.append(row)
        del items, pre
    rows += sweep_mlp(dev)
    return rows


def sweep_mlp(dev):
    """The MLP of either set as ONE call per layer (phyai_fp8_mlp: gate_up + GeGLU, then down on its output) beside the
    sum of its two GEMMs alone on ready codes, per batch size: what the second projection's quantizer costs when its
    row maxima come from the first projection's epilogue (M <= 128) and when it is a launch of its own."""
    from phyai_amd import ops
    from phyai_amd.runtime import HipGraph

    rows = []
    for set_name, shapes, m1 in (("expert", EXPERT_SET, 50), ("prefill", PREFILL_SET, 816)):
        (_, n1, H, epi), (_, O, I, _) = shapes[2], shapes[3]
        for B in (1, 2, 4, 8, 16):
            M = m1 * B
            g = torch.Generator(device=dev).manual_seed(B * 77 + n1)
            items = []
            for _ in range(6):
                x = torch.randn(M, H, generator=g, device=dev).to(torch.bfloat16)
                q1, s1 = ops.fp8_weight_quant((torch.randn(n1, H, generator=g, device=dev) * 0.02).to(torch.bfloat16))
                q2, s2 = ops.fp8_weight_quant((torch.randn(O, I, generator=g, device=dev) * 0.02).to(torch.bfloat16))
                p1, p2 = ops.fp8_weight_to_operand_order(q1), ops.fp8_weight_to_operand_order(q2)
                w1, l1, w2, l2 = q1, None, q2, None
                if OPTS["operand"]:
                    w1, l1, w2, l2 = ops.fp8_weight_to_operand_order(q1, gated=True), "operand_gated", p2, "operand"
                items.append(dict(x=x, w1=w1, l1=l1, s1=s1, w2=w2, l2=l2, s2=s2, p1=p1, p2=p2,
                                  out=torch.empty(M, O, dtype=torch.bfloat16, device=dev)))

            def whole():
                for t in items:
                    ops.fp8_mlp(t["x"], t["w1"], t["s1"], None, t["w2"], t["s2"], None, epilogue=epi, out=t["out"],
                                weight1_layout=t["l1"], weight2_layout=t["l2"])

            whole()
            for t in items:      # ready codes of both projections' inputs, outputs of the GEMMs alone
                t["c1"] = ops.fp8_quant_rowwise(t["x"])
                t["c2"] = ops.fp8_quant_rowwise(torch.randn(M, I, generator=g, device=dev).to(torch.bfloat16))
                t["o1"] = torch.empty(M, n1, dtype=torch.bfloat16, device=dev)

            def alone():
                for t in items:
                    ops.fp8_gemm(*t["c1"], t["p1"], t["s1"], None, out=t["o1"], weight_layout="operand")
                    ops.fp8_gemm(*t["c2"], t["p2"], t["s2"], None, out=t["out"], weight_layout="operand")

            us = {}
            for key, f in (("us", whole), ("gemm_us", alone)):
                f()
                torch.cuda.synchronize()
                gr = HipGraph()
                gr.capture(f, {})
                ts, _ = time_replays(gr, 15, 3)
                us[key] = round(statistics.median(ts) * 1e3 / len(items), 2)
                del gr
            t_hbm = (algorithmic_bytes(M, n1, H, epi, False) + algorithmic_bytes(M, O, I, None, False)) / (HBM_PEAK_GBS * 1e9) * 1e6
            t_mfma = 2.0 * M * (n1 * H + O * I) / (FP8_PEAK_TFLOPS * 1e12) * 1e6
            rows.append({"set": set_name, "B": B, "M": M, "shape": "mlp (gate_up + GeGLU, down)", "us": us["us"],
                         "bound": "hbm" if t_hbm >= t_mfma else "mfma", "roofline_us": round(max(t_hbm, t_mfma), 3),
                         "frac": round(max(t_hbm, t_mfma) / us["us"], 4), "gemm_us": us["gemm_us"], "scaled_mm_us": "-",
                         "plan": ops.describe_mlp_plan(M, H, I, O, epi)})
            del items
    return rows


def probe(dev, layers, M, shapes=EXPERT_SET):
    """Counter probe: per shape one launch per layer of the kernel that reads the weights (the whole
    linear where it is one kernel, else the GEMM on ready codes; distinct weight sets, so the
    weights come from HBM), then a 64 MiB device-to-device copy whose traffic is known (64 MiB
    read, 64 MiB written) to calibrate the counters."""
    from phyai_amd import ops

    names = [name for name, _, _, _ in shapes]
    for i, name in enumerate(names):
        pre = [(ops.fp8_quant_rowwise(layer[name]["x"]), layer[name]) for layer in layers]
        torch.cuda.synchronize()
        if i > 0 and mlp_hands_over(layers[0][names[i - 1]], layers[0][name]):
            # the second projection of an MLP exists only behind the first: the pair, one call per layer
            # (the first projection's kernel appears a second time in the trace)
            for layer in layers:
                mlp(layer[names[i - 1]], layer[name])
        else:
            for (xq, xs), t in pre:
                weight_kernel_launch(xq, xs, t)
        torch.cuda.synchronize()
    src = torch.empty(64 << 20, dtype=torch.uint8, device=dev).fill_(1)
    dst = torch.empty_like(src)
    torch.cuda.synchronize()
    for _ in range(4):
        dst.copy_(src)
    torch.cuda.synchronize()
    print("probe done")


def tile_kernel(plan):
    """The kernel behind a plan of a large-M GEMM."""
    return "gemm_fp8_tall_kernel" if "x256 " in plan and "in registers" in plan else "gemm_fp8_big_kernel"


def stamps_report(dev):
    """`--stamps`: the cycle budget of the GEMM kernels from inside (debug build of the library, whose kernels record the
    shader clock at the ends of their phases; csrc/stamps.h).  Per workload one launch with fresh weights; per phase the
    median over the wavefronts of the cycles between two stamps, the shader clock the launch ran at (against the 100 MHz
    counter), and the span from the first wavefront's start to the last one's end.  Prints a markdown table."""
    from phyai_amd import ops

    big = ["start -> first stage published", "main loop", "split-K sums gathered", "epilogue arithmetic, tile staged",
           "stores issued", "stores through"]
    # (one workgroup per CU takes tile after tile: of its last one)
    tall = ["start, tiles before -> first stage published", "main loop but for two stages", "everyone there", "last two stages and epilogue",
            "", "stores through"]
    small = ["start -> rows landed", "row scales known", "codes written", "MFMAs done", "partial sums exchanged",
             "epilogue, stores issued", "stores through"]
    work = [("prefill gate_up + GeGLU", 816, 32768, 2048, "geglu_tanh"), ("prefill down", 816, 2048, 16384, None),
            ("prefill qkv", 816, 2560, 2048, None), ("prefill o", 816, 2048, 2048, None),
            ("batched gate_up + GeGLU (B = 8)", 6528, 32768, 2048, "geglu_tanh"),
            ("expert qkv", 50, 2560, 1024, None), ("expert o", 50, 1024, 2048, None),
            ("expert gate_up + GeGLU", 50, 8192, 1024, "geglu_tanh")]
    only = os.environ.get("PHYAI_BENCH_STAMPS_ONLY")
    if only:
        work = [w for w in work if only in w[0]]
    print("| workload | kernel | clock GHz | first start -> last end, us | phase: median cycles per wavefront (10 % .. 90 %) |")
    print("|---|---|---|---|---|")
    for label, M, N, K, epi in work:
        lay = make_layers(dev, [("x", N, K, epi)], M, 2, seed0=4321)
        for t in (lay[0]["x"], lay[1]["x"]):      # first a warm-up launch on other weights, stamps off
            ops.debug_stamps(0)
            linear(lay[0]["x"])
            torch.cuda.synchronize()
        t = lay[1]["x"]
        small_m = one_launch(M, N, K, epi)
        if not small_m:
            xq, xs = ops.fp8_quant_rowwise(t["x"])
        rec = ops.debug_stamps(8192)
        if small_m:
            linear(t)
        else:
            w, wl = weight_of(t)
            ops.fp8_gemm(xq, xs, w, t["ws"], None, epilogue=t["epi"], out=t["out"], weight_layout=wl)
        torch.cuda.synchronize()
        ops.debug_stamps(0)
        r = rec.cpu().double()
        r = r[r[:, 0] > 0]
        plan = ops_plan(M, N, K, epi) if small_m else ops.describe_plan(M, N, K, epi, weight_layout=wl)
        names = small if small_m else tall if tile_kernel(plan) == "gemm_fp8_tall_kernel" else big
        last = ops.STAMP_WORDS - 3
        marks = [0] + [i for i in range(1, last) if bool((r[:, i] > 0).any())] + [last]
        clock = ((r[:, last] - r[:, 0]) / ((r[:, -1] - r[:, -2]).clamp_min(1) / 100e6) / 1e9).median().item()
        span = (r[:, -1].max() - r[:, -2].min()).item() / 100.0      # 100 MHz counter, common to the chip -> us
        cells = []
        for a, b in zip(marks[:-1], marks[1:]):
            d = (r[:, b] - r[:, a]).sort().values
            name = names[b - 1] if b != last else names[-1]
            cells.append(f"{name}: {d[len(d) // 2].item():.0f} ({d[len(d) // 10].item():.0f} .. {d[(9 * len(d)) // 10].item():.0f})")
        print(f"| {label} {M} x {N} x {K} | {plan}, {len(r)} wavefronts | {clock:.2f} | {span:.1f} | " + "; ".join(cells) + " |")
        del lay, rec


def cpu_info():
    """CPU model string and physical core count of the host (from /proc/cpuinfo)."""
    model, cores = "unknown", set()
    try:
        phys = core = None
        for line in open("/proc/cpuinfo", encoding="utf-8"):
            key, _, val = line.partition(":")
            key, val = key.strip(), val.strip()
            if key == "model name":
                model = val
            elif key == "physical id":
                phys = val
            elif key == "core id":
                core = val
            elif not key and phys is not None:
                cores.add((phys, core))
                phys = core = None
        if phys is not None:
            cores.add((phys, core))
    except OSError:
        pass
    return model, (len(cores) or os.cpu_count() or 1)


def _cpu_time(fn, budget_s, min_iters=20, warmup=5):
    for _ in range(warmup):
        fn()
    ts = []
    t_end = time.perf_counter() + budget_s
    while len(ts) < min_iters or (time.perf_counter() < t_end and len(ts) < 200):
        t0 = time.perf_counter()
        fn()
        ts.append(time.perf_counter() - t0)
    return {"p50_us": round(statistics.median(ts) * 1e6, 1), "min_us": round(min(ts) * 1e6, 1), "iters": len(ts)}


def cpu_baseline(layers, shapes, M, n_layers):
    """The reference's CPU form of the same linears - torch dequantize + matmul - on this box's host
    cores, on layer 0's tensors (the bits the GPU run uses): GEMM only (codes and scales ready) and
    quantizer + GEMM (+ GeGLU), at all threads and at one thread, plus benchmark configuration 1
    (50 x 4096 x 1024 with bias).  Per-layer times; the headline value scales the all-threads
    quantizer + GEMM figure by the number of layers."""
    from oracle import ref

    items = []
    for name, N, K, epi in shapes:
        t = layers[0][name]
        wq, ws = ref.weight_quant(t["w_bf16_cpu"])
        xq, xs = ref.quant_rowwise(t["x_cpu"])
        items.append((t["x_cpu"], xq, xs, wq, ws, {None: 0, "geglu_tanh": 1}[epi]))
    g = torch.Generator().manual_seed(0)
    x1 = torch.randn(50, 1024, generator=g).to(torch.bfloat16)
    w1q, w1s = ref.weight_quant((torch.randn(4096, 1024, generator=g) * 0.02).to(torch.bfloat16))
    b1 = (torch.randn(4096, generator=g) * 0.01).to(torch.bfloat16)

    def layer_full():
        for x, _, _, wq, ws, epi in items:
            ref.linear(x, wq, ws, None, epi)

    def layer_gemm_only():
        for _, xq, xs, wq, ws, epi in items:
            ref.epilogue(ref.gemm_f32(xq, xs, wq, ws, None), epi)

    def config1():
        ref.linear(x1, w1q, w1s, b1, 0)

    all_threads = torch.get_num_threads()
    out = {}
    try:
        for label, nthreads, budget in (("all_threads", all_threads, 4.0), ("one_thread", 1, 2.5)):
            torch.set_num_threads(nthreads)
            out[label] = {"threads": nthreads,
                          "layer_quantizer_gemm": _cpu_time(layer_full, budget),
                          "layer_gemm_only": _cpu_time(layer_gemm_only, budget),
                          "config1_linear": _cpu_time(config1, budget / 4)}
        # benchmark configuration 3: one layer of the prefix-prefill set (M = 816, 180 GFLOP), all threads,
        # a handful of passes (own seeded tensors: the GPU run's prefill layers are not kept on the host)
        torch.set_num_threads(all_threads)
        pitems = []
        for i, (name, N, K, epi) in enumerate(PREFILL_SET):
            gp = torch.Generator().manual_seed(20_000 + i)
            wq, ws = ref.weight_quant((torch.randn(N, K, generator=gp) * 0.02).to(torch.bfloat16))
            pitems.append((torch.randn(816, K, generator=gp).to(torch.bfloat16), wq, ws, {None: 0, "geglu_tanh": 1}[epi]))

        def prefill_layer():
            for x, wq, ws, epi in pitems:
                ref.linear(x, wq, ws, None, epi)

        out["all_threads"]["prefill_layer_quantizer_gemm_M816"] = _cpu_time(prefill_layer, 6.0, min_iters=5, warmup=1)
        del pitems
    finally:
        torch.set_num_threads(all_threads)
    model, phys = cpu_info()
    full = out["all_threads"]["layer_quantizer_gemm"]
    return {"value": round(full["p50_us"] * n_layers, 1), "unit": "us per denoise step", "cores": all_threads,
            "kind": "port", "cpu_model": model, "physical_cores": phys,
            "sample": f"torch CPU dequantize+matmul incl. quantizer and GeGLU on 1 of {n_layers} layers (4 linears, "
                      f"M={M}), p50 of {full['iters']} passes at {all_threads} threads, scaled x{n_layers}; `variants` "
                      "holds the per-layer times (us) of GEMM only and quantizer+GEMM at all threads and at one "
                      "thread, benchmark configuration 1, and one layer of the prefix-prefill set (configuration 3, "
                      "M = 816, at least 5 passes at all threads)",
            "variants": out}


def main() -> int:
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=200)
    ap.add_argument("--warmup", type=int, default=20)
    ap.add_argument("--no-cpu-baseline", action="store_true")
    ap.add_argument("--no-prefill", action="store_true")
    ap.add_argument("--no-cache-plan", action="store_true",
                    help="read every weight matrix with ordinary loads (no matrix is streamed past the Infinity Cache)")
    ap.add_argument("--no-extras", action="store_true",
                    help="skip the comparisons in `extra` (fused decoder-layer path, torch reference path): "
                         "only this library's kernels run, for profiler sessions")
    ap.add_argument("--sweep", action="store_true",
                    help="also time the batched-serving sweep (B = 1..16, both linear sets, outlier channels)")
    ap.add_argument("--probe", action="store_true",
                    help="launch each expert GEMM shape a few times plus a 64 MiB device copy and exit; "
                         "meant to run under `rocprofv3 --pmc FETCH_SIZE` / `--pmc WRITE_SIZE`")
    ap.add_argument("--probe-prefill", action="store_true",
                    help="the same for the prefill GEMM shapes (M = 816, 4 weight sets), for the MFMA / LDS counters")
    ap.add_argument("--probe-m", type=int, default=816,
                    help="token rows of --probe-prefill (816 x batch for the batched-serving shapes)")
    ap.add_argument("--stamps", action="store_true",
                    help="cycle budgets of the GEMM kernels from time stamps inside them: needs the debug build of the "
                         "library (`make -C phyai_amd/csrc stamps`), prints a markdown table and exits")
    ap.add_argument("--row-major", action="store_true",
                    help="A/B: pass the weights row-major [N, K] instead of in MFMA operand order")
    ap.add_argument("--separate-linears", action="store_true",
                    help="A/B: gate_up and down as two phyai_fp8_linear calls instead of one phyai_fp8_mlp call")
    args = ap.parse_args()
    OPTS["operand"] = not args.row_major
    OPTS["mlp"] = not args.separate_linears
    if args.stamps:
        os.environ["PHYAI_FP8_LIBRARY"] = "stamps"            # before the library is opened
    if args.gpus != 1 or int(os.environ.get("WORLD_SIZE", "1")) != 1:
        print("bench.py: this path is built and measured on ONE GPU (TP=1, no collectives); "
              "run with --gpus 1", file=sys.stderr)
        return 2
    if not torch.cuda.is_available():
        print("bench.py: no GPU visible", file=sys.stderr)
        return 2

    from phyai_amd.runtime import HipGraph

    dev = torch.device("cuda", 0)
    torch.cuda.set_device(dev)
    M, n_layers, denoise_steps = 50, 18, 10

    if args.stamps:
        stamps_report(dev)
        return 0
    if args.probe_prefill:
        probe(dev, make_layers(dev, PREFILL_SET, args.probe_m, 4, seed0=10_000), args.probe_m, PREFILL_SET)
        return 0

    layers = make_layers(dev, EXPERT_SET, M, n_layers)
    # What a runner does once per model: the weights of one denoise step (311 MB) exceed the 256 MB
    # Infinity Cache, so the largest matrices are read past it and the others stay resident from
    # step to step (phyai_amd/cache_plan.py).
    from phyai_amd.cache_plan import choose_streamed
    entries = [layer[name] for layer in layers for name, _, _, _ in EXPERT_SET]
    frac = float(os.environ.get("PHYAI_BENCH_RESIDENT_FRACTION", "0.7"))
    for t, streamed in zip(entries, choose_streamed([t["N"] * t["K"] for t in entries], resident_fraction=frac)):
        t["stream"] = streamed and not args.no_cache_plan
    streamed_mb = sum(t["N"] * t["K"] for t in entries if t["stream"]) / 1e6
    resident_mb = sum(t["N"] * t["K"] for t in entries if not t["stream"]) / 1e6

    if args.probe:
        probe(dev, layers, M)
        return 0

    def chunk():
        for _ in range(denoise_steps):
            run_layers(layers, EXPERT_SET)

    graph = HipGraph()
    graph.capture(chunk, {})
    torch.cuda.synchronize()
    ts_ms, wall = time_replays(graph, args.steps, args.warmup)
    ms_per_step = wall * 1e3 / args.steps
    p50_replay_ms = statistics.median(ts_ms)
    value_us = p50_replay_ms * 1e3 / denoise_steps

    # ---- roofline of the dominant kernel (the small-M GEMM) --------------------
    per_launch_us = gemm_only_times(dev, layers, EXPERT_SET, M)
    layer_bytes = sum(algorithmic_bytes(M, N, K, epi) for _, N, K, epi in EXPERT_SET)
    layer_us = gemm_only_layer_time(dev, layers, EXPERT_SET)
    achieved = layer_bytes / (layer_us * 1e-6) / 1e9
    roofline = {
        "bound": "hbm", "achieved": round(achieved, 1), "peak": HBM_PEAK_GBS, "unit": "GB/s",
        "frac": round(achieved / HBM_PEAK_GBS, 4), "traffic": profiled_layer_traffic(),
        "kernel": "gemm_fp8_fusedq_kernel (M=50, four expert shapes)",   # completed below from the plans
        "bytes_per_layer": layer_bytes, "us_per_layer": round(layer_us, 3),
        "note": "achieved = bytes_per_layer / us_per_layer, the four weight-reading launches of a layer (the whole "
                "linear where it is one kernel that quantizes its own rows, else the GEMM behind the quantizer) timed "
                "in a graph of those launches only that walks all 18 layers (311 MB of weights per pass); per_shape "
                "times come from graphs of one shape alone, whose 47-151 MB of weights fit the Infinity Cache",
        "plans": layer_plans(layers[0], EXPERT_SET, M),
        "weight_layout": "MFMA operand order (re-laid once after loading)" if OPTS["operand"] else "row-major [N, K]",
        "gemm_on_ready_codes": None,
        "per_shape": {name: {"us": round(per_launch_us[name], 3),
                             "GB/s": round(algorithmic_bytes(M, N, K, epi) / per_launch_us[name] / 1e3, 1)}
                      for name, N, K, epi in EXPERT_SET},
        "per_pair_us": {k: round(v, 3) for k, v in per_launch_us.items() if "+" in k},
        "whole_path_frac": round(layer_bytes * n_layers / (value_us * 1e-6) / 1e9 / HBM_PEAK_GBS, 4),
    }
    if not all(p.startswith("one launch") for p in roofline["plans"].values()):
        roofline["kernel"] = "gemm_fp8_fusedq_kernel + gemm_fp8_skinny_kernel (M=50, four expert shapes)"
    if not args.no_extras:
        codes_us = gemm_only_layer_time(dev, layers, EXPERT_SET, ready_codes=True)
        roofline["gemm_on_ready_codes"] = {
            "us_per_layer": round(codes_us, 3), "frac": round(layer_bytes / (codes_us * 1e-6) / 1e9 / HBM_PEAK_GBS, 4),
            "note": "the four GEMM launches of a layer on codes and scales the quantizer left (phyai_fp8_gemm): what "
                    "`frac` measured before a linear could be one kernel; the quantization is not in this figure"}
    # (profiler sessions pass --no-extras: then only the benchmark's own kernels run)
    measured = None if args.no_extras else hardware_probe(dev)
    if measured is not None:
        roofline["measured_peak_GBps"] = measured["copy_GBps"]
        roofline["frac_of_measured_peak"] = round(achieved / measured["copy_GBps"], 4)
    node_us = launch_floor_us(dev)
    # one kernel per linear where it quantizes its own rows, else a quantizer and a GEMM
    nodes_per_layer = sum(1 if p.startswith("one launch") else 2 for p in roofline["plans"].values())
    floor_us = node_us * nodes_per_layer
    launch_floor = {
        "node_us": round(node_us, 3), "nodes_per_layer": nodes_per_layer, "floor_us_per_layer": round(floor_us, 2),
        "floor_us_per_denoise_step": round(floor_us * n_layers, 1),
        "ceiling_whole_path_frac": round(layer_bytes / (floor_us * 1e-6) / 1e9 / HBM_PEAK_GBS, 4),
        "note": "time of a kernel node that moves nothing, times the nodes a layer's four quantized linears take "
                "(one where the GEMM quantizes its own rows, else quantizer + GEMM): no kernel, however fast, brings "
                "the layer below floor_us_per_layer in this "
                "structure, i.e. the whole path cannot exceed ceiling_whole_path_frac of HBM peak"}

    # ---- prefix prefill (M = 816): MFMA-bound regime -----------------------------
    # `value` is the median of exactly --steps replays; the distribution beside it is taken over at
    # least 200 (more replays of the same graph, outside the timed region, when --steps is smaller)
    more_ms = list(ts_ms)
    if len(more_ms) < 200:
        more_ms += time_replays(graph, 200 - len(more_ms), 0)[0]
    srt = sorted(more_ms)
    extra = {"denoise_step_us": {"p50": round(statistics.median(srt) * 1e3 / denoise_steps, 2),
                                 "p90": round(srt[min(len(srt) - 1, (9 * len(srt)) // 10)] * 1e3 / denoise_steps, 2),
                                 "min": round(srt[0] * 1e3 / denoise_steps, 2), "replays": len(srt),
                                 "p50_of_the_timed_steps": round(value_us, 2), "timed_steps": len(ts_ms)}}
    roofline_prefill = None
    if not args.no_prefill:
        # all 18 layers of the prefix backbone in one graph (2 GB of fp8 weights): with a handful of
        # layers the ~20 us a graph launch costs would be a few us per layer
        pl = make_layers(dev, PREFILL_SET, 816, n_layers, seed0=10_000)
        pg = HipGraph()
        pg.capture(lambda: run_layers(pl, PREFILL_SET), {})
        pts, _ = time_replays(pg, 30, 3)
        p_layer_us = statistics.median(pts) * 1e3 / len(pl)
        flops = sum(2 * 816 * N * K for _, N, K, _ in PREFILL_SET)
        tref = "skipped" if args.no_extras else torch_reference_times(dev, pl, PREFILL_SET, 1, 10, 3)
        extra["prefill_M816"] = {"torch_reference_path_us_per_layer": (round(tref / len(pl), 2) if not isinstance(tref, str) else tref),
                                 "us_per_layer": round(p_layer_us, 2),
                                 "TFLOP/s": round(flops / (p_layer_us * 1e-6) / 1e12, 1),
                                 "frac_fp8_peak": round(flops / (p_layer_us * 1e-6) / 1e12 / FP8_PEAK_TFLOPS, 4)}
        # the MFMA-bound regime's own roofline object: the GEMM launches alone, per shape, and the
        # dominant one (gate_up + GeGLU, 61 % of the layer's flops) against the fp8 peak
        p_gemm_us = gemm_only_times(dev, pl, PREFILL_SET, 816, reps=1, iters=15)
        per_shape = {name: {"us": round(p_gemm_us[name], 2),
                            "TFLOP/s": round(2.0 * 816 * N * K / p_gemm_us[name] / 1e6, 1),
                            "kernel": ops_plan(816, N, K, epi)}
                     for name, N, K, epi in PREFILL_SET}
        dom = per_shape["gate_up"]
        roofline_prefill = {
            "bound": "mfma", "kernel": tile_kernel(dom["kernel"]) + " (gate_up 2048->32768 + GeGLU at M=816: " + dom["kernel"] + ")",
            "achieved": dom["TFLOP/s"], "peak": FP8_PEAK_TFLOPS, "unit": "TFLOP/s",
            "frac": round(dom["TFLOP/s"] / FP8_PEAK_TFLOPS, 4), "us": dom["us"],
            "measured_peak_TFLOPs": measured["fp8_TFLOPs"] if measured else None,
            "frac_of_measured_peak": round(dom["TFLOP/s"] / measured["fp8_TFLOPs"], 4) if measured else None,
            "per_shape": per_shape,
            "layer_gemms_us": round(sum(v["us"] for v in per_shape.values()), 2),
            "layer_gemms_frac": round(flops / (sum(v["us"] for v in per_shape.values()) * 1e-6) / 1e12 / FP8_PEAK_TFLOPS, 4),
            "whole_layer_frac": extra["prefill_M816"]["frac_fp8_peak"],
            "note": "GEMM launches alone on ready codes (graphs of one shape over the 18 layers' distinct weights); whole_layer_frac "
                    "includes the four quantizer launches"}
        del pl, pg
    if not args.no_extras:
        dl = decoder_layer_times(dev, layers, M, denoise_steps, max(20, args.steps // 4), 5)
        lin = {name: (1 if one_launch(M, N, K, epi) else 2) for name, N, K, epi in EXPERT_SET}
        extra["expert_step_with_norms_and_residuals_us"] = {
            **dl, "note": "per denoise step, 18 layers: adaptive norm -> qkv, o -> gated residual, adaptive norm -> "
                          "gate_up+GeGLU, down -> gated residual; kernels per layer: separate = "
                          f"{4 + sum(lin.values())} (2 norms, 2 addcmul, the four linears), fused = "
                          f"{4 + lin['o'] + lin['down']} (2 norm+quantizer, qkv and gate_up GEMMs on their codes, o and down "
                          "with the gated residual in the epilogue), one_launch_linears = 6 (2 norms writing bf16, qkv and "
                          "o + residual as one-launch linears, the MLP as one call of two kernels with the residual behind it)"}
        extra["torch_reference_path_us"] = {
            "expert_step": torch_reference_times(dev, layers, EXPERT_SET, denoise_steps, max(10, args.steps // 10), 3),
            "note": "same linears through the reference's own arithmetic on this GPU: torch-op quantizer + "
                    "torch._scaled_mm (+ torch GELU*up); compare with `value`"}
        extra["separate_q_k_v_step_us"] = {
            **separate_qkv_times(dev, M, n_layers, denoise_steps, max(10, args.steps // 10), 3),
            "note": "q / k / v as three projections (1024->2048/256/256) as the benchmark definition lists them; the "
                    "headline uses the reference's fused qkv projection (one 1024->2560 GEMM)"}
        extra["whole_denoise_step_us"] = {
            **whole_step_times(dev, layers, M, 816, denoise_steps, max(10, args.steps // 10), 3),
            "note": "per denoise step with everything between the linears: action embedding, RoPE, joint attention "
                    "over 816 prefix + 50 chunk positions (torch SDPA stand-in, same in both), norms, gated "
                    "residuals, final norm, projection, Euler update; data chains through the 18 layers"}
    if args.sweep:
        extra["batched_sweep"] = sweep(dev)
        # the same rows as a markdown table, on stderr (stdout carries the one JSON line)
        print("| set | B | M | shape | us per linear | bound | roofline us | fraction | GEMM alone us | torch._scaled_mm us |", file=sys.stderr)
        print("|---|---|---|---|---|---|---|---|---|---|", file=sys.stderr)
        for r in extra["batched_sweep"]:
            print(f"| {r['set']} | {r['B']} | {r['M']} | {r['shape']} | {r['us']} | {r['bound']} | {r['roofline_us']} | {r['frac']} | "
                  f"{r.get('gemm_us', '-')} | {r.get('scaled_mm_us', '-')} |", file=sys.stderr)

    cpu = None
    if not args.no_cpu_baseline:
        cpu = cpu_baseline(layers, EXPERT_SET, M, n_layers)

    line = {
        "metric": "p50 \u00b5s per Pi0.5 expert denoise-step linears (fp8 W8A8) + % HBM/MFMA roofline",
        "value": round(value_us, 2), "unit": "us", "n_gpus": 1, "steps": args.steps, "warmup": args.warmup,
        "ms_per_step": round(ms_per_step, 4), "higher_is_better": False, "scaling": "weak",
        "vs_baseline": None, "dtype": "fp8_e4m3fn x fp8_e4m3fn -> fp32 acc -> bf16", "data": "synthetic",
        "config": {"workload": "action-expert linear set: 18 layers x {qkv 1024->2560, o 2048->1024, "
                               "gate_up 1024->8192 + GeGLU, down 4096->1024}, M=50, distinct weights per layer",
                   "step": "one hipGraph replay = 10 denoise steps = 720 quantized linears",
                   "denoise_steps_per_replay": denoise_steps, "cache_policy":
                   (f"311 MB of weights per denoise step against a 256 MB Infinity Cache: {streamed_mb:.0f} MB (the largest "
                    f"matrices) are read with non-temporal loads, the other {resident_mb:.0f} MB may stay cached from "
                    "step to step; nothing is pinned" if streamed_mb else
                    "311 MB of weights per denoise step cycle through HBM; every matrix is read with ordinary loads")},
        "roofline": roofline, "roofline_prefill": roofline_prefill, "launch_floor": launch_floor,
        "measured_peaks": measured, "cpu_baseline": cpu, "extra": extra,
    }
    print(json.dumps(line))
    return 0


if __name__ == "__main__":
    sys.exit(main())
