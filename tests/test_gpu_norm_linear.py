"""An adaptive RMSNorm in front of a linear or an MLP as one C call (phyai_fp8_adarmsnorm_linear / _mlp): bit-equal to
the norm + quantizer kernel followed by the same linear on its codes, wherever the norm runs - inside the one-launch
small-M kernel (one modulation row, up to 128 token rows, K <= 2048) or as a launch of its own - and for both weight
layouts, one and two K steps per wavefront, K that is no multiple of 512, and rows that hold Inf or NaN."""

from __future__ import annotations

import pytest
import torch

from conftest import seeded

pytestmark = pytest.mark.gpu

EPS = 1e-6
EPI = {None: 0, "geglu_tanh": 1, "swiglu": 3}


def _workspace(nbytes, dev):
    ws = torch.full((nbytes,), 0xAB, dtype=torch.uint8, device=dev)
    ws[:16384] = 0
    return ws


def _same(a, b):
    assert a.shape == b.shape and torch.equal(a.isnan(), b.isnan()) and torch.equal(a.nan_to_num(), b.nan_to_num())


def _weights(dev, n, k, seed, layout):
    from phyai_amd import ops

    w, s = ops.fp8_weight_quant(seeded((n, k), seed, 0.02).to(dev))
    return (ops.fp8_weight_to_operand_order(w, gated=layout == "operand_gated") if layout else w), s


def _rows(dev, M, K, mod_rows, odd_rows):
    x, mod = seeded((M, K), M + K, 1.5), seeded((mod_rows, 3 * K), M + K + 1, 0.2)
    if odd_rows:
        x[0, K - 1] = float("inf")
        x[M // 2, 3] = float("nan")
        x[M - 1] = 0.0
    return x.to(dev), mod.to(dev)


def _norm_linear(x, mod, w, s, bias, epi, layout):
    """(output, whether the norm ran inside the linear: the region of the workspace that holds codes is untouched)"""
    from phyai_amd import _lib, ops

    M, K = x.shape
    N = w.shape[0]
    need = _lib.load().phyai_fp8_linear_workspace_bytes(M, N, K, EPI[epi])
    ws = _workspace(need, x.device)
    out = torch.full((M, N // 2 if epi else N), -7.0, dtype=torch.bfloat16, device=x.device)
    rc = _lib.load().phyai_fp8_adarmsnorm_linear(
        x.data_ptr(), K, mod.data_ptr(), 3 * K, mod.shape[0], EPS, w.data_ptr(), s.data_ptr(), bias.data_ptr() if bias is not None else None,
        out.data_ptr(), out.shape[1], M, N, K, EPI[epi] | ops.WEIGHT_LAYOUTS[layout], ws.data_ptr(), need, torch.cuda.current_stream().cuda_stream)
    _lib.check(rc, "phyai_fp8_adarmsnorm_linear")
    return out, bool((ws[16384:] == 0xAB).all())


def _want_linear(x, mod, w, s, bias, epi, layout):
    from phyai_amd import ops

    xq, xs, _ = ops.adarmsnorm_fp8(x, mod, EPS)
    return ops.fp8_gemm(xq, xs, w, s, bias, epilogue=epi, weight_layout=layout)


@pytest.mark.parametrize("K", [128, 384, 512, 896, 1024, 1152, 1664, 2048])
@pytest.mark.parametrize("M,odd_rows", [(1, False), (7, True), (50, False), (50, True), (128, True)])
@pytest.mark.parametrize("epi", [None, "geglu_tanh"])
@pytest.mark.parametrize("operand", [False, True])
def test_norm_inside_the_linear(dev, operand, epi, M, odd_rows, K):
    N = 512 if M == 128 else 1056
    layout = None if not operand else ("operand_gated" if epi else "operand")
    x, mod = _rows(dev, M, K, 1, odd_rows)
    w, s = _weights(dev, N, K, K + N, layout)
    bias = seeded((N,), 3).to(dev)
    got, inside = _norm_linear(x, mod, w, s, bias, epi, layout)
    assert inside, "this shape is meant to take the kernel that normalises its own rows"
    _same(got, _want_linear(x, mod, w, s, bias, epi, layout))


@pytest.mark.parametrize("M,N,K,mod_rows,epi,layout", [
    (50, 512, 1024, 2, None, None),                     # a modulation row per sample: the kernel takes one for all
    (48, 512, 1024, 48, "geglu_tanh", "operand_gated"),
    (129, 512, 1024, 1, None, "operand"),               # more token rows than it serves
    (300, 544, 640, 3, "geglu_tanh", None),
    (50, 512, 2176, 1, None, "operand"),                # K beyond its registers
    (50, 528, 1040, 1, None, None),                     # K that is no multiple of a K step
    (50, 512, 1024, 1, "swiglu", None),                 # an epilogue it does not have
    (128, 8192, 1024, 1, None, None),                   # more workgroups than one round
])
def test_norm_in_front_of_the_linear(dev, M, N, K, mod_rows, epi, layout):
    x, mod = _rows(dev, M, K, mod_rows, M == 50)
    w, s = _weights(dev, N, K, K + N, layout)
    got, inside = _norm_linear(x, mod, w, s, None, epi, layout)
    assert not inside
    _same(got, _want_linear(x, mod, w, s, None, epi, layout))


@pytest.mark.parametrize("M,H,I,mod_rows,epi,operand", [
    (1, 128, 256, 1, "geglu_tanh", False), (50, 1024, 4096, 1, "geglu_tanh", True), (50, 1024, 4096, 1, "geglu_tanh", False),
    (33, 896, 1280, 1, "geglu_tanh", True), (20, 1664, 2048, 1, "geglu_tanh", True), (128, 384, 512, 1, "geglu_tanh", False),
    (50, 1024, 2048, 5, "geglu_tanh", True), (50, 512, 1040, 1, "swiglu", False), (260, 512, 1024, 2, "geglu_tanh", True),
    (40, 2176, 512, 1, "geglu_tanh", False)])
@pytest.mark.parametrize("residual", [False, True])
def test_norm_in_front_of_an_mlp(dev, M, H, I, mod_rows, epi, operand, residual):
    from phyai_amd import _lib, ops

    lib, O = _lib.load(), H
    x, mod = _rows(dev, M, H, mod_rows, False)
    w1, s1 = _weights(dev, 2 * I, H, 1, "operand_gated" if operand else None)
    w2, s2 = _weights(dev, O, I, 2, "operand" if operand else None)
    f1, f2 = (ops.FLAG_W_OPERAND_GATED, ops.FLAG_W_OPERAND_ORDER) if operand else (0, 0)
    need = lib.phyai_fp8_mlp_workspace_bytes(M, H, I, O, EPI[epi])
    ws, out = _workspace(need, dev), torch.empty(M, O, dtype=torch.bfloat16, device=dev)
    gate = mod[:, 2 * H:]                                # the gate part of the modulation, where it lies
    res_args = (x.data_ptr(), H, gate.data_ptr(), 3 * H, mod_rows) if residual else (None, 0, None, 0, 0)
    rc = lib.phyai_fp8_adarmsnorm_mlp(x.data_ptr(), H, mod.data_ptr(), 3 * H, mod_rows, EPS, w1.data_ptr(), s1.data_ptr(), None, f1,
                                      w2.data_ptr(), s2.data_ptr(), None, f2, *res_args, out.data_ptr(), O, M, H, I, O, EPI[epi],
                                      ws.data_ptr(), need, torch.cuda.current_stream().cuda_stream)
    _lib.check(rc, "phyai_fp8_adarmsnorm_mlp")
    h = _want_linear(x, mod, w1, s1, None, epi, "operand_gated" if operand else None)
    extra = dict(residual=x, gate=gate.contiguous()) if residual else {}
    _same(out, ops.fp8_linear(h, w2, s2, weight_layout="operand" if operand else None, **extra))
    assert not ws[:16384].any(), "the counters are left at zero"


@pytest.mark.parametrize("M,mod_rows", [(50, 1), (50, 2), (200, 1), (200, 4)])
@pytest.mark.parametrize("operand", [False, True])
def test_decoder_layer_equals_its_separate_calls(dev, M, mod_rows, operand):
    """The layer's three calls at other sizes than the denoise loop's, with weights re-laid as a serving engine has them."""
    import phyai_amd.linear as L
    from phyai_amd.runtime.expert_loop import ExpertLayer, ExpertLayerModulation

    L.init()
    try:
        H, HD, heads, I = 640, 128, 4, 1280
        layer = ExpertLayer(H, HD, heads, 1, I, H, spec=L.Fp8Spec(operand_order=operand))
        for j, lin in enumerate((layer.qkv_proj, layer.o_proj, layer.mlp.gate_up_proj, layer.mlp.down_proj)):
            lin.spec.quantize_weight_(lin, seeded(tuple(lin.weight.shape), 50 + j, 0.02).to(dev))
            lin.post_load()
            assert bool(lin.weight_layout) == operand
        mod = ExpertLayerModulation(seeded((mod_rows, 3 * H), 60, 0.1).to(dev), seeded((mod_rows, 3 * H), 61, 0.1).to(dev))
        x, attend = seeded((M, H), 62).to(dev), lambda fused, index: fused[:, :HD * heads]
        n, g1 = layer.input_layernorm(x, modulation=mod.input_ln)
        per_row = lambda g: g.repeat_interleave(M // mod_rows, 0)
        h = torch.addcmul(x, layer.o_proj(attend(layer.qkv_proj(n)[0], 0))[0], per_row(g1))
        n, g2 = layer.post_attention_layernorm(h, modulation=mod.post_attention_ln)
        assert torch.equal(layer(x, attend, 0, mod), torch.addcmul(h, layer.mlp(n), per_row(g2)))
    finally:
        L._reset_for_test()
