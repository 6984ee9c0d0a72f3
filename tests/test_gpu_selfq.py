"""Small-M linears that quantize their own rows at any K (csrc/gemm_selfq.h) against quantizer + GEMM, bit for bit:
partial and missing K steps, row groups of four, every number of weight tiles, own / handed-over / static scales, NaN and
Inf in rows; the reciprocal form of the static and weight quantizers against the division on the CPU; and weights re-laid in place."""

from __future__ import annotations

import pytest
import torch

from conftest import seeded

pytestmark = pytest.mark.gpu


def _two_launches(monkeypatch, call):
    with monkeypatch.context() as m:
        m.setenv("PHYAI_FP8_FUSED", "0")
        return call()


def _same(a, b):
    assert torch.equal(a.isnan(), b.isnan()) and torch.equal(a.nan_to_num(), b.nan_to_num())


@pytest.mark.parametrize("K", [16, 144, 1040, 1392, 2064, 4224, 6016, 8192, 12160, 16384])
@pytest.mark.parametrize("M,N,layout", [(1, 48, None), (3, 1040, "operand"), (8, 4112, None), (13, 3072, "operand"), (48, 208, None), (125, 1040, "operand")])
@pytest.mark.parametrize("source", ["rows", "scalar"])
def test_linear(dev, monkeypatch, source, M, N, layout, K):
    from phyai_amd import ops

    if layout and K % 128:
        pytest.skip("operand order needs whole K steps")
    x = seeded((M, K), K + M).to(dev)
    if K > 1000 and M > 1:
        x[1, K - 3] = float("inf" if K % 32 else "nan")
    w, ws = ops.fp8_weight_quant(seeded((N, K), N + K, 0.02).to(dev))
    bias, res, gate = seeded((N,), 7).to(dev), seeded((M, N), 8).to(dev), seeded((1, N), 9).to(dev)
    if source == "scalar":
        import phyai_amd.linear as L

        L.init()
        try:
            lin = L.ColumnParallelLinear(K, N, bias=True, params_dtype=torch.bfloat16, 
                                         spec=L.Fp8Spec(granularity=L.Granularity.PER_TENSOR, operand_order=layout is not None))
            lin.weight.data.copy_(w)
            lin.weight_scale.data.fill_(0.01)
            lin.input_scale.data.fill_(0.0357)
            lin.bias.data.copy_(bias)
            lin.post_load()
            _same(lin(x)[0], _two_launches(monkeypatch, lambda: lin(x)[0]))
        finally:
            L._reset_for_test()
        return
    if layout:
        w = ops.fp8_weight_to_operand_order(w)
    call = lambda **kw: ops.fp8_linear(x, w, ws, bias, weight_layout=layout, **kw)
    _same(call(), _two_launches(monkeypatch, call))
    _same(call(residual=res, gate=gate), _two_launches(monkeypatch, lambda: call(residual=res, gate=gate)))


@pytest.mark.parametrize("H,I", [(1040, 1392), (512, 12032), (560, 6016)])
@pytest.mark.parametrize("M", [1, 6, 33])
@pytest.mark.parametrize("epi", ["geglu_tanh", "swiglu", "gelu"])
def test_mlp_hands_the_maxima_on(dev, monkeypatch, M, H, I, epi):
    from phyai_amd import ops

    n1 = I if epi == "gelu" else 2 * I
    w1, s1 = ops.fp8_weight_quant(seeded((n1, H), 1, 0.02).to(dev))
    w2, s2 = ops.fp8_weight_quant(seeded((H, I), 2, 0.02).to(dev))
    x = seeded((M, H), 3).to(dev)
    call = lambda: ops.fp8_mlp(x, w1, s1, None, w2, s2, None, epilogue=epi)
    _same(call(), _two_launches(monkeypatch, call))


@pytest.mark.parametrize("scale", [16.0 / 448.0, 0.25, 3.0e-3, 1e-39, 7.0, float("inf")])
def test_static_quantizer_equals_the_division(dev, scale):
    from phyai_amd import ops

    x = torch.arange(65536, dtype=torch.int32).to(torch.int16).view(torch.bfloat16).reshape(64, 1024)   # every bf16 value
    s = torch.tensor([scale])
    got = ops.fp8_quant_static(x.to(dev), s.to(dev)).view(torch.uint8).cpu()
    q = (x.float() / s).clamp(-448.0, 448.0)
    want = q.to(torch.float8_e4m3fn).view(torch.uint8)
    nan = q.isnan()
    assert torch.equal(got[~nan], want[~nan]) and bool(((got[nan] & 0x7F) == 0x7F).all())


def test_weight_quantizer_equals_the_division(dev):
    from phyai_amd import ops

    w = (seeded((512, 2048), 5) * torch.logspace(-6, 3, 512)[:, None]).to(torch.bfloat16)
    q, s = ops.fp8_weight_quant(w.to(dev))
    want_s = w.float().abs().amax(1) / 448.0
    assert torch.equal(s.cpu(), want_s)
    assert torch.equal(q.view(torch.uint8).cpu(), (w.float() / want_s[:, None]).clamp(-448, 448).to(torch.float8_e4m3fn).view(torch.uint8))


@pytest.mark.parametrize("N,K", [(16, 128), (48, 1024), (1040, 1152), (32, 2176), (64, 8192), (48, 8320), (16, 16384)])
def test_weights_relaid_in_place(dev, N, K):
    from phyai_amd import ops

    w = torch.randint(0, 256, (N, K), dtype=torch.uint8, generator=torch.Generator().manual_seed(N + K)).to(dev)
    want = ops.fp8_weight_to_operand_order(w.view(torch.float8_e4m3fn)).view(torch.uint8)
    assert ops._native().relay_weight(w, False) is True
    assert torch.equal(w, want)
