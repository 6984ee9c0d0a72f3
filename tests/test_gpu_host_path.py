"""The eager call path in C++ (csrc/host_ext.cpp) against the Python one: same kernels, so equal bits, for
every form it takes; forms it declines still come out right and bad arguments still raise."""

from __future__ import annotations

import pytest
import torch

from conftest import seeded

pytestmark = pytest.mark.gpu


class _Declines:
    def __getattr__(self, name):
        return lambda *a: None


def _both(monkeypatch, call):
    from phyai_amd import ops

    ops._native()
    fast = call()
    with monkeypatch.context() as m:
        m.setattr(ops, "_host", _Declines())
        slow = call()
    flat = (lambda r: [t for t in r if t is not None] if isinstance(r, tuple) else [r])
    assert len(flat(fast)) == len(flat(slow))
    for a, b in zip(flat(fast), flat(slow)):
        assert a.shape == b.shape and a.dtype == b.dtype and torch.equal(a.view(torch.uint8), b.view(torch.uint8))


@pytest.mark.parametrize("lead,strided", [((1,), False), ((50,), True), ((3, 7), False), ((300,), False)])
@pytest.mark.parametrize("scheme", ["per_channel", "per_tensor"])
def test_layer_call(dev, monkeypatch, lead, strided, scheme):
    import phyai_amd.linear as L

    L.init()
    try:
        n, k = 272, 256
        lin = L.ColumnParallelLinear(k, n, bias=True, params_dtype=torch.bfloat16,
                                     spec=L.Fp8Spec(granularity=L.Granularity[scheme.upper()]))
        lin.weight.data.copy_(seeded((n, k), 3, 4.0).to(dev).to(torch.float8_e4m3fn))
        lin.bias.data.copy_(seeded((n,), 4))
        if scheme == "per_tensor":
            lin.input_scale.data.fill_(0.02)
        lin.post_load()
        x = seeded((*lead, 2 * k if strided else k), 5).to(dev)[..., :k]
        _both(monkeypatch, lambda: lin(x)[0])
        res, gate = seeded((*lead, n), 6).to(dev), seeded((1, n), 7).to(dev)
        _both(monkeypatch, lambda: lin.forward_addcmul(x, res, gate))
    finally:
        L._reset_for_test()


def test_ops_mlp_and_norms(dev, monkeypatch):
    from phyai_amd import ops

    M, H, I = 50, 256, 512
    x, mod = seeded((M, H), 1).to(dev), seeded((2, 3 * H), 2, 0.1).to(dev)
    w1, s1 = ops.fp8_weight_quant(seeded((2 * I, H), 3, 0.02).to(dev))
    w2, s2 = ops.fp8_weight_quant(seeded((H, I), 4, 0.02).to(dev))
    out = torch.empty(M, H, dtype=torch.bfloat16, device=dev)
    xq, xs = ops.fp8_quant_rowwise(x)
    for call in (lambda: ops.fp8_quant_rowwise(x), lambda: ops.rmsnorm(x, mod[0, :H]), lambda: ops.rmsnorm_fp8(x, mod[0, :H], want_out=True),
                 lambda: ops.adarmsnorm(x, mod), lambda: ops.adarmsnorm_fp8(x, mod),
                 lambda: ops.fp8_gemm(xq, xs, w1, s1, epilogue="geglu_tanh"),
                 lambda: ops.fp8_mlp(x, w1, s1, None, w2, s2, None, epilogue="swiglu", residual=x, gate=mod[:, :H].contiguous()),
                 lambda: ops.fp8_linear(x, w1, s1, out=torch.empty(M, 2 * I, dtype=torch.bfloat16, device=dev))):
        _both(monkeypatch, call)
    assert ops.fp8_mlp(x, w1, s1, None, w2, s2, None, epilogue="swiglu", out=out) is out
    assert ops.fp8_linear(x[:0], w1, s1).shape == (0, 2 * I)                       # declined forms
    _both(monkeypatch, lambda: ops.fp8_linear(seeded((M, H + 4), 8).to(dev)[:, 4:], w1, s1))
    with pytest.raises(RuntimeError, match="fp8_linear: weight K="):
        ops.fp8_linear(x, w2, s2)
    with pytest.raises(RuntimeError, match="residual and gate go together"):
        ops.fp8_linear(x, w1, s1, residual=x)
