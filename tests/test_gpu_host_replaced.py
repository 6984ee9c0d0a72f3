"""What a program may put in the place of a module, a hook, a method or a spec is honoured on the GPU's eager path as
well: the native calls (csrc/host_ext.cpp) stand for the package's own methods and for nothing else."""

from __future__ import annotations

import pytest
import torch

from conftest import seeded

pytestmark = pytest.mark.gpu

H, HEAD, HEADS, I, M = 256, 128, 2, 512, 40


@pytest.fixture
def linear():
    import phyai_amd.linear as L

    L.init()
    yield L
    L._reset_for_test()


def _fill(lin, seed):
    if hasattr(lin, "input_scale"):
        lin.weight.data.copy_(seeded(tuple(lin.weight.shape), seed, 4.0).to(lin.weight.device).to(torch.float8_e4m3fn))
        lin.input_scale.data.fill_(0.02)
        lin.post_load()
    else:
        lin.spec.quantize_weight_(lin, seeded(tuple(lin.weight.shape), seed, 0.02).to(lin.weight.device))
    return lin


@pytest.fixture
def expert(dev, linear):
    """(layer, call): call() is one pass of a small decoder layer in the fused form, its output."""
    from phyai_amd.runtime.expert_loop import ExpertLayer, ExpertLayerModulation

    layer = ExpertLayer(H, HEAD, HEADS, 1, I, H)
    for j, lin in enumerate((layer.qkv_proj, layer.o_proj, layer.mlp.gate_up_proj, layer.mlp.down_proj)):
        _fill(lin, 10 + j)
    mod = ExpertLayerModulation(seeded((1, 3 * H), 20, 0.1).to(dev), seeded((1, 3 * H), 21, 0.1).to(dev))
    x = seeded((M, H), 22).to(dev)
    return layer, lambda: layer(x, lambda fused, index: fused[:, :HEAD * HEADS], 0, mod)


def test_hooks_of_qkv_proj_run(expert):
    layer, call = expert
    want, seen = call(), []
    handle = layer.qkv_proj.register_forward_hook(lambda mod, args, out: seen.append("after"))
    before = layer.qkv_proj.register_forward_pre_hook(lambda mod, args: seen.append("before"))
    assert torch.equal(call(), want) and seen == ["before", "after"]
    handle.remove()
    before.remove()
    assert torch.equal(call(), want) and len(seen) == 2


@pytest.mark.parametrize("what", ["instance", "class", "wrapper", "not a registered module"])
def test_a_replaced_qkv_proj_is_called(expert, what):
    layer, call = expert
    want, own, seen = call(), layer.qkv_proj, []
    if what == "instance":
        forward = own.forward
        own.forward = lambda x: (seen.append(1), forward(x))[1]
    elif what == "class":
        class Watched(type(own)):
            def forward(self, x):
                seen.append(1)
                return super().forward(x)

        own.__class__ = Watched
    else:
        class Wrapper(torch.nn.Module):
            def __init__(self):
                super().__init__()
                self.inner = own

            def forward(self, x):
                seen.append(1)
                return self.inner(x)

        wrapper = Wrapper()
        if what == "wrapper":
            layer.qkv_proj = wrapper
        else:
            del layer.qkv_proj
            layer.__dict__["qkv_proj"] = wrapper
    assert torch.equal(call(), want) and seen == [1]


@pytest.mark.parametrize("name,method", [("input_layernorm", "forward_fp8"), ("post_attention_layernorm", "forward_fp8"),
                                         ("o_proj", "forward_addcmul"), ("mlp.gate_up_proj", "forward_fused"),
                                         ("mlp.down_proj", "forward_addcmul")])
def test_replaced_methods_of_the_other_parts_are_called(expert, name, method):
    layer, call = expert
    want, seen = call(), []
    part = layer.get_submodule(name)
    own = getattr(part, method)
    setattr(part, method, lambda *a, **k: (seen.append(1), own(*a, **k))[1])
    assert torch.equal(call(), want) and seen == [1]


def test_an_overridden_activation_quantizer_is_called(dev, linear):
    """Static scales: the layer's spec makes the codes (the reference's kernels call it, linear/backends/torch.py:132)."""
    L = linear

    class Halved(L.Fp8Spec):
        def quantize_activation(self, x, layer):
            return super().quantize_activation(x * 0.5, layer)

    def made(spec):
        return _fill(L.ColumnParallelLinear(H, 256, bias=False, params_dtype=torch.bfloat16, spec=spec), 30)

    x = seeded((M, H), 31).to(dev)
    plain, halved = made(L.Fp8Spec(granularity=L.Granularity.PER_TENSOR)), made(Halved(granularity=L.Granularity.PER_TENSOR))
    want = plain(x * 0.5)[0]
    assert not torch.equal(plain(x)[0], want)
    assert torch.equal(halved(x)[0], want)
    patched = made(L.Fp8Spec(granularity=L.Granularity.PER_TENSOR))
    own = patched.spec.quantize_activation
    patched.spec.quantize_activation = lambda x, layer: own(x * 0.5, layer)
    assert torch.equal(patched(x)[0], want)


@pytest.mark.parametrize("where", ["class", "instance"])
def test_an_instrumented_kernel_is_called(dev, linear, monkeypatch, where):
    from phyai_amd.linear.dispatch import get_linear_dispatcher
    from phyai_amd.linear.kernels import HipFp8Kernel

    lin = _fill(linear.ColumnParallelLinear(H, 256, bias=False, params_dtype=torch.bfloat16, spec=linear.Fp8Spec()), 40)
    x, seen = seeded((M, H), 41).to(dev), []
    want = lin(x)[0]
    if where == "class":
        own = HipFp8Kernel.apply
        monkeypatch.setattr(HipFp8Kernel, "apply", lambda self, *a, **k: (seen.append(1), own(self, *a, **k))[1])
    else:
        kernel = next(k for k in get_linear_dispatcher()._cache.values() if type(k) is HipFp8Kernel)
        own = kernel.apply
        monkeypatch.setattr(kernel, "apply", lambda *a, **k: (seen.append(1), own(*a, **k))[1], raising=False)
    assert torch.equal(lin(x)[0], want) and seen == [1]


@pytest.mark.parametrize("gated,which", [(True, "gate_up_proj"), (True, "down_proj"), (False, "fc1")])
def test_a_projection_that_refuses_fused_epilogues_gets_none(dev, linear, gated, which):
    """supports_fused_epilogue is the question that DenseMLP and forward_addcmul ask; an override answers it."""
    from phyai_amd.mlp import DenseMLP

    mlp = DenseMLP(H, I, activation="gelu_tanh", gated=gated, params_dtype=torch.bfloat16, spec_in=linear.Fp8Spec(), spec_out=linear.Fp8Spec())
    for j, name in enumerate(("gate_up_proj", "down_proj") if gated else ("fc1", "fc2")):
        _fill(getattr(mlp, name), 50 + j)
    x, gate = seeded((M, H), 52).to(dev), seeded((1, H), 53).to(dev)
    want, asked = mlp(x), []
    part = getattr(mlp, which)
    part.supports_fused_epilogue = lambda x: bool(asked.append(1))
    got = mlp(x)
    assert asked and torch.allclose(got.float(), want.float(), rtol=2e-2, atol=1e-2 * want.float().abs().max().item())
    if which == "down_proj":
        h, asked[:] = part(mlp.gate_up_proj.forward_fused(x, "geglu_tanh"))[0], []
        got = part.forward_addcmul(mlp.gate_up_proj.forward_fused(x, "geglu_tanh"), x, gate)
        assert asked and torch.equal(got, torch.addcmul(x, h, gate))
