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
