"""The package's Python side against programs that replace, hook or share its parts, and against threads: everything
here runs without a GPU (tests/test_gpu_host_replaced.py holds what needs kernels)."""

from __future__ import annotations

import threading
import time
import weakref

import pytest
import torch
import torch.nn as nn

import phyai_amd.linear as L
from phyai_amd import _lib, ops
from phyai_amd.mlp import DenseMLP
from phyai_amd.norm import GemmaRMSNorm
from phyai_amd.quant import Fp8Spec, Granularity


@pytest.fixture(autouse=True)
def _dispatcher():
    L.init()
    yield
    L._reset_for_test()


def _bf16_linear(**kw):
    lin = L.ColumnParallelLinear(32, 16, params_dtype=torch.bfloat16, device="cpu", **kw)
    nn.init.normal_(lin.weight, std=0.1)
    return lin


def test_two_threads_bind_the_native_path_once(monkeypatch):
    opened, open_extension = [], _lib.open_host_extension

    def slowly():
        opened.append(threading.get_ident())
        time.sleep(0.2)
        return open_extension()

    monkeypatch.setattr(_lib, "open_host_extension", slowly)
    ops._host = None            # (the binding made here stays: it is as good as the one before)
    got, start = [], threading.Barrier(2)

    def call():
        start.wait()
        got.append(ops._native())

    threads = [threading.Thread(target=call) for _ in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert len(opened) == 1 and got[0] is got[1] is ops._host


def test_a_native_call_keeps_the_parameters_it_read():
    """Python code that runs in the middle of a call (a property of the spec, another thread while the GIL is released)
    may give the layer another weight: the call goes on with the tensors it read, and they live until it returns."""
    native, alive = ops._native(), []

    class Swapping(Fp8Spec):
        @property
        def granularity(self):
            if hasattr(self, "layer"):
                layer, self.__dict__["layer"] = self.layer, None
                if layer is not None:
                    layer.weight = nn.Parameter(torch.empty_like(layer.weight), requires_grad=False)
            return Granularity.PER_CHANNEL

        @granularity.setter
        def granularity(self, value):
            pass

    class Epilogue:   # looked up in a dictionary behind the layer's parameters
        def __hash__(self):
            alive.append(old() is not None)
            return 0

    lin = L.ColumnParallelLinear(128, 64, bias=False, params_dtype=torch.bfloat16, spec=Swapping(), device="cpu")
    old = weakref.ref(lin.weight)
    lin.spec.layer = lin
    assert native.layer_apply(lin, torch.zeros(4, 128, dtype=torch.bfloat16), None, Epilogue(), None, None) is None
    assert alive == [True]
    assert old() is None, "and no longer"


def test_a_replaced_module_call_is_called(monkeypatch):
    """torch.fx records calls of modules by replacing nn.Module.__call__ while it traces."""
    ops._native()
    lin = _bf16_linear()

    class Leaves(torch.fx.Tracer):
        def is_leaf_module(self, m, name):
            return isinstance(m, (L.ColumnParallelLinear, DenseMLP))

    class Model(nn.Module):
        def __init__(self):
            super().__init__()
            self.lin = lin
            self.mlp = DenseMLP(16, 32, params_dtype=torch.bfloat16)

        def forward(self, x):
            return self.mlp(self.lin(x)[0])

    graph = Leaves().trace(Model())
    assert [n.target for n in graph.nodes if n.op == "call_module"] == ["lin", "mlp"]
    seen, own = [], nn.Module.__call__
    monkeypatch.setattr(nn.Module, "__call__", lambda self, *a, **k: (seen.append(type(self)), own(self, *a, **k))[1])
    lin(torch.zeros(2, 32, dtype=torch.bfloat16))
    assert seen == [L.ColumnParallelLinear]


def test_parameters_that_are_plain_attributes():
    """A bias or weight replaced by a plain tensor (merged, shared, parametrized) is still the layer's bias or weight."""
    x = torch.randn(3, 32).to(torch.bfloat16)
    for skip in (False, True):
        lin = _bf16_linear(bias=True, skip_bias_add=skip)
        lin.bias.data.normal_()
        want = lin(x)
        bias = lin.bias.data
        del lin.bias
        lin.bias = bias
        got = lin(x)
        assert torch.equal(got[0], want[0]) and (got[1] is bias if skip else got[1] is None)
    spec = Fp8Spec(operand_order=True)
    lin = L.ColumnParallelLinear(128, 64, bias=False, params_dtype=torch.bfloat16, spec=spec, device="cpu")
    weight = lin.weight.data
    del lin.weight
    lin.weight = weight
    assert spec.to_operand_order_(lin) is False                       # a weight on the CPU is left alone
    norm = GemmaRMSNorm(32, device="cpu")
    weight = norm.weight.data
    del norm.weight
    norm.weight = weight
    for call in (norm, norm.forward_fp8):
        with pytest.raises(RuntimeError, match="must live on the GPU"):
            call(x)


def test_projections_that_are_not_registered_modules():
    """An MLP whose projection is shared with another owner and held as a plain attribute."""
    mlp = DenseMLP(32, 64, activation="gelu", gated=False, params_dtype=torch.bfloat16)
    for p in mlp.parameters():
        nn.init.normal_(p, std=0.1)
    x = torch.randn(3, 32).to(torch.bfloat16)
    want, shared = mlp(x), mlp.fc1
    del mlp.fc1
    mlp.__dict__["fc1"] = shared
    assert torch.equal(mlp(x), want)
