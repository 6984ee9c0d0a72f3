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
