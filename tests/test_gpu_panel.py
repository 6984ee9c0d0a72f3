"""Linears of more than 48 rows in one launch (csrc/gemm_panel.hip) against quantizer + GEMM, bit for bit: the edges of its
tiles and of its K, both orders of sums, both kinds of scale, rows that are not finite, scales at the ends of the range,
strided rows and outputs, a gated residual; and what it does not take over: an output inside its own rows, a call without a
workspace."""

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


def _weights(ops, n, k, dev, operand):
    wq, ws = ops.fp8_weight_quant(seeded((n, k), n + k, 0.02).to(dev))
    return (ops.fp8_weight_to_operand_order(wq), ws, "operand") if operand else (wq, ws, None)


# M, N, K, operand order, weight tiles per wavefront
SHAPES = [(49, 4016, 752, False, 1), (113, 8192, 256, True, 2), (129, 16, 128, True, 1), (144, 64, 1024, True, 1), (145, 2048, 896, True, 1), (512, 1024, 1024, True, 1), (8192, 16, 512, True, 1),
          (129, 3648, 256, True, 2), (400, 2560, 1024, True, 2), (1000, 1024, 512, True, 2), (4100, 112, 896, True, 2),
          (129, 80, 272, False, 1), (400, 1200, 752, False, 1), (131, 5392, 272, False, 1), (777, 960, 640, False, 1), (3000, 160, 528, False, 1)]


@pytest.mark.parametrize("scale", ["rows", 0.013, 1e-30, 3e38])
@pytest.mark.parametrize("M,N,K,operand,nt", SHAPES)
def test_one_launch_equals_two(dev, monkeypatch, M, N, K, operand, nt, scale):
    from phyai_amd import _lib, ops

    lib, st = _lib.load(), torch.cuda.current_stream().cuda_stream
    w, ws, layout = _weights(ops, N, K, dev, operand)
    assert ops.describe_linear_plan(M, N, K, weight_layout=layout).startswith(f"one launch: panel of 16 rows, nt={nt} ")
    rows = torch.empty(M, K + 40, dtype=torch.bfloat16, device=dev)
    rows[:, :K] = seeded((M, K), M + K).to(dev)
    rows[:, K:] = float("nan")                       # behind each row: nobody's
    rows[0, :K] = 0
    rows[M // 2, K - 1] = float("inf")
    rows[M - 1, 0] = float("nan")
    rows[5, :K] *= 2.0 ** 100
    bias, res, gate, one = seeded((N,), 5).to(dev), seeded((M, N), 8).to(dev), seeded((1, N), 9).to(dev), torch.zeros(1, device=dev)
    need = lib.phyai_fp8_linear_workspace_bytes(M, N, K, 0)
    flag = ops.FLAG_W_OPERAND_ORDER if operand else 0

    def call(residual):
        scratch = torch.full((need,), 0xAB, dtype=torch.uint8, device=dev)
        scratch[:16384] = 0
        out = torch.full((M, N + 24), 7.0, dtype=torch.bfloat16, device=dev)
        extra = (res.data_ptr(), N, gate.data_ptr(), N, 1)
        tail = (out.data_ptr(), N + 24, M, N, K, flag, scratch.data_ptr(), need, st)
        head = (rows.data_ptr(), K + 40)
        mid = (w.data_ptr(), ws.data_ptr(), bias.data_ptr())
        if scale != "rows":
            one.fill_(scale)
            rc = lib.phyai_fp8_linear_per_tensor(*head, one.data_ptr(), *mid, *(extra if residual else (None, 0, None, 0, 0)), *tail)
        elif residual:
            rc = lib.phyai_fp8_linear_addcmul(*head, *mid, *extra, *tail)
        else:
            rc = lib.phyai_fp8_linear(*head, *mid, *tail)
        _lib.check(rc, "linear")
        assert bool((out[:, N:] == 7.0).all())
        return out[:, :N], bool((scratch[16384:] == 0xAB).all())

    for residual in (False, True):
        got, one_launch = call(residual)
        want, other = _two_launches(monkeypatch, lambda: call(residual))
        assert one_launch and not other
        _same(got, want)


def test_an_output_inside_its_own_rows_takes_two_launches(dev):
    from phyai_amd import _lib, ops

    lib, M, K = _lib.load(), 400, 512
    w, ws, _ = _weights(ops, K, K, dev, True)
    x = seeded((M, K), 3).to(dev)
    want = ops.fp8_linear(x, w, ws, weight_layout="operand")
    need = lib.phyai_fp8_linear_workspace_bytes(M, K, K, 0)
    scratch = torch.zeros(need, dtype=torch.uint8, device=dev)
    tail = (M, K, K, ops.FLAG_W_OPERAND_ORDER, scratch.data_ptr(), need, torch.cuda.current_stream().cuda_stream)
    _lib.check(lib.phyai_fp8_linear(x.data_ptr(), K, w.data_ptr(), ws.data_ptr(), None, x.data_ptr(), K, *tail), "linear")
    assert torch.equal(x, want) and not bool((scratch == 0).all())


def test_a_call_without_a_workspace_stays_refused(dev):
    from phyai_amd import _lib, ops

    lib, M, K = _lib.load(), 400, 512
    w, ws, _ = _weights(ops, K, K, dev, True)
    x, out = seeded((M, K), 3).to(dev), torch.full((M, K), 7.0, dtype=torch.bfloat16, device=dev)
    rc = lib.phyai_fp8_linear(x.data_ptr(), K, w.data_ptr(), ws.data_ptr(), None, out.data_ptr(), K, M, K, K, ops.FLAG_W_OPERAND_ORDER, None, 0,
                              torch.cuda.current_stream().cuda_stream)
    assert rc == -3 and bool((out == 7.0).all())
