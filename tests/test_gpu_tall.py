"""Tall tiles (csrc/gemm_tall.hip): 144 .. 256 rows x 256 columns, weights in operand order.  Their sums run along K in the
order of every other unsplit tile shape and the epilogue does the same arithmetic, so the bits are those of the staged 192 x 128
tiles, which the other tests hold against the oracle; one case is held against it here."""

from __future__ import annotations

import pytest
import torch

from conftest import seeded

pytestmark = pytest.mark.gpu
ROWS = list(range(144, 257, 16))


def _bits(t):
    return t.view(torch.int16)


def _operands(dev, M, N, K, gated, seed=0):
    from phyai_amd import ops

    xq, xs = ops.fp8_quant_rowwise(seeded((M, K), M + K + seed).to(dev))
    wq, ws = ops.fp8_weight_quant(seeded((N, K), N + K + seed, 0.05).to(dev))
    return xq, xs, wq, ws, ops.fp8_weight_to_operand_order(wq, gated=gated)


def _both(monkeypatch, rows, call, M, N, K, epi=None):
    """The call with tall tiles of that many rows, and with staged 192 x 128 tiles."""
    from phyai_amd import ops

    layout = "operand_gated" if epi and epi.startswith(("geglu", "swiglu")) else "operand"
    monkeypatch.setenv("PHYAI_FP8_BIG", "192")
    want = call(layout)
    monkeypatch.setenv("PHYAI_FP8_TALL", str(rows))
    plan = ops.describe_plan(M, N, K, epi, weight_layout=layout)
    assert plan.startswith(f"tile {rows}x256 ") and plan.endswith("weights in registers, ring of 4"), plan
    got = call(layout)
    monkeypatch.delenv("PHYAI_FP8_TALL")
    return got, want


# one trip round the ring of stages (K = 512) and several, one to three stages of 128 beyond; one row, a row short of a tile, a row over, many; columns that end in
# the first, second and last 16 of a tile; gated: half of them, in steps of 16
@pytest.mark.parametrize("rows", ROWS)
@pytest.mark.parametrize("epi", [None, "gelu", "gelu_tanh", "geglu_tanh", "geglu_erf", "swiglu"])
def test_edges_of_tiles(dev, monkeypatch, rows, epi):
    from phyai_amd import ops

    gated = bool(epi) and epi.startswith(("geglu", "swiglu"))
    for M, N, K in ((rows - 1, 272, 512), (rows + 1, 1056, 1024), (129, 2048, 1536), (2 * rows + 17, 288, 2048), (3 * rows, 512, 512),
                    (rows + 33, 288, 640), (rows, 544, 768), (rows + 1, 288, 896), (2 * rows, 288, 1152), (rows - 7, 288, 1664), (rows + 2, 288, 1408)):
        N = (N + 31) // 32 * 32 if gated else N
        xq, xs, wq, ws, wo = _operands(dev, M, N, K, gated)
        bias = seeded((N + 1,), N, 0.1).to(dev)
        for b in (None, bias[:N], bias[1:]):        # rides into LDS as words, or value by value
            got, want = _both(monkeypatch, rows, lambda lay: ops.fp8_gemm(xq, xs, wo, ws, b, epilogue=epi, weight_layout=lay), M, N, K, epi)
            assert torch.equal(_bits(got), _bits(want)), (M, N, K, b is None)


@pytest.mark.parametrize("rows", ROWS)
@pytest.mark.parametrize("epi", [None, "geglu_tanh"])
def test_several_tiles_per_workgroup(dev, monkeypatch, rows, epi):
    """More tiles than workgroups (256): openings under epilogues, both halves of the constants' place, the order of the tiles
    with and without columns beyond the last eight, tiles that open on every stage of the ring; every pass gives the same."""
    from phyai_amd import ops

    for M, N, K in ((5 * rows + 40, 16384 + 32, 512), (40 * rows - 5, 2048, 1024), (17 * rows, 5 * 1024, 512),
                    (41 * rows + 1, 4096, 640), (40 * rows - 5, 4096 + 32, 768), (36 * rows, 4096, 896), (35 * rows, 2048, 1664)):
        xq, xs, wq, ws, wo = _operands(dev, M, N, K, epi is not None)
        for _ in range(2):
            got, want = _both(monkeypatch, rows, lambda lay: ops.fp8_gemm(xq, xs, wo, ws, epilogue=epi, weight_layout=lay), M, N, K, epi)
            assert torch.equal(_bits(got), _bits(want)), (M, N, K)


# 257 to 600 tiles: a workgroup takes two or three, the constants of the second ride along under the epilogue of the first
MANY = [(144, 40, 2048, 512), (208, 17, 4096 + 32, 768), (256, 35, 2048, 640)]


@pytest.mark.parametrize("rows,blocks,N,K", MANY)
@pytest.mark.parametrize("epi", [None, "gelu", "gelu_tanh", "geglu_tanh", "geglu_erf", "swiglu"])
@pytest.mark.parametrize("one_scale", [False, True])
def test_bias_and_scales_of_several_tiles(dev, monkeypatch, rows, blocks, N, K, epi, one_scale):
    """Bias as words and value by value (an odd offset), row scales or one for all rows, every activation, over several tiles a
    workgroup."""
    from phyai_amd import ops

    M, gated = blocks * rows - 7, bool(epi) and epi.startswith(("geglu", "swiglu"))
    N = 2 * N if gated else N
    xq, xs, wq, ws, wo = _operands(dev, M, N, K, gated)
    xs = xs.flatten()[:1].contiguous() if one_scale else xs
    bias = seeded((N + 1,), N, 0.1).to(dev)
    for b in (bias[:N], bias[1:]):
        got, want = _both(monkeypatch, rows, lambda lay: ops.fp8_gemm(xq, xs, wo, ws, b, epilogue=epi, weight_layout=lay), M, N, K, epi)
        assert torch.equal(_bits(got), _bits(want))


@pytest.mark.parametrize("rows,blocks,N,K", MANY)
@pytest.mark.parametrize("gates", [1, 3, 0])
def test_gated_residual_of_several_tiles(dev, monkeypatch, rows, blocks, N, K, gates):
    """... with one gate row, with groups of token rows that end inside tiles, with a gate row each; into its own place too, and
    out of rows that lie further apart than the output's."""
    from phyai_amd import _lib, ops

    M = 3 * ((blocks * rows - 7) // 3)
    xq, xs, wq, ws, wo = _operands(dev, M, N, K, False)
    bias = seeded((N + 1,), N, 0.1).to(dev)
    gate = seeded((gates or M, N), 4, 0.3).to(dev)
    wide = seeded((M, N + 40), 3).to(dev)
    res = wide[:, 8:8 + N].contiguous()
    scratch = torch.empty(1 << 20, dtype=torch.uint8, device=dev)
    for b in (bias[:N], bias[1:]):
        def spread(lay):
            out = torch.empty(M, N, dtype=torch.bfloat16, device=dev)
            _lib.check(_lib.load().phyai_fp8_gemm_addcmul(
                xq.data_ptr(), xs.data_ptr(), 0, wo.data_ptr(), ws.data_ptr(), b.data_ptr(), wide[:, 8:].data_ptr(), N + 40, gate.data_ptr(), N,
                gate.shape[0], out.data_ptr(), N, M, N, K, 0x200, scratch.data_ptr(), scratch.numel(), torch.cuda.current_stream().cuda_stream), "addcmul")
            return out

        def in_place(lay):
            out = res.clone()
            return ops.fp8_gemm(xq, xs, wo, ws, b, residual=out, gate=gate, out=out, weight_layout=lay)

        plain = lambda lay: ops.fp8_gemm(xq, xs, wo, ws, b, residual=res, gate=gate, weight_layout=lay)
        got, want = _both(monkeypatch, rows, plain, M, N, K)
        assert torch.equal(_bits(got), _bits(want))
        for other in (in_place, spread):
            again, _ = _both(monkeypatch, rows, other, M, N, K)
            assert torch.equal(_bits(again), _bits(want)), other.__name__


@pytest.mark.parametrize("epi", [None, "gelu", "geglu_tanh"])
def test_operands_that_are_not_finite(dev, monkeypatch, epi):
    """A NaN code or scale reaches its own rows and columns, an infinite scale or bias too, and nothing else changes."""
    from phyai_amd import ops

    rows, gated = 144, epi == "geglu_tanh"
    M, N, K = 40 * rows - 5, 4096 if gated else 2048, 512
    xq, xs, wq, ws, _ = _operands(dev, M, N, K, gated)
    half = N // 2 if gated else N
    bias = seeded((N,), N, 0.1).to(dev)
    xs = xs.abs() + 0.01
    call = lambda lay: ops.fp8_gemm(xq, xs, wo, ws, bias, epilogue=epi, weight_layout=lay)
    wo = ops.fp8_weight_to_operand_order(wq, gated=gated)
    clean = call("operand_gated" if gated else "operand")
    x8, w8 = xq.view(torch.uint8), wq.view(torch.uint8)
    x8[7, 3], x8[M - 1, K - 1], w8[33, 5] = 0x7F, 0xFF, 0x7F
    xs.view(-1)[200] = float("inf")
    xs.view(-1)[3 * rows] = float("nan")
    ws[half - 1], bias[300] = float("nan"), float("inf")
    wo = ops.fp8_weight_to_operand_order(wq, gated=gated)
    got, want = _both(monkeypatch, rows, call, M, N, K, epi)
    nan = torch.isnan(want)
    assert torch.equal(torch.isnan(got), nan) and torch.equal(_bits(got)[~nan], _bits(want)[~nan])
    assert bool(nan[[7, M - 1, 3 * rows]].all()) and bool(nan[:, [33, half - 1]].all())
    keep_r, keep_c = torch.ones(M, dtype=torch.bool, device=dev), torch.ones(half, dtype=torch.bool, device=dev)
    keep_r[[7, 200, 3 * rows, M - 1]] = False
    keep_c[[33, 300, half - 1]] = False
    assert torch.equal(_bits(got[keep_r][:, keep_c]), _bits(clean[keep_r][:, keep_c]))


@pytest.mark.parametrize("rows", ROWS)
@pytest.mark.parametrize("gates", [1, 4, 0])
def test_gated_residual(dev, monkeypatch, rows, gates):
    """One gate row for all token rows, for a quarter of them each, for each."""
    from phyai_amd import ops

    M, N, K = 2 * rows + 32, 1040, 1024
    xq, xs, wq, ws, wo = _operands(dev, M, N, K, False)
    res, gate = seeded((M, N), 3).to(dev), seeded((gates or M, N), 4, 0.3).to(dev)
    got, want = _both(monkeypatch, rows, lambda lay: ops.fp8_gemm(xq, xs, wo, ws, residual=res, gate=gate, weight_layout=lay), M, N, K)
    assert torch.equal(_bits(got), _bits(want))


def _into(out, row_stride, xq, xs, w, ws, M, N, K):
    """phyai_fp8_gemm on operand-order weights, rows of the result `row_stride` elements apart."""
    from phyai_amd import _lib

    _lib.check(_lib.load().phyai_fp8_gemm(xq.data_ptr(), xs.data_ptr(), 0, w.data_ptr(), ws.data_ptr(), None, out.data_ptr(), row_stride, M, N, K,
                                          0x200, None, 0, torch.cuda.current_stream().cuda_stream), "gemm")


@pytest.mark.parametrize("rows", [144, 208, 256])
def test_against_the_oracle_and_into_a_wider_matrix(dev, monkeypatch, rows):
    """fp32 sums of exact products, rounded once: within half a bf16 step (2^-8 of the value at
    most: 8 significant bits) and the sums' own rounding of the fp64 result.  The
    output is a part of a wider matrix: nothing beside it, and no row past it, is written."""
    M, N, K = 3 * rows + 5, 784, 1024
    xq, xs, _, ws, wo = _operands(dev, M, N, K, False)
    wq = _operands(dev, M, N, K, False)[2]
    wide = torch.full((M + 300, N + 64), 7.0, dtype=torch.bfloat16, device=dev)
    monkeypatch.setenv("PHYAI_FP8_BIG", "192")
    monkeypatch.setenv("PHYAI_FP8_TALL", str(rows))
    _into(wide[:, 16:], N + 64, xq, xs, wo, ws, M, N, K)
    exact = (xq.cpu().double() @ wq.cpu().double().T) * xs.cpu().double().view(-1, 1) * ws.cpu().double().view(1, -1)
    got = wide[:M, 16:16 + N].cpu().double()
    assert ((got - exact).abs() <= exact.abs() * 2.0 ** -8 + exact.abs().max() * K * 2.0 ** -24).all()
    wide[:M, 16:16 + N] = 7.0
    assert bool((wide == 7.0).all())


def test_rows_of_output_too_far_apart(dev, monkeypatch):
    """The epilogue's offsets are 32-bit: from 2^21 elements between rows on another shape does the work, with the same bits."""
    from phyai_amd import ops

    M, N, K, far = 150, 256, 512, 1 << 21
    xq, xs, _, ws, wo = _operands(dev, M, N, K, False)
    monkeypatch.setenv("PHYAI_FP8_BIG", "192")
    want = ops.fp8_gemm(xq, xs, wo, ws, weight_layout="operand")
    monkeypatch.setenv("PHYAI_FP8_TALL", "208")
    for stride in (far - 8, far):
        room = torch.empty(M * stride, dtype=torch.bfloat16, device=dev)
        _into(room, stride, xq, xs, wo, ws, M, N, K)
        assert torch.equal(_bits(torch.as_strided(room, (M, N), (stride, 1)).contiguous()), _bits(want))


def test_planner_takes_tall_tiles_of_the_height_that_fills_the_rounds():
    from phyai_amd import ops

    d = ops.describe_linear_plan
    R4 = "weights in registers, ring of 4"
    for (m, n, k, epi), rows in {(816, 32768, 2048, "geglu_tanh"): 208, (4800, 2048, 8192, None): 160, (4800, 2048, 2048, None): 160}.items():
        plan = d(m, n, k, epi, weight_layout="operand_gated" if epi else "operand")
        assert plan.startswith(f"quantizer + tile {rows}x256 ") and plan.endswith(R4), plan
    assert "x256" not in d(816, 2048, 2048, weight_layout="operand")                 # 32 tiles
    assert R4 not in d(4800, 2048, 8192) and R4 not in d(4800, 2048, 8192 + 32, weight_layout="operand")
    assert d(5000, 1280, 5120, weight_layout="operand").endswith(R4) and d(4800, 2048, 8192 + 128, weight_layout="operand").endswith(R4)
