"""Epilogue of the pipelined tile kernels (csrc/gemm_big.hip): row scales, weight scales and bias reach it through LDS,
the gated residual is added where the tile leaves row by row."""

from __future__ import annotations

import pytest
import torch

from conftest import seeded
from oracle import ref

pytestmark = pytest.mark.gpu

TILES = ["256", "224", "192", "128", "128/2", "96", "12864"]
SPLIT = "128x2"   # 128 x 128 tiles, K split in two


def _force(monkeypatch, tile):
    t, _, depth = tile.partition("/")
    if tile == SPLIT:
        t = "128"
        monkeypatch.setenv("PHYAI_FP8_BIG_SPLITS", "2")
    monkeypatch.setenv("PHYAI_FP8_BIG", t)
    if depth:
        monkeypatch.setenv("PHYAI_FP8_BIG_DEPTH", depth)


def _codes(dev, m, k, seed):
    from phyai_amd import ops

    return ops.fp8_quant_rowwise(seeded((m, k), seed).to(dev))


@pytest.mark.parametrize("layout", [None, "operand"])
@pytest.mark.parametrize("tile", TILES + [SPLIT])
@pytest.mark.parametrize("M,N,K,epi", [(97, 144, 512, None), (225, 272, 640, "gelu"), (257, 544, 1024, "geglu_tanh"), (130, 160, 1040, "swiglu"),
                                       (257, 528, 1024, None)])
def test_constants_from_any_address(dev, monkeypatch, tile, layout, M, N, K, epi):
    """Bias in whole words, at an odd 16-bit address (filled in by hand) and absent; tiles that end past M and N; one scale
    for all rows.  Every form against the values it stands for: the address changes no bit, no bias is a bias of zeros, one
    scale is a row of equal scales."""
    from phyai_amd import ops

    gated = epi in ("geglu_tanh", "swiglu")
    if tile in ("96", "12864") and gated or layout and K % 128 or tile == SPLIT and K != 1024:
        pytest.skip("no such kernel")
    assert not gated or N % 32 == 0 and N // 2 > 64     # more than one tile column of gate | up pairs
    _force(monkeypatch, tile)
    lay = None if layout is None else ("operand_gated" if gated else "operand")
    xq, xs = _codes(dev, M, K, M + N)
    wq, ws = ops.fp8_weight_quant(seeded((N, K), M + K, 0.02).to(dev))
    if layout:
        wq = ops.fp8_weight_to_operand_order(wq, gated=gated)
    room = seeded((N + 8,), 7, 0.5).to(dev)
    run = lambda bias, scale=xs: ops.fp8_gemm(xq, scale, wq, ws, bias, epilogue=epi, weight_layout=lay).view(torch.int16)
    plan = ops.describe_plan(M, N, K, epi, weight_layout=lay)
    assert plan.startswith("tile ") and ("splits=2" in plan) == (tile == SPLIT)
    if layout and not gated and K == 1024 and tile in ("128", SPLIT):   # (K / 2 is no trip round the ring of eight)
        assert plan.endswith("ring of 8") == (tile == "128")
    odd = room[1:N + 1]
    assert odd.data_ptr() % 4 == 2
    assert torch.equal(run(odd), run(odd.clone()))
    assert torch.equal(run(None), run(torch.zeros_like(odd)))
    one = torch.full((1,), 0.03, device=dev)
    assert torch.equal(run(room[:N], one), run(room[:N], one.expand(M).contiguous()))
    # rows and columns keep their own constants: a scale or a bias value that differs in one place changes that place only
    base = run(room[:N])
    xs2, ws2, b2 = xs.clone().view(-1), ws.clone().view(-1), room[:N].clone()
    xs2[M - 1] *= 2
    got = ops.fp8_gemm(xq, xs2.view_as(xs), wq, ws, b2, epilogue=epi, weight_layout=lay).view(torch.int16)
    assert torch.equal(got[:M - 1], base[:M - 1]) and not torch.equal(got[M - 1], base[M - 1])
    b2[N - 1] += 4
    got, col = run(b2), (N // 2 - 1 if gated else N - 1)
    keep = torch.arange(base.shape[1], device=dev) != col
    assert torch.equal(got[:, keep], base[:, keep]) and not torch.equal(got[:, col], base[:, col])
    ws2[0] *= 2
    got = ops.fp8_gemm(xq, xs, wq, ws2.view_as(ws), room[:N], epilogue=epi, weight_layout=lay).view(torch.int16)
    assert torch.equal(got[:, 1:], base[:, 1:]) and not torch.equal(got[:, 0], base[:, 0])


@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("M,N,K,groups", [(96, 144, 512, 1), (230, 272, 640, 5), (387, 528, 1024, 387)])
def test_residual_row_by_row(dev, monkeypatch, tile, M, N, K, groups):
    """out = residual + bf16(linear) * gate with strided residual rows, one gate row for all, for a few or for each token
    row, and in place: torch.addcmul on the kernel's own linear output, bit for bit."""
    from phyai_amd import ops

    _force(monkeypatch, tile)
    xq, xs = _codes(dev, M, K, M)
    wq, ws = ops.fp8_weight_quant(seeded((N, K), K, 0.02).to(dev))
    bias = seeded((N,), 3).to(dev)
    wide = seeded((M, N + 24), 4).to(dev)
    res, gate = wide[:, 8:8 + N], seeded((groups, N), 5, 0.5).to(dev)
    assert ops.describe_plan(M, N, K).startswith("tile ")
    y = ops.fp8_gemm(xq, xs, wq, ws, bias)
    want = ref.addcmul(res.cpu(), y.cpu(), gate.cpu().repeat_interleave(M // groups, 0))
    assert torch.equal(ops.fp8_gemm(xq, xs, wq, ws, bias, residual=res, gate=gate).cpu(), want)
    own = res.contiguous()
    ops.fp8_gemm(xq, xs, wq, ws, bias, residual=own, gate=gate, out=own)
    assert torch.equal(own.cpu(), want)
