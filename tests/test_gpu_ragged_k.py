"""K that is a multiple of 16 but not of the 128-byte K step in the pipelined tile kernel and the weight-streaming
kernel: the partial last step, in every tile shape, against the generic kernel bit for bit (same order of K) or on
exact integers.  Weight rows begin with NaN codes in places: a row's missing chunks must not read its neighbour."""

from __future__ import annotations

import pytest
import torch

from conftest import seeded

pytestmark = pytest.mark.gpu


def _operands(dev, M, N, K, seed):
    g = torch.Generator().manual_seed(seed)
    xq = torch.randint(-4, 5, (M, K), generator=g).float().to(torch.float8_e4m3fn).to(dev)
    w = torch.randint(-4, 5, (N, K), generator=g).float()
    xs = (2.0 ** torch.randint(-3, 3, (M,), generator=g).float()).to(dev)
    nan_rows = torch.arange(5, N, 37)
    w[nan_rows, :16] = float("nan")
    return xq, xs, w.to(torch.float8_e4m3fn).to(dev), torch.ones(N, device=dev), nan_rows


@pytest.mark.parametrize("K", [528, 640 + 112, 1168, 4304])
@pytest.mark.parametrize("tile", ["256", "224", "192", "128", "128/2", "12864", "96", "split"])
@pytest.mark.parametrize("M,N,epi", [(300, 528, None), (129, 272, "gelu"), (260, 288, "swiglu")])
def test_tile_kernel_equals_the_generic_one(dev, monkeypatch, tile, M, N, K, epi):
    from phyai_amd import ops

    if epi == "swiglu" and tile in ("12864", "96"):
        pytest.skip("plain epilogues only")
    xq, xs, w, ws, nan_rows = _operands(dev, M, N, K, seed=M + N + K)
    bias = seeded((N,), 5).to(dev)
    monkeypatch.setenv("PHYAI_FP8_TILE", "128,128,1")
    want = ops.fp8_gemm(xq, xs, w, ws, bias, epilogue=epi)
    monkeypatch.delenv("PHYAI_FP8_TILE")
    if tile == "split":
        if K < 1152:
            pytest.skip("a range per split must fill the ring")
        monkeypatch.setenv("PHYAI_FP8_BIG", "128")
        monkeypatch.setenv("PHYAI_FP8_BIG_SPLITS", "2")
    else:
        t, _, depth = tile.partition("/")
        monkeypatch.setenv("PHYAI_FP8_BIG", t)
        if depth:
            monkeypatch.setenv("PHYAI_FP8_BIG_DEPTH", depth)
    assert ops.describe_plan(M, N, K, epi).startswith("tile ")
    got = ops.fp8_gemm(xq, xs, w, ws, bias, epilogue=epi)
    assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.nan_to_num(), want.nan_to_num())
    assert bool(got.isnan().any()) and not bool(got.isnan().all())


@pytest.mark.parametrize("K", [272, 528, 1040, 4304, 16368])
@pytest.mark.parametrize("M,N,epi", [(1, 1040, None), (50, 272, None), (64, 544, "swiglu"), (70, 1040, None), (500, 1024, None)])
def test_weight_streaming_kernel_on_exact_integers(dev, M, N, K, epi):
    from phyai_amd import ops

    assert ops.describe_plan(M, N, K, epi).startswith("small-m ")
    xq, xs, w, ws, nan_rows = _operands(dev, M, N, K, seed=M + N + K + 1)
    got = ops.fp8_gemm(xq, xs, w, ws, epilogue=epi).float()
    y = (xq.float() @ w.float().T * xs[:, None]).to(torch.bfloat16).float()
    if epi:
        y = torch.nn.functional.silu(y[:, :N // 2]) * y[:, N // 2:]
    assert torch.equal(got.isnan(), y.isnan())
    if epi:
        assert (got - y).nan_to_num().abs().max() <= 1e-2 * y.nan_to_num().abs().max()
    else:
        assert torch.equal(got.nan_to_num(), y.nan_to_num())
