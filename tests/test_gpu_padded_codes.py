"""Codes that a linear stages for its own GEMM begin every row on a 128-byte line (csrc/launch.h, padded_row_bytes): the same
kernel on dense and on padded codes gives the same bits, and the workspace that the library asks for holds them."""

from __future__ import annotations

import pytest
import torch

from conftest import seeded

pytestmark = pytest.mark.gpu

KERNELS = {"256": "BIG=256", "224": "BIG=224", "192": "BIG=192", "128": "BIG=128", "128/2": "BIG=128 BIG_DEPTH=2", "96": "BIG=96",
           "12864": "BIG=12864", "split": "BIG=128 BIG_SPLITS=2", "generic": "TILE=128,128,1", "generic split": "TILE=64,128,2"}


def _force(monkeypatch, kernel):
    for pair in KERNELS[kernel].split():
        name, _, value = pair.partition("=")
        monkeypatch.setenv("PHYAI_FP8_" + name, value)


def _rows(m, k, seed):
    x = seeded((m, k), seed)
    x[0] = 0
    x[m // 2, k - 1] = float("inf")      # the scale of this row is not finite: nothing of it may reach its neighbours
    x[m - 1, 0] = float("nan")
    return x


def _same(a, b):
    return torch.equal(a.isnan(), b.isnan()) and torch.equal(a.nan_to_num(), b.nan_to_num())


@pytest.mark.parametrize("K", [528, 1168, 4304])
@pytest.mark.parametrize("M,N,epi", [(140, 528, None), (261, 272, "gelu"), (200, 288, "swiglu")])
@pytest.mark.parametrize("kernel", list(KERNELS))
def test_linear_equals_gemm_on_dense_codes(dev, monkeypatch, kernel, M, N, K, epi):
    from phyai_amd import ops

    if epi == "swiglu" and kernel in ("96", "12864") or kernel == "split" and K < 1152:
        pytest.skip("no such kernel")
    x = _rows(M, K, M + K).to(dev)
    wq, ws = ops.fp8_weight_quant(seeded((N, K), K, 0.02).to(dev))
    wq.view(torch.uint8)[5::37, :16] = 0x7F          # rows that begin with NaN codes: not the end of the row before
    bias = seeded((N,), 5).to(dev)
    _force(monkeypatch, kernel)
    xq, xs = ops.fp8_quant_rowwise(x)
    assert _same(ops.fp8_linear(x, wq, ws, bias, epilogue=epi), ops.fp8_gemm(xq, xs, wq, ws, bias, epilogue=epi))
    if epi is None:
        res, gate = seeded((M, N), 8).to(dev), seeded((1, N), 9).to(dev)
        assert _same(ops.fp8_linear(x, wq, ws, bias, residual=res, gate=gate), ops.fp8_gemm(xq, xs, wq, ws, bias, residual=res, gate=gate))


@pytest.mark.parametrize("K", [272, 400, 1040, 1264, 16368])
@pytest.mark.parametrize("M,N,epi", [(65, 512, None), (200, 640, "gelu"), (130, 544, "swiglu"), (1100, 272, None)])
def test_weight_streaming_takes_every_padded_width(dev, monkeypatch, M, N, K, epi):
    """Against the generic kernel, whose sums come in another order
    (fp32 sums of up to K products: a relative 2^-9 of the largest output covers the bf16 rounding on both sides)."""
    from phyai_amd import ops

    x = seeded((M, K), M + K).to(dev)
    wq, ws = ops.fp8_weight_quant(seeded((N, K), K, 0.02).to(dev))
    monkeypatch.setenv("PHYAI_FP8_FUSED", "0")
    monkeypatch.setenv("PHYAI_FP8_BIG", "0")
    assert ops.describe_linear_plan(M, N, K, epi).startswith("quantizer + small-m ")
    got = ops.fp8_linear(x, wq, ws, epilogue=epi).float()
    xq, xs = ops.fp8_quant_rowwise(x)
    monkeypatch.setenv("PHYAI_FP8_TILE", "128,128,1")
    want = ops.fp8_gemm(xq, xs, wq, ws, epilogue=epi).float()
    assert (got - want).abs().max() <= 2.0 ** -7 * want.abs().max()
    assert (got - want).norm() <= 2.0 ** -9 * want.norm()


@pytest.mark.parametrize("M,K", [(140, 272), (1, 528), (150, 1040), (140, 2064), (139, 4112), (140, 8208), (70, 16400), (3, 33808)])
def test_quantizers_fill_the_rest_of_a_row_with_zeros(dev, monkeypatch, M, K):
    """Through the linears, whose scratch starts out full of NaN codes: per-token, static, and the adaptive norm's.  One K that
    is padded in each of the launch forms of the quantizers (64, 128 and 256 threads, 1 - 16 chunks each, the loop)."""
    from phyai_amd import _lib, ops

    monkeypatch.setenv("PHYAI_FP8_FUSED", "0")       # codes staged at every size
    assert K % 128 != 0
    lib, N, ldq = _lib.load(), 64, (K + 127) // 128 * 128
    x = _rows(max(M, 3), K, K)[-M:].nan_to_num(0.0, 1.0, -1.0).to(dev)
    wq, ws = ops.fp8_weight_quant(seeded((N, K), K, 0.02).to(dev))
    scale, mod = torch.full((1,), 0.02, device=dev), seeded((1, 3 * K), 3, 0.1).to(dev)
    st = torch.cuda.current_stream().cuda_stream
    need = lib.phyai_fp8_linear_workspace_bytes(M, N, K, 0)
    up = lambda n: (n + 255) // 256 * 256
    codes_at = need - up(4 * M) - up(M * ldq)        # (the scratch ends in the codes and a scale per row)
    ref = {}
    for fill in (0, 0x7F):
        for name in ("token", "static", "norm"):
            wsp = torch.full((need,), fill, dtype=torch.uint8, device=dev)
            wsp[:16384] = 0                                    # (split-K counters start at zero)
            out = torch.empty(M, N, dtype=torch.bfloat16, device=dev)
            tail = (wq.data_ptr(), ws.data_ptr(), None)
            if name == "token":
                rc = lib.phyai_fp8_linear(x.data_ptr(), K, *tail, out.data_ptr(), N, M, N, K, 0, wsp.data_ptr(), need, st)
            elif name == "static":
                rc = lib.phyai_fp8_linear_per_tensor(x.data_ptr(), K, scale.data_ptr(), *tail, None, 0, None, 0, 0, out.data_ptr(), N, M, N, K, 0,
                                                     wsp.data_ptr(), need, st)
            else:
                rc = lib.phyai_fp8_adarmsnorm_linear(x.data_ptr(), K, mod.data_ptr(), 3 * K, 1, 1e-6, *tail, out.data_ptr(), N, M, N, K, 0,
                                                     wsp.data_ptr(), need, st)
            _lib.check(rc, name)
            torch.cuda.synchronize()
            assert not bool(out.isnan().any())
            codes = wsp[codes_at:codes_at + M * ldq].view(M, ldq)
            assert not bool(codes[:, K:].any()) and bool(codes[:, :K].any())
            assert torch.equal(ref.setdefault(name, out), out)
