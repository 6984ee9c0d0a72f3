"""Small-M linears that quantize their own rows (csrc/gemm_selfq.h) against quantizer + GEMM, bit for bit: every form
that exists at the shortest and the longest K it is taken for (partial and missing K steps), own / handed-over / static
scales, NaN and Inf in rows, each time with a check that one side is that form and the other is not; the reciprocal form of the static and weight quantizers against the division on the CPU; and weights re-laid in place."""

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


# Every form that exists: layout, weight tiles per workgroup, K steps per wavefront, for 4-row and 8-row workgroups.
STEPS = (1, 2, 4, 6, 8, 12, 16)
LONGEST = {  # csrc/gemm_selfq.h, selfq_max_k: (operand order, tiles, groups of four rows) -> K
    (False, 1, 1): 8192, (False, 1, 2): 8192, (False, 2, 1): 8192, (False, 2, 2): 4096, (False, 4, 1): 2048, (False, 4, 2): 2048,
    (False, 8, 1): 1088, (False, 8, 2): 1088, (True, 1, 1): 16384, (True, 1, 2): 16384, (True, 2, 1): 16384, (True, 2, 2): 12288,
    (True, 4, 1): 4096, (True, 4, 2): 4096, (True, 8, 1): 2048, (True, 8, 2): 2048}
LONGEST_STATIC = {**LONGEST, (True, 1, 2): 8192, (True, 2, 2): 8192, (False, 8, 1): 1600, (False, 8, 2): 1600}


def _forms(source):
    for (operand, nt, rg), longest in (LONGEST_STATIC if source == "scalar" else LONGEST).items():
        for i, steps in enumerate(STEPS):
            first = 1024 * (STEPS[i - 1] if i else 0) + (128 if operand else 16)
            if first > longest:
                continue
            if operand and source == "rows" and steps <= 4 and (nt, steps) != (4, 4):
                continue      # gemm_skinny_fused.hip serves these
            if operand and source == "maxima" and steps == 1 and nt != 8:
                continue
            last = min(longest, 1024 * steps)
            if not operand and source != "scalar" and last % 128 == 0 and last <= 4096:
                last -= 16        # whole K steps are served by gemm_skinny_fused.hip as well
            yield pytest.param(operand, nt, rg, steps, first, last, id=f"{'operand' if operand else 'row-major'}-nt{nt}-rows{4 * rg}-steps{steps}")


def _rows_and_columns(rg, nt):
    """Token rows and the fewest columns for which a grid of at most 256 workgroups needs nt tiles each."""
    M = 3 if rg == 1 else 13
    return M, 48 if nt == 1 else 16 * (nt // 2) * (256 // (1 if rg == 1 else 2)) + 16


def _codes(dev, n, k, seed):
    """fp8 weights without the cost of quantizing them: finite codes of both signs, small exponents."""
    g = torch.Generator(device=dev).manual_seed(seed)
    return (torch.randint(0, 256, (n, k), dtype=torch.uint8, generator=g, device=dev) & 0xB7).view(torch.float8_e4m3fn)


def _activations(dev, M, K):
    x = seeded((M, K), K + M)
    if K > 1000:
        x[1, K - 3] = float("inf" if K % 32 else "nan")
    return x.to(dev)


@pytest.mark.parametrize("operand,nt,rg,steps,first,last", _forms("rows"))
def test_every_form_that_finds_its_own_maxima(dev, monkeypatch, operand, nt, rg, steps, first, last):
    from phyai_amd import ops

    M, N = _rows_and_columns(rg, nt)
    layout = "operand" if operand else None
    for K in {first, last}:
        assert ops.describe_linear_plan(M, N, K, weight_layout=layout).startswith(f"one launch: rows in registers, rows={4 * rg} nt={nt} steps={steps} ")
        x, w, ws = _activations(dev, M, K), _codes(dev, N, K, K), torch.rand(N, device=dev) * 0.02
        if operand:
            w = ops.fp8_weight_to_operand_order(w)
        bias, res, gate = seeded((N,), 7).to(dev), seeded((M, N), 8).to(dev), seeded((1, N), 9).to(dev)
        for kw in ({}, dict(residual=res, gate=gate)):
            call = lambda: ops.fp8_linear(x, w, ws, bias, weight_layout=layout, **kw)
            _same(call(), _two_launches(monkeypatch, call))


@pytest.mark.parametrize("operand,nt,rg,steps,first,last", _forms("scalar"))
def test_every_form_with_one_static_scale(dev, monkeypatch, operand, nt, rg, steps, first, last):
    """(The quantizer's codes would be in the workspace behind the GEMM's region: one launch leaves it untouched.)"""
    from phyai_amd import _lib, ops

    lib, st = _lib.load(), torch.cuda.current_stream().cuda_stream
    M, N = _rows_and_columns(rg, nt)
    for K in {first, last}:
        x, w, ws, scale = _activations(dev, M, K), _codes(dev, N, K, K), torch.rand(N, device=dev) * 0.02, torch.tensor([0.0357], device=dev)
        if operand:
            w = ops.fp8_weight_to_operand_order(w)
        bias, res, gate = seeded((N,), 7).to(dev), seeded((M, N), 8).to(dev), seeded((1, N), 9).to(dev)
        need = lib.phyai_fp8_linear_workspace_bytes(M, N, K, 0)

        def call(residual):
            scratch, out = torch.full((need,), 0xAB, dtype=torch.uint8, device=dev), torch.empty(M, N, dtype=torch.bfloat16, device=dev)
            scratch[:16384] = 0
            extra = (res.data_ptr(), N, gate.data_ptr(), N, 1) if residual else (None, 0, None, 0, 0)
            _lib.check(lib.phyai_fp8_linear_per_tensor(x.data_ptr(), K, scale.data_ptr(), w.data_ptr(), ws.data_ptr(), bias.data_ptr(), *extra,
                                                       out.data_ptr(), N, M, N, K, ops.FLAG_W_OPERAND_ORDER if operand else 0, scratch.data_ptr(), need, st), "per_tensor")
            return out, bool((scratch[16384:] == 0xAB).all())

        for residual in (False, True):
            got, one_launch = call(residual)
            want, other = _two_launches(monkeypatch, lambda: call(residual))
            assert one_launch and not other
            _same(got, want)


@pytest.mark.parametrize("operand,nt,rg,steps,first,last", _forms("maxima"))
def test_every_form_on_maxima_handed_on(dev, monkeypatch, operand, nt, rg, steps, first, last):
    """As the second projection of an MLP (K is its intermediate width), whose first one leaves the maxima."""
    from phyai_amd import ops

    M, O = _rows_and_columns(rg, nt)
    H = 128
    for I in {first, last}:
        plan = ops.describe_mlp_plan(M, H, I, O, "geglu_tanh", operand_order=operand)
        assert plan.startswith("row maxima handed over") and f"| one launch: rows in registers, rows={4 * rg} nt={nt} steps={steps} " in plan, plan
        x, w1, w2 = seeded((M, H), 3).to(dev), _codes(dev, 2 * I, H, 1), _codes(dev, O, I, 2)
        s1, s2 = torch.rand(2 * I, device=dev) * 0.01, torch.rand(O, device=dev) * 0.01
        if operand:
            w1, w2 = ops.fp8_weight_to_operand_order(w1, gated=True), ops.fp8_weight_to_operand_order(w2)
        call = lambda: ops.fp8_mlp(x, w1, s1, None, w2, s2, None, epilogue="geglu_tanh", weight1_layout="operand_gated" if operand else None,
                                   weight2_layout="operand" if operand else None)
        _same(call(), _two_launches(monkeypatch, call))


@pytest.mark.parametrize("M,N,layout,K", [(1, 48, None, 144), (48, 208, None, 5504), (33, 3072, "operand", 4096), (48, 1040, "operand", 12160),
                                          (128, 512, "operand", 1024), (125, 1040, None, 1392), (100, 2048, "operand", 2048)])
def test_up_to_48_rows_or_128_with_one_scale(dev, monkeypatch, M, N, layout, K):
    """The module's call with a static scale on every row count; with per-token scales up to 48 rows."""
    import phyai_amd.linear as L
    from phyai_amd import ops

    x, w, bias = _activations(dev, max(M, 2), K)[:M], _codes(dev, N, K, N), seeded((N,), 7).to(dev)
    if M <= 48:
        assert "rows in registers" in ops.describe_linear_plan(M, N, K, weight_layout=layout)
    L.init()
    try:
        for scheme in ["PER_TENSOR"] + (["PER_CHANNEL"] if M <= 48 else []):
            lin = L.ColumnParallelLinear(K, N, bias=True, params_dtype=torch.bfloat16,
                                         spec=L.Fp8Spec(granularity=L.Granularity[scheme], operand_order=layout is not None))
            lin.weight.data.copy_(w)
            lin.weight_scale.data.fill_(0.01)
            if scheme == "PER_TENSOR":
                lin.input_scale.data.fill_(0.0357)
            lin.bias.data.copy_(bias)
            lin.post_load()
            _same(lin(x)[0], _two_launches(monkeypatch, lambda: lin(x)[0]))
    finally:
        L._reset_for_test()


@pytest.mark.parametrize("H,I,operand", [(1040, 1392, False), (560, 6016, False), (128, 8192, False), (512, 12032, True)])
@pytest.mark.parametrize("M", [1, 6, 15])
@pytest.mark.parametrize("epi", ["geglu_tanh", "swiglu", "gelu"])
def test_mlp_hands_the_maxima_on(dev, monkeypatch, M, H, I, operand, epi):
    from phyai_amd import ops

    assert ops.describe_mlp_plan(M, H, I, H, epi, operand_order=operand).startswith("row maxima handed over")
    gated = epi != "gelu"
    w1, s1 = ops.fp8_weight_quant(seeded(((2 if gated else 1) * I, H), 1, 0.02).to(dev))
    w2, s2 = ops.fp8_weight_quant(seeded((H, I), 2, 0.02).to(dev))
    lay1, lay2 = ("operand_gated" if gated else "operand", "operand") if operand else (None, None)
    if operand:
        w1, w2 = ops.fp8_weight_to_operand_order(w1, gated=gated), ops.fp8_weight_to_operand_order(w2)
    x = seeded((M, H), 3).to(dev)
    call = lambda: ops.fp8_mlp(x, w1, s1, None, w2, s2, None, epilogue=epi, weight1_layout=lay1, weight2_layout=lay2)
    _same(call(), _two_launches(monkeypatch, call))


@pytest.mark.parametrize("scale", [16.0 / 448.0, 0.25, 3.0e-3, 1e-39, 7.0, float("inf")])
def test_static_quantizer_equals_the_division(dev, scale):
    from phyai_amd import ops

    x = torch.arange(65536, dtype=torch.int32).to(torch.int16).view(torch.bfloat16).reshape(64, 1024)   # every bf16 value
    s = torch.tensor([scale])
    got = ops.fp8_quant_static(x.to(dev), s.to(dev)).view(torch.uint8).cpu()
    q = (x.float() / s).clamp(-448.0, 448.0)
    want = q.to(torch.float8_e4m3fn).view(torch.uint8)
    nan = q.isnan()
    assert torch.equal(got[~nan], want[~nan]) and bool(((got[nan] & 0x7F) == 0x7F).all())


def test_weight_quantizer_equals_the_division(dev):
    from phyai_amd import ops

    w = (seeded((512, 2048), 5) * torch.logspace(-6, 3, 512)[:, None]).to(torch.bfloat16)
    q, s = ops.fp8_weight_quant(w.to(dev))
    want_s = w.float().abs().amax(1) / 448.0
    assert torch.equal(s.cpu(), want_s)
    assert torch.equal(q.view(torch.uint8).cpu(), (w.float() / want_s[:, None]).clamp(-448, 448).to(torch.float8_e4m3fn).view(torch.uint8))


@pytest.mark.parametrize("N,K", [(16, 128), (48, 1024), (1040, 1152), (32, 2176), (64, 8192), (48, 8320), (16, 16384)])
def test_weights_relaid_in_place(dev, N, K):
    from phyai_amd import ops

    w = torch.randint(0, 256, (N, K), dtype=torch.uint8, generator=torch.Generator().manual_seed(N + K)).to(dev)
    want = ops.fp8_weight_to_operand_order(w.view(torch.float8_e4m3fn)).view(torch.uint8)
    assert ops._native().relay_weight(w, False) is True
    assert torch.equal(w, want)
