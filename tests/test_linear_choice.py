"""The kernel that a linear's staged codes go to (choose_gemm with the fitted costs of csrc/gemm_big.hip), or that takes its rows."""

from __future__ import annotations

import random

import pytest
import torch

from conftest import seeded

GATED = "geglu_tanh"

# where the rules' lines alone or the width of a row of dense codes would have ready codes add in another order than staged ones
APART = [(947, 768, 768), (1435, 640, 512), (738, 768, 1040), (1847, 1152, 8192), (643, 1280, 1024), (964, 768, 1040), (300, 384, 272),
         (200, 512, 1040), (1894, 256, 736), (248, 2384, 704), (412, 2176, 15488), (178, 3584, 512)]


def _shapes(n):
    rng = random.Random(1)
    for _ in range(n):
        m, k = rng.randint(129, 9000), 128 * rng.randint(4, 128)
        yield m, 32 * rng.randint(8, 512), k, rng.choice([None, "gelu", GATED])


def _kind(plan):
    """What decides the order of the sums: weight streaming, tiles, tiles split along K."""
    plan = plan.removeprefix("quantizer + ")
    return plan.split()[0] + (plan.split("splits=")[1].split()[0] if "splits=" in plan else "")


def test_layout_does_not_change_the_order_of_the_sums(monkeypatch):
    from phyai_amd import ops

    for var in ("BIG", "BIG_DEPTH", "BIG_SPLITS", "TILE", "RULES"):
        monkeypatch.delenv("PHYAI_FP8_" + var, raising=False)
    monkeypatch.setenv("PHYAI_FP8_FUSED", "0")   # (one launch in their place keeps their order: tests/test_gpu_panel.py)
    changed = 0
    for m, n, k, epi in _shapes(1500):
        if epi == GATED and n % 32 or m * k >= 1 << 31:
            continue
        lay = "operand_gated" if epi == GATED else "operand"
        row, op = ops.describe_linear_plan(m, n, k, epi), ops.describe_linear_plan(m, n, k, epi, weight_layout=lay)
        assert _kind(row) == _kind(op), (m, n, k, epi, row, op)
        rule = ops.describe_plan(m, n, k, epi)
        assert _kind(row) in (_kind(rule), "tile1", "small-m"), (m, n, k, epi, rule, row)   # nothing is newly split
        changed += row.removeprefix("quantizer + ") != rule
    assert changed > 50


def test_ready_codes_add_in_the_order_of_staged_ones(monkeypatch):
    """A norm's forward_fp8 and the linear behind it stand for the norm and the linear: a GEMM on ready codes adds in the order
    of the linear that stages its own, at every size (one launch in the place of the two keeps that order, on the GPU)."""
    from phyai_amd import ops

    for var in ("BIG", "BIG_DEPTH", "BIG_SPLITS", "TILE", "RULES", "SKINNY_PLAN", "SKINNY_MAXM"):
        monkeypatch.delenv("PHYAI_FP8_" + var, raising=False)
    monkeypatch.setenv("PHYAI_FP8_FUSED", "0")
    rng, shapes = random.Random(3), [(m, n, k, None) for m, n, k in APART]
    for _ in range(4000):
        m, n = round(2 ** rng.uniform(0, 13.7)), rng.choice([32 * rng.randint(1, 64), 128 * rng.randint(1, 100)])
        k = rng.choice([16 * rng.randint(1, 128), 16 * rng.randint(1, 1024), 128 * rng.randint(1, 128)])
        if m * k < 1 << 31:
            shapes.append((m, n, k, rng.choice([None, None, "gelu", GATED])))
    for m, n, k, epi in shapes:
        for lay in [None, "operand_gated" if epi == GATED else "operand"][:2 if k % 128 == 0 else 1]:
            ready, staged = ops.describe_plan(m, n, k, epi, weight_layout=lay), ops.describe_linear_plan(m, n, k, epi, weight_layout=lay)
            assert _kind(ready) == _kind(staged), (m, n, k, epi, lay, ready, staged)


def test_rules_alone(monkeypatch):
    from phyai_amd import ops

    monkeypatch.setenv("PHYAI_FP8_RULES", "1")
    monkeypatch.setenv("PHYAI_FP8_FUSED", "0")
    for m, n, k, epi in _shapes(200):
        assert ops.describe_linear_plan(m, n, k, epi).removeprefix("quantizer + ") == ops.describe_plan(m, n, k, epi)


def test_where_one_launch_takes_more_rows(monkeypatch):
    """csrc/gemm_panel.hip: only in the place of weight streaming or an unsplit tile, within the K and grid that were measured."""
    from phyai_amd import ops

    for var in ("BIG", "TILE", "SKINNY_PLAN", "FUSED", "RULES"):
        monkeypatch.delenv("PHYAI_FP8_" + var, raising=False)
    rng, seen = random.Random(2), 0
    for _ in range(3000):
        m, n, k = rng.randint(1, 2000), 16 * rng.randint(1, 300), rng.choice([16 * rng.randint(1, 80), 128 * rng.randint(1, 10)])
        lay = rng.choice([None, "operand"]) if k % 128 == 0 else None
        epi = rng.choice([None, None, None, "gelu"])
        plan = ops.describe_linear_plan(m, n, k, epi, weight_layout=lay)
        if not plan.startswith("one launch: panel"):
            continue
        seen += 1
        grid = [int(v) for v in plan.split("grid=")[1].split("x")]
        assert epi is None and m > 48 and k <= 1024 and (lay or k < 768) and grid[0] * grid[1] <= (512 if lay else 768), (m, n, k, lay, plan)
        with monkeypatch.context() as two:
            two.setenv("PHYAI_FP8_FUSED", "0")
            assert _kind(ops.describe_linear_plan(m, n, k, epi, weight_layout=lay)) in ("small-m", "tile1"), (m, n, k, lay)
    assert seen > 100


def test_weights_stay_out_of_registers_where_that_is_asked_for(monkeypatch):
    """PHYAI_FP8_BIG_DIRECT=0: no tile shape, chosen by rule or by cost, takes weights in operand order straight into registers."""
    from phyai_amd import ops

    for var in ("BIG", "BIG_DEPTH", "BIG_SPLITS", "TALL", "TILE", "RULES"):
        monkeypatch.delenv("PHYAI_FP8_" + var, raising=False)
    monkeypatch.setenv("PHYAI_FP8_FUSED", "0")
    shapes = [(*s, "operand_gated" if s[3] == GATED else "operand") for s in _shapes(300) if s[0] * s[2] < 1 << 31]
    plans = lambda: [f(m, n, k, epi, weight_layout=lay) for m, n, k, epi, lay in shapes for f in (ops.describe_linear_plan, ops.describe_plan)]
    assert sum("in registers" in p and "x256" in p for p in plans()) > 50
    monkeypatch.setenv("PHYAI_FP8_BIG_DIRECT", "0")
    staged = plans()
    assert not [p for p in staged if "tile" in p and "in registers" in p]


@pytest.mark.parametrize("M,N,K,epi,tile", [
    # slower in tall tiles, by 4 to 16 % as cards differ
    (6741, 8960, 1408, GATED, "192x128"), (5398, 17856, 768, GATED, "192x128"), (6693, 15616, 768, GATED, "192x128"),
    (8689, 11840, 896, "gelu_tanh", "192x128"), (5360, 32512, 512, "swiglu", "192x128"),
    # faster in them, where less than 5.5 % in favour would not have it so
    (2307, 26336, 640, "swiglu", "x256"), (4467, 23072, 896, "swiglu", "x256"), (3996, 15776, 768, GATED, "x256"),
    # 14 - 23 % faster in them
    (816, 32768, 2048, GATED, "208x256"), (4800, 8192, 2048, "gelu", "208x256"), (4800, 6144, 2048, None, "240x256"),
    (5000, 5120, 1280, None, "x256"), (3264, 2560, 2048, None, "144x256")])
def test_tall_tiles_beside_staged_ones(monkeypatch, M, N, K, epi, tile):
    from phyai_amd import ops

    for var in ("BIG", "BIG_DEPTH", "BIG_SPLITS", "BIG_DIRECT", "TALL", "TILE", "RULES"):
        monkeypatch.delenv("PHYAI_FP8_" + var, raising=False)
    gated = epi is not None and not epi.startswith("gelu")
    plan = ops.describe_linear_plan(M, N, K, epi, weight_layout="operand_gated" if gated else "operand")
    assert tile in plan and ("in registers" in plan) == (tile != "192x128"), plan


# (rows, columns, K, epilogue): rule's shape -> chosen shape, one per pair that occurs
CHANGED = [(2032, 9216, 640, "gelu"), (4310, 3648, 640, None), (497, 2432, 8320, None), (2489, 384, 1792, None), (2553, 864, 8320, None),
           (400, 6144, 8192, None), (3548, 3392, 5120, None), (3531, 8160, 640, None), (2740, 1056, 8448, None), (278, 3072, 9600, None)]


@pytest.mark.parametrize("M,N,K,epi", CHANGED)
def test_costs_choose_another_shape_than_the_rules(monkeypatch, M, N, K, epi):
    from phyai_amd import ops

    for var in ("BIG", "BIG_DEPTH", "BIG_SPLITS", "TILE", "RULES", "FUSED"):
        monkeypatch.delenv("PHYAI_FP8_" + var, raising=False)
    chosen = ops.describe_linear_plan(M, N, K, epi)
    monkeypatch.setenv("PHYAI_FP8_RULES", "1")
    assert chosen.startswith("quantizer + ") and ops.describe_linear_plan(M, N, K, epi) != chosen


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,epi", CHANGED)
def test_chosen_kernel_in_both_layouts_and_without_a_workspace_of_its_own(dev, monkeypatch, M, N, K, epi):
    """Operand order changes no bit, the static-scratch form gives the same where its array holds the codes, and the result is
    the rules' kernel's up to the order of fp32 sums (2^-7 of the largest output covers one bf16 step on either side)."""
    from phyai_amd import _lib, ops

    x = seeded((M, K), M + K).to(dev)
    wq, ws = ops.fp8_weight_quant(seeded((N, K), K, 0.02).to(dev))
    got = ops.fp8_linear(x, wq, ws, epilogue=epi)
    relaid = ops.fp8_linear(x, ops.fp8_weight_to_operand_order(wq), ws, epilogue=epi, weight_layout="operand")
    assert torch.equal(got.view(torch.int16), relaid.view(torch.int16))
    xq, xs = ops.fp8_quant_rowwise(x)
    ready = ops.fp8_gemm(xq, xs, wq, ws, epilogue=epi)
    assert torch.equal(got.view(torch.int16), ready.view(torch.int16))
    with monkeypatch.context() as rules:
        rules.setenv("PHYAI_FP8_RULES", "1")
        want = ops.fp8_linear(x, wq, ws, epilogue=epi).float()
    assert (got.float() - want).abs().max() <= 2.0 ** -7 * want.abs().max()
    out = torch.empty_like(got)
    rc = _lib.load().phyai_fp8_linear_static(x.data_ptr(), K, wq.data_ptr(), ws.data_ptr(), None, out.data_ptr(), N, M, N, K,
                                             {"gelu": 5}.get(epi, 0), torch.cuda.current_stream().cuda_stream)
    if M * K < 24 << 20:
        _lib.check(rc, "static")
        assert torch.equal(got.view(torch.int16), out.view(torch.int16))


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", APART)
def test_ready_codes_give_the_bits_of_the_linear(dev, M, N, K):
    """Per token, one static scale, and the adaptive norm in front: separate calls and the one that stands for them."""
    from test_gpu_norm_linear import _norm_linear

    from phyai_amd import _lib, ops

    lib = _lib.load()
    x, bias, mod = seeded((M, K), M + K).to(dev), seeded((N,), 4).to(dev), seeded((1, 3 * K), 6, 0.2).to(dev)
    w, ws = ops.fp8_weight_quant(seeded((N, K), K, 0.02).to(dev))
    one = torch.full((1,), 0.02, device=dev)
    for layout in (None, "operand")[:2 if K % 128 == 0 else 1]:
        wq = ops.fp8_weight_to_operand_order(w) if layout else w
        how = dict(weight_layout=layout)
        same = lambda a, b: torch.equal(a.view(torch.int16), b.view(torch.int16))
        assert same(ops.fp8_linear(x, wq, ws, bias, **how), ops.fp8_gemm(*ops.fp8_quant_rowwise(x), wq, ws, bias, **how))
        out = torch.empty(M, N, dtype=torch.bfloat16, device=dev)
        scratch = torch.zeros(lib.phyai_fp8_linear_workspace_bytes(M, N, K, 0), dtype=torch.uint8, device=dev)
        _lib.check(lib.phyai_fp8_linear_per_tensor(
            x.data_ptr(), K, one.data_ptr(), wq.data_ptr(), ws.data_ptr(), bias.data_ptr(), None, 0, None, 0, 0, out.data_ptr(), N, M, N, K,
            ops.WEIGHT_LAYOUTS[layout], scratch.data_ptr(), scratch.numel(), torch.cuda.current_stream().cuda_stream), "per tensor")
        assert same(out, ops.fp8_gemm(ops.fp8_quant_static(x, one), one, wq, ws, bias, **how))
        xq, xs, _ = ops.adarmsnorm_fp8(x, mod, 1e-6)
        ready = ops.fp8_gemm(xq, xs, wq, ws, bias, **how)
        assert same(ops.fp8_linear(ops.adarmsnorm(x, mod, 1e-6)[0], wq, ws, bias, **how), ready)
        assert same(_norm_linear(x, mod, wq, ws, bias, None, layout)[0], ready)
