"""What the library keeps per shape between calls (csrc/call_memo.h, used by choose_gemm and the workspace carve).  The
rest of the suite runs with the tuning switch on, under which nothing is kept; here it is off: the container by itself
on the CPU, and on the GPU a process of its own whose calls differ in one thing at a time."""

from __future__ import annotations

import os
import shutil
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

CLIENT = r"""
#include <stdio.h>
#include "call_memo.h"
int main() {
    phyai::CallMemo<long, 8> memo;
    long made = 0;
    auto get = [&](long a, long b, long c, long d) {
        return memo.get(a, b, c, d, [&]() { ++made; return ((a * 31 + b) * 31 + c) * 31 + d; });
    };
    // every one of the four words is part of the key, negative and 64-bit values included
    const long keys[][4] = {{1, 2, 3, 4}, {2, 2, 3, 4}, {1, 3, 3, 4}, {1, 2, 4, 4}, {1, 2, 3, 5}, {-1, 2, 3, 4}, {1L << 40, 2, 3, 4}, {0, 0, 0, 0}};
    for (int round = 0; round < 3; ++round)
        for (auto& k : keys)
            if (get(k[0], k[1], k[2], k[3]) != ((k[0] * 31 + k[1]) * 31 + k[2]) * 31 + k[3]) return 1;
    // more keys than slots: those that meet in a slot take turns and never see each other's value
    for (int round = 0; round < 3; ++round)
        for (long a = 0; a < 1000; ++a)
            if (get(a, a % 7, 128, 64) != ((a * 31 + a % 7) * 31 + 128) * 31 + 64) return 2;
    // a second call is served from the slot; a maker that throws leaves none
    made = 0;
    get(5, 6, 7, 8); get(5, 6, 7, 8);
    const bool kept = made == 1;
    struct Thrown {};
    try { memo.get(9, 9, 9, 9, [&]() -> long { throw Thrown(); }); } catch (Thrown&) {}
    if (get(9, 9, 9, 9) != ((9 * 31 + 9) * 31 + 9) * 31 + 9) return 3;
    puts(kept ? "kept" : "made again");
    return 0;
}
"""


def test_the_container(tmp_path):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("no C++ compiler")
    src, exe = tmp_path / "memo.cpp", tmp_path / "memo"
    src.write_text(CLIENT)
    subprocess.check_call([gxx, "-std=c++17", "-Wall", "-Werror", "-I", os.path.join(ROOT, "phyai_amd", "csrc"), str(src), "-o", str(exe)])
    env = {k: v for k, v in os.environ.items() if not k.startswith("PHYAI_FP8_")}
    for tuning, want in ((None, "kept"), ("1", "made again")):     # a tuning run follows the environment: nothing is kept
        out = subprocess.run([str(exe)], env={**env, **({"PHYAI_FP8_TUNING": tuning} if tuning else {})}, capture_output=True, text=True, timeout=60)
        assert out.returncode == 0 and out.stdout.strip() == want, (out.returncode, out.stdout, out.stderr)


# Calls that differ in one of the things a choice depends on: rows, widths, epilogue, layout, scale kind, where the codes
# come from, the alignment of bias and output, the output's row stride, the norm, maxima handed on.
CALLS = r"""
import sys
import torch
from phyai_amd import _lib, ops
dev, lib = torch.device("cuda", 0), _lib.load()
g = torch.Generator().manual_seed(1)
rnd = lambda *s, scale=1.0: (torch.randn(*s, generator=g) * scale).to(torch.bfloat16).to(dev)
st = torch.cuda.current_stream().cuda_stream
ws = torch.zeros(64 << 20, dtype=torch.uint8, device=dev)
N, K = 1056, 1024
# a linear that one launch takes (csrc/gemm_panel.hip) unless its output lies inside its rows; K that is padded where it is staged
rows = rnd(400, 512)
square, s_sq = ops.fp8_weight_quant(rnd(512, 512, scale=0.02))
square = ops.fp8_weight_to_operand_order(square)
ragged = [(rnd(m, k), *ops.fp8_weight_quant(rnd(n, k, scale=0.02))) for m, n, k in ((300, 1056, 656), (900, 272, 720), (70, 512, 1040))]
xs = {m: rnd(m, K) for m in (1, 40, 100, 130, 300)}
mod, gate = rnd(1, 3 * K, scale=0.2), rnd(1, N)
w, s = ops.fp8_weight_quant(rnd(N, K, scale=0.02))
w2, s2 = ops.fp8_weight_quant(rnd(K, N // 2, scale=0.02))
plain, pairs = ops.fp8_weight_to_operand_order(w), ops.fp8_weight_to_operand_order(w, gated=True)
bias_store = rnd(N + 8)
scalar = torch.tensor([0.05], device=dev)
FLAG = {"row": 0, "op": ops.FLAG_W_OPERAND_ORDER, "opg": ops.FLAG_W_OPERAND_GATED}

def calls():
    for m, x in xs.items():
        xq, xsc = ops.fp8_quant_rowwise(x)
        for epi, layout in ((0, "row"), (0, "op"), (1, "row"), (1, "opg"), (4, "row"), (4, "op")):
            W, n_out = {"row": w, "op": plain, "opg": pairs}[layout], N // 2 if epi == 1 else N
            for bias_at in (0, 1):                     # elements: a bias that is 2-byte aligned is no bias for vector loads
                for pad, out_at in ((0, 0), (8, 0), (4, 0), (1, 0), (0, 4), (0, 1)):
                    out = torch.zeros(m * (n_out + pad) + 16, dtype=torch.bfloat16, device=dev)
                    ldo = n_out + pad
                    o, b, e = out.data_ptr() + 2 * out_at, bias_store.data_ptr() + 2 * bias_at, epi | FLAG[layout]
                    tail = (o, ldo, m, N, K, e, ws.data_ptr(), ws.numel(), st)
                    yield ("linear", m, epi, layout, bias_at, pad, out_at), out, lambda: lib.phyai_fp8_linear(x.data_ptr(), K, W.data_ptr(), s.data_ptr(), b, *tail)
                    yield ("gemm", m, epi, layout, bias_at, pad, out_at), out, lambda: lib.phyai_fp8_gemm(xq.data_ptr(), xsc.data_ptr(), 0, W.data_ptr(), s.data_ptr(), b, *tail)
                    yield ("static", m, epi, layout, bias_at, pad, out_at), out, lambda: lib.phyai_fp8_linear_per_tensor(
                        x.data_ptr(), K, scalar.data_ptr(), W.data_ptr(), s.data_ptr(), b, None, 0, None, 0, 0, *tail)
                    yield ("norm", m, epi, layout, bias_at, pad, out_at), out, lambda: lib.phyai_fp8_adarmsnorm_linear(
                        x.data_ptr(), K, mod.data_ptr(), 3 * K, 1, 1e-6, W.data_ptr(), s.data_ptr(), b, *tail)
        out = torch.zeros(m, K, dtype=torch.bfloat16, device=dev)
        for epi in (1, 3):
            yield ("mlp", m, epi), out, lambda: lib.phyai_fp8_mlp(x.data_ptr(), K, w.data_ptr(), s.data_ptr(), None, 0, w2.data_ptr(), s2.data_ptr(), None, 0,
                None, 0, None, 0, 0, out.data_ptr(), K, m, K, N // 2, K, epi, ws.data_ptr(), ws.numel(), st)

    apart, inside = torch.zeros_like(rows), torch.zeros_like(rows)
    square_call = lambda x, out: lib.phyai_fp8_linear(x.data_ptr(), 512, square.data_ptr(), s_sq.data_ptr(), None, out.data_ptr(), 512, 400, 512, 512,
                                                      FLAG["op"], ws.data_ptr(), ws.numel(), st)
    yield ("apart",), apart, lambda: square_call(rows, apart)
    yield ("inside",), inside, lambda: square_call(inside.copy_(rows), inside)
    for x, W, sc in ragged:
        (m, k), n = x.shape, W.shape[0]
        xq, xsc = ops.fp8_quant_rowwise(x)
        out = torch.zeros(m, n, dtype=torch.bfloat16, device=dev)
        tail = (out.data_ptr(), n, m, n, k, 0, ws.data_ptr(), ws.numel(), st)
        yield ("ragged linear", m), out, lambda: lib.phyai_fp8_linear(x.data_ptr(), k, W.data_ptr(), sc.data_ptr(), None, *tail)
        yield ("ragged static", m), out, lambda: lib.phyai_fp8_linear_per_tensor(x.data_ptr(), k, scalar.data_ptr(), W.data_ptr(), sc.data_ptr(), None,
                                                                                 None, 0, None, 0, 0, *tail)
        yield ("ragged gemm", m), out, lambda: lib.phyai_fp8_gemm(xq.data_ptr(), xsc.data_ptr(), 0, W.data_ptr(), sc.data_ptr(), None, *tail)

results = {}
for sweep in range(2):
    for name, out, call in calls():
        out.zero_()
        _lib.check(call(), str(name))
        got = out.cpu().clone()
        if sweep and not torch.equal(got.view(torch.int16), results[name].view(torch.int16)):
            sys.exit(f"second sweep differs: {name}")
        results[name] = got
same = lambda a, b: torch.equal(results[a].view(torch.int16), results[b].view(torch.int16))
assert same(("apart",), ("inside",)) and all(same(("ragged linear", x.shape[0]), ("ragged gemm", x.shape[0])) for x, _, _ in ragged)
torch.save(results, sys.argv[1])
print(len(results), "calls")
"""


@pytest.mark.gpu
def test_calls_that_differ_in_one_thing_give_the_same_with_and_without_the_memory(dev, tmp_path):
    import torch

    got = {}
    env = {k: v for k, v in os.environ.items() if not k.startswith("PHYAI_FP8_")}
    for tuning in ("0", "1"):
        path = str(tmp_path / f"out{tuning}.pt")
        run = subprocess.run([sys.executable, "-c", CALLS, path], env={**env, "PYTHONPATH": ROOT, "PHYAI_FP8_TUNING": tuning}, capture_output=True,
                             text=True, timeout=100)
        assert run.returncode == 0, run.stderr[-2000:]
        got[tuning] = torch.load(path, weights_only=True)
    assert got["0"].keys() == got["1"].keys() and len(got["0"]) > 1000
    for name, a in got["0"].items():
        assert torch.equal(a.view(torch.int16), got["1"][name].view(torch.int16)), name
