"""The one-launch small-M linear loads its activation rows with inline-assembly loads the compiler cannot
see (phyai_amd/csrc/gemm_skinny_fused.hip).  What must hold of the code the compiler makes around them is
checked on the gfx950 assembly by phyai_amd/csrc/check_fused_asm.py (no GPU needed); the library's build
runs the same check.  Here: the check passes on the current sources, and it does catch each kind of
violation when one is planted in the assembly text."""

from __future__ import annotations

import importlib.util
import os
import re

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def guard():
    spec = importlib.util.spec_from_file_location("check_fused_asm", os.path.join(ROOT, "phyai_amd", "csrc", "check_fused_asm.py"))
    mod = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(mod)
    return mod


@pytest.fixture(scope="module")
def asm(guard):
    problems = guard.check_file(make=True)
    assert not problems, "\n".join(problems[:20])
    return open(guard.ASM, encoding="utf-8").read()


def test_every_instantiation_passes(guard, asm):
    kernels = guard.kernels_of(asm)
    assert len(kernels) >= 400
    # all variants are there: weights staged / straight into registers, own / handed-over row maxima
    names = "\n".join(k.split(":", 1)[0] for k in kernels)
    for tail in ("ELb0ELb0ELb0E", "ELb0ELb1ELb0E", "ELb0ELb0ELb1E", "ELb1ELb1ELb1E"):
        assert tail in names, tail


def test_planted_violations_are_caught(guard, asm):
    k = next(k for k in guard.kernels_of(asm) if "ILi8ELi2ELi4ELi0ELb0ELb1ELb1E" in k.split(":", 1)[0])
    name = k.split(":", 1)[0]
    rows = guard.rows_loaded(name)
    assert rows == 9 and not guard.check_kernel(k, rows)
    body, waited = guard.stretch(k)
    first = body[0]
    dest = re.search(r"v\[(\d+):\d+\]", first).group(1)
    lines = k.split("\n")
    at = next(i for i, line in enumerate(lines) if line.strip() == first)
    # a copy of a register in flight
    planted = "\n".join(lines[: at + 1] + [f"\tv_mov_b32_e32 v250, v{dest}"] + lines[at + 1:])
    assert any("touches a register" in p for p in guard.check_kernel(planted, rows))
    # a branch in the stretch
    planted = "\n".join(lines[: at + 1] + ["\ts_cbranch_scc1 .LBB0_99"] + lines[at + 1:])
    assert any("s_cbranch" in p for p in guard.check_kernel(planted, rows))
    # one more vector-memory instruction than the wait counts
    last = max(i for i, line in enumerate(lines[: at + 200]) if line.strip() in body and line.strip().startswith("global_load_dwordx4"))
    planted = "\n".join(lines[: last + 1] + ["\tglobal_load_dword v251, v252, s[0:1]"] + lines[last + 1:])
    assert any("vmcnt" in p for p in guard.check_kernel(planted, rows))
    # scratch
    planted = k + "\n\tscratch_store_dword off, v1, s0\n"
    assert any("scratch" in p for p in guard.check_kernel(planted, rows))


def test_tile_kernels_use_no_scratch(guard):
    """The pipelined tile kernels count their global -> LDS copies by hand (s_waitcnt vmcnt(N)): a spill would put
    scratch loads and stores of the compiler's among them.  The Makefile keeps the compiler's resource-usage remarks
    beside every object; the guard reads them (the library's build runs the same check)."""
    usage = os.path.join(ROOT, "phyai_amd", "csrc", "_obj", "gemm_big.o.usage")
    if not os.path.exists(usage):
        pytest.skip("no resource-usage remarks here (the library was built elsewhere)")
    assert not guard.check_tile_usage(), "\n".join(guard.check_tile_usage()[:20])
    planted = ("x.hip:1:1: remark: Function Name: _ZN5phyai19gemm_fp8_big_kernelILi2ELi2EEEvv [-Rpass-analysis=kernel-resource-usage]\n"
               "x.hip:1:1: remark:     ScratchSize [bytes/lane]: 268 [-Rpass-analysis=kernel-resource-usage]\n"
               "x.hip:1:1: remark: Function Name: _ZN5phyai5otherEv [-Rpass-analysis=kernel-resource-usage]\n"
               "x.hip:1:1: remark:     ScratchSize [bytes/lane]: 16 [-Rpass-analysis=kernel-resource-usage]\n")
    bad = guard.usage_problems(planted, min_kernels=1)
    assert len(bad) == 1 and "268 bytes" in bad[0]
    assert any("only 1" in p for p in guard.usage_problems(planted, min_kernels=2))


def test_copies_keep_their_distance_from_writes_of_their_base(guard):
    """Five wait states between a VALU write of an SGPR and a vector-memory instruction that reads it, in every kernel of
    the built library; the compiler does not see to that in front of inline assembly (the library's build runs the same
    check, of the time-stamp build too)."""
    if not os.path.exists(os.path.join(guard.LIB, "libphyai_fp8.so")) or not os.path.exists(guard.OBJDUMP):
        pytest.skip("no built library or no disassembler here")
    bad = guard.check_library()
    assert not bad, "\n".join(bad[:20])


HEAD = "<_Zkernel>:\n\ts_load_dwordx2 s[4:5], s[0:1], 0x0   // 000000001900: C0060080\n"


@pytest.mark.parametrize("code,found", [
    # in front of a copy: its own two states, four, five; a pointer in the middle of a longer run of SGPRs
    ("v_readlane_b32 s4, v1, 3|s_mov_b32 m0, s6|s_nop 0|global_load_lds_dwordx4 v2, s[4:5]", 2),
    ("v_readlane_b32 s4, v1, 3|v_readlane_b32 s5, v1, 4|v_add_u32_e32 v3, v3, v4|s_mov_b32 m0, s6|s_nop 0|global_load_lds_dword v2, s[4:5]", 3),
    ("v_readfirstlane_b32 s5, v1|s_mov_b32 m0, s6|s_nop 3|global_load_lds_dwordx4 v2, s[4:5]", None),
    ("v_readfirstlane_b32 s6, v1|s_nop 3|buffer_load_dwordx4 v2, s[4:7], s9 offen lds", 4),
    ("v_readfirstlane_b32 s9, v1|s_nop 3|buffer_load_dwordx4 v2, s[4:7], s9 offen lds", 4),
    ("v_readfirstlane_b32 s8, v1|buffer_load_dwordx4 v2, s[4:7], s9 offen lds", None),
    # not a VALU write, or of another register
    ("s_mov_b32 s4, s8|global_load_lds_dwordx4 v2, s[4:5]", None),
    ("v_readlane_b32 s14, v1, 3|global_load_dword v9, v2, s[4:5]", None),
    # a compare, a carry, a second result
    ("v_cmp_lt_u32_e64 s[4:5], v1, v2|global_store_dword v2, v3, s[4:5]", 0),
    ("v_cmp_lt_u32_e32 vcc, v1, v2|s_nop 1|global_store_dword v2, v3, vcc", 2),
    ("v_add_co_u32_e64 v1, s[4:5], v2, v3|global_load_dword v9, v2, s[4:5]", 0),
    # by way of a branch, round a loop, and only on the other arm
    ("v_readlane_b32 s4, v1, 3|s_cbranch_scc0 L0|s_nop 7|<L0>:|global_load_lds_dwordx4 v2, s[4:5]", 1),
    ("<L0>:|global_load_lds_dwordx4 v2, s[4:5]|v_readlane_b32 s5, v1, 3|s_cbranch_vccnz L0", 1),
    ("v_readlane_b32 s4, v1, 3|s_branch L1|<L0>:|global_load_lds_dwordx4 v2, s[4:5]|s_endpgm|<L1>:|s_nop 2|s_cbranch_scc0 L0", None),
    ("v_readlane_b32 s4, v1, 3|s_branch L1|<L0>:|global_load_lds_dwordx4 v2, s[4:5]|s_endpgm|<L1>:|s_nop 1|s_cbranch_scc0 L0", 4),
])
def test_planted_copies_too_close_are_caught(guard, code, found):
    text = HEAD + "".join((t if t.startswith("<") else "\t" + t + "      // 00000000: 0") + "\n" for t in code.split("|")) + "\ts_endpgm   // 0\n"
    bad, functions, _ = guard.check_disassembly(text)
    assert functions == 1
    if found is None:
        assert not bad, bad
    else:
        assert len(bad) == 1 and f"reads an SGPR {found} wait states after" in bad[0], bad
