"""Static check of the scalar operands of inline-assembly memory instructions.

gfx950 needs five wait states between a VALU instruction that writes a
scalar register (v_readlane_b32, with which the compiler reloads a spilled
one, v_readfirstlane_b32, a compare) and a vector-memory instruction that
reads it.  The compiler inserts them for its own instructions and not for
those inside inline assembly, so a reload right before such a load gives it a
stale base address.  Every kernel that issues vector-memory instructions
from inline assembly is checked on every path of its control flow.

M0, the LDS address of a global -> LDS load, must reach such a load as an
operand that the compiler writes: the compiler uses M0 itself, and does not
know of a write inside inline assembly.
"""

from __future__ import annotations

import importlib
import re

import pytest

from test_asm_loads import HIPCC, VMEM_RE, _blocks, _device_asm, _kernels

SREG_RE = re.compile(r"\bs\[(\d+):(\d+)\]|\bs(\d+)\b")
WAIT_STATES = 5


def _sregs(text: str) -> set[int]:
    out = set()
    for m in SREG_RE.finditer(text):
        out.update([int(m.group(3))] if m.group(3) else range(int(m.group(1)), int(m.group(2)) + 1))
    return out


def _step(state: dict, ins: str, in_asm: bool, problems=None, where=0) -> dict:
    """state: scalar register -> wait states since a VALU wrote it (< 5)."""
    op, _, rest = ins.partition(" ")
    if problems is not None and in_asm and VMEM_RE.match(ins):
        for r in _sregs(rest) & state.keys():
            problems.append(f"line {where}: {ins} reads s{r}, written by a VALU {state[r]} wait states before")
    passed = int(rest.strip(), 0) + 1 if op == "s_nop" else 1
    state = {r: a + passed for r, a in state.items() if a + passed < WAIT_STATES}
    if op.startswith("v_"):
        for r in _sregs(rest.split(",")[0]):
            state[r] = 0
    elif op.startswith("s_") and not op.startswith(("s_cmp", "s_cbranch", "s_branch", "s_waitcnt", "s_nop", "s_barrier")):
        for r in _sregs(rest.split(",")[0]):  # rewritten by the scalar unit
            state.pop(r, None)
    return state


def check_scalar_operands(lines: list[str]) -> list[str]:
    blocks = _blocks(lines)
    if not blocks:
        return []
    state_in = [None] * len(blocks)
    state_in[0] = {}
    work = [0]
    while work:
        k = work.pop()
        out = state_in[k]
        for _, ins, in_asm in blocks[k][0]:
            out = _step(out, ins, in_asm)
        for s in blocks[k][1]:
            old = state_in[s]
            new = dict(out) if old is None else {r: min(out.get(r, WAIT_STATES), old.get(r, WAIT_STATES))
                                                 for r in out.keys() | old.keys()}
            if new != old:
                state_in[s] = new
                work.append(s)
    problems: list[str] = []
    for k, (block, _) in enumerate(blocks):
        if state_in[k] is not None:
            st = state_in[k]
            for i, ins, in_asm in block:
                st = _step(st, ins, in_asm, problems, i)
    return problems


def _has_asm_vmem(lines: list[str]) -> bool:
    in_asm = False
    for raw in lines:
        if ";;#ASMSTART" in raw or ";;#ASMEND" in raw:
            in_asm = ";;#ASMSTART" in raw
        elif in_asm and VMEM_RE.match(raw.split(";")[0].strip()):
            return True
    return False


@pytest.mark.skipif(not HIPCC, reason="hipcc not available")
def test_asm_memory_instructions_wait_for_their_scalar_operands():
    b = importlib.import_module("15642_moe_amd.build")
    found = {}
    for source in b.SOURCES:
        found[source] = 0
        for name, lines in _kernels(_device_asm(source)):
            if not _has_asm_vmem(lines):
                continue
            problems = check_scalar_operands(lines)
            assert not problems, f"{source}: {name}:\n" + "\n".join(problems[:10])
            found[source] += 1
    assert found["gemm.hip"] >= 4 and found["upstream.hip"] >= 1 and found["prefill_wide.hip"] >= 2, found


def test_checker_flags_a_reload_before_a_load():
    load = [";;#ASMSTART", "global_load_dwordx4 v[0:3], v8, s[4:5]", ";;#ASMEND"]
    assert check_scalar_operands(["v_readlane_b32 s5, v221, 15", *load])
    assert check_scalar_operands(["v_readlane_b32 s4, v221, 15", "s_nop 3", *load])
    assert not check_scalar_operands(["v_readlane_b32 s4, v221, 15", "s_nop 4", *load])
    assert not check_scalar_operands(["v_readlane_b32 s6, v221, 15", *load])
    assert not check_scalar_operands(["v_readlane_b32 s4, v221, 15", "s_mov_b32 s4, 0", *load])
    assert check_scalar_operands(["v_readlane_b32 s4, v221, 15", "s_cbranch_scc1 .LBB0_2", "s_endpgm", ".LBB0_2:", *load])


def asm_writes_of_m0(lines: list[str]) -> list[str]:
    """Instructions inside inline assembly whose destination is M0."""
    in_asm, found = False, []
    for raw in lines:
        if ";;#ASMSTART" in raw or ";;#ASMEND" in raw:
            in_asm = ";;#ASMSTART" in raw
            continue
        _, _, rest = raw.split(";")[0].strip().partition(" ")
        if in_asm and rest.split(",")[0].strip() == "m0":
            found.append(raw.strip())
    return found


@pytest.mark.skipif(not HIPCC, reason="hipcc not available")
def test_inline_assembly_leaves_m0_to_the_compiler():
    lds_loads = 0
    for name, lines in _kernels(_device_asm("prefill_wide.hip")):
        assert not asm_writes_of_m0(lines), f"{name} writes M0 in inline assembly"
        lds_loads += sum("global_load_lds" in line for line in lines)
    assert lds_loads > 0
    assert asm_writes_of_m0([";;#ASMSTART", "s_mov_b32 m0, s4", ";;#ASMEND"])
    assert not asm_writes_of_m0(["s_mov_b32 m0, s4", ";;#ASMSTART", "s_nop 4", "global_load_lds_dword v1, s[2:3]", ";;#ASMEND"])
