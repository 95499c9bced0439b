"""Static check of the counted waits on direct global -> LDS loads.

Such a load has no destination register, so no register tells when it has
landed: the wide prefill GEMMs count on `s_waitcnt vmcnt(N)` leaving only
loads outstanding that the following barrier's readers do not need.  Each load
carries what it brings (LoadKind) as a comment in the assembly, and on every path
through the kernel's control flow

  a counted wait leaves no activations, scales or tables outstanding, only
  weights (of a K-block further on, which the next barrier waits for), and
  no global store is issued while activations, scales or tables are outstanding:
  loads and stores share one counter, and the barrier of an item's first step
  does not wait for it (the item's first weights are older than these).

Each weight load stands twice, plain and non-temporal (nt), under one condition
that the compiler turns into two skipped blocks.  One of the two runs: the
check follows the plain one, always, and the numbers of both must agree.

A VGPR spill would add loads and stores of the compiler's own, and is an error.
"""

from __future__ import annotations

import re

import pytest

from test_asm_loads import HIPCC, VMEM_RE, _blocks, _device_asm, _kernels

KIND_RE = re.compile(r"global_load_lds_dword.*; kind (\d)")
NT_RE = re.compile(r"global_load_lds_dword.* nt(\s|$)")
WEIGHTS, ACTIVATIONS, TABLES = "012"
OTHER = "other"
WAIT_RE = re.compile(r"s_waitcnt\b.*vmcnt\((\d+)\)")
MAX_QUEUE = 40  # older entries fold into the last position


def _transfer(state: tuple, block, lines, problems=None) -> tuple:
    """state[k]: what the k-th youngest outstanding vector-memory instruction may be."""
    for i, ins, in_asm in block:
        m = WAIT_RE.match(ins)
        if m:
            n = int(m.group(1))
            left = frozenset().union(*state[:n]) if in_asm else frozenset()
            if problems is not None and left & {ACTIVATIONS, TABLES}:
                problems.append(f"line {i}: {ins} may leave activations or tables outstanding")
            state = state[:n]
        elif NT_RE.match(ins):
            continue
        elif ins.startswith("global_load_lds"):
            kind = KIND_RE.search(lines[i])
            if problems is not None and not kind:
                problems.append(f"line {i}: {ins} does not say what it brings")
            state = (frozenset(kind.group(1) if kind else OTHER),) + state
        elif VMEM_RE.match(ins):
            needed = frozenset().union(*state) & {ACTIVATIONS, TABLES}
            if problems is not None and ins.startswith("global_store") and needed:
                problems.append(f"line {i}: {ins} is issued before loads of the next item's first step have landed")
            if problems is not None and ins.startswith(("scratch_", "buffer_")):
                problems.append(f"line {i}: {ins}: a spill")
            state = (frozenset([OTHER]),) + state
        if len(state) > MAX_QUEUE:
            state = state[:MAX_QUEUE - 1] + (frozenset().union(*state[MAX_QUEUE - 1:]),)
    return state


def _merge(a: tuple, b: tuple) -> tuple:
    n = max(len(a), len(b))
    return tuple((a[k] if k < len(a) else frozenset()) | (b[k] if k < len(b) else frozenset()) for k in range(n))


def _always_plain(blocks, lines):
    """The blocks with the edges taken out that skip a plain weight load: a
    forward branch with, on one side, a block of nothing but such loads and
    scalar instructions keeps that side only."""
    def plain_weights(i, ins):
        kind = KIND_RE.search(lines[i])
        return bool(kind) and kind.group(1) == WEIGHTS and not NT_RE.match(ins)

    def twin(k):
        vector = [(i, ins) for i, ins, _ in blocks[k][0] if not ins.startswith("s_")]
        return bool(vector) and all(plain_weights(i, ins) for i, ins in vector)
    out = []
    for n, (block, succ) in enumerate(blocks):
        keep = [k for k in succ if k > n and twin(k)]
        out.append((block, keep if len(keep) == 1 and len(succ) == 2 else succ))
    return out


def check_lds_loads(lines: list[str]) -> list[str]:
    blocks = _always_plain(_blocks(lines), lines)
    if not blocks:
        return []
    state_in = [None] * len(blocks)
    state_in[0] = ()
    work = [0]
    while work:
        k = work.pop()
        out = _transfer(state_in[k], blocks[k][0], lines)
        for s in blocks[k][1]:
            new = out if state_in[s] is None else _merge(state_in[s], out)
            if new != state_in[s]:
                state_in[s] = new
                work.append(s)
    problems: list[str] = []
    for k, (block, _) in enumerate(blocks):
        if state_in[k] is not None:
            _transfer(state_in[k], block, lines, problems)
    return problems


@pytest.mark.skipif(not HIPCC, reason="hipcc not available")
def test_counted_waits_cover_the_lds_loads():
    asm = _device_asm("prefill_wide.hip")
    kernels = [(name, lines) for name, lines in _kernels(asm) if any("global_load_lds" in line for line in lines)]
    assert len(kernels) == 2
    for name, lines in kernels:
        kinds = {m.group(1) for line in lines if (m := KIND_RE.search(line))}
        assert kinds == {WEIGHTS, ACTIVATIONS, TABLES}
        assert any(WAIT_RE.search(line) and "vmcnt(4)" in line for line in lines)
        loads = [line for line in lines if (m := KIND_RE.search(line)) and m.group(1) == WEIGHTS]
        assert len(loads) == 2 * sum(" nt " in line for line in loads)
        problems = check_lds_loads(lines)
        assert not problems, f"{name}:\n" + "\n".join(problems[:10])
    assert re.findall(r"\.vgpr_spill_count:\s*(\d+)", asm) == ["0", "0"]
    assert all(int(n) <= 256 for n in re.findall(r"\.vgpr_count:\s*(\d+)", asm))
    assert all(int(n) <= 160 * 1024 for n in re.findall(r"\.group_segment_fixed_size:\s*(\d+)", asm))


def _asm(*ins):
    return [line for i in ins for line in (";;#ASMSTART", i, ";;#ASMEND")]


def _load(kind, n=1):
    return _asm(*[f"global_load_lds_dwordx4 v1, s[2:3] ; kind {kind}"] * n)


def test_checker_flags_a_wait_that_leaves_activations():
    wait = _asm("s_waitcnt vmcnt(4) lgkmcnt(0)", "s_barrier")
    assert not check_lds_loads([*_load(ACTIVATIONS, 5), *_load(WEIGHTS, 4), *wait, "s_endpgm"])
    assert check_lds_loads([*_load(ACTIVATIONS, 5), *_load(WEIGHTS, 3), *wait, "s_endpgm"])
    assert check_lds_loads([*_load(WEIGHTS, 4), *_load(ACTIVATIONS, 1), *wait, "s_endpgm"])
    # on one path only: the branch skips a weight load (with work of its own, so no twin of an nt one)
    head, skipped = [*_load(ACTIVATIONS), *_load(WEIGHTS, 3), "s_cbranch_scc1 .LBB0_2"], [*_load(WEIGHTS), ".LBB0_2:"]
    assert check_lds_loads([*head, "v_mov_b32_e32 v9, v1", *skipped, *wait, "s_endpgm"])
    nt = ["s_cbranch_scc0 .LBB0_3", *[i.replace(" ;", " nt ;") for i in _load(WEIGHTS)], ".LBB0_3:"]
    assert not check_lds_loads([*head, *skipped, *nt, *wait, "s_endpgm"])
    # around a loop: the last pass's activations are younger than its weights
    loop = [".LBB0_1:", *_load(WEIGHTS, 4), *_load(ACTIVATIONS), "s_cbranch_scc1 .LBB0_1", *wait, "s_endpgm"]
    assert check_lds_loads(loop)


def test_checker_flags_a_store_before_the_next_item_has_landed():
    store = "global_store_dwordx4 v2, v[4:7], s[4:5]"
    drain = _asm("s_waitcnt vmcnt(4)")
    assert not check_lds_loads([*_load(WEIGHTS, 4), *_load(ACTIVATIONS), *_load(WEIGHTS, 4), *drain, store, "s_endpgm"])
    assert check_lds_loads([*_load(WEIGHTS, 4), *_load(ACTIVATIONS), store, *drain, "s_endpgm"])
    assert check_lds_loads([*_load(TABLES), store, "s_endpgm"])
    assert check_lds_loads(["scratch_store_dword off, v1, s32", "s_endpgm"])
    assert check_lds_loads(_asm("global_load_lds_dword v1, s[2:3]"))
