"""The choices of a launch that follow from sizes alone (csrc/plan.h, the code
that the launchers and kernels call), compiled for the CPU."""

from __future__ import annotations

import ctypes
import shutil
import subprocess
from pathlib import Path

import numpy as np
import pytest

from conftest import REPO

CSRC = REPO / "15642_moe_amd" / "csrc"


def build_plan(out_dir: Path) -> ctypes.CDLL:
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ not found")
    so = out_dir / "plan_host.so"
    subprocess.run([gxx, "-O1", "-std=c++17", "-Wall", "-Werror", "-shared", "-fPIC", f"-I{CSRC}",
                    str(REPO / "tests" / "plan_host.cpp"), "-o", str(so)], check=True)
    return ctypes.CDLL(str(so))


def wide_tile(plan, counts, nblk, workgroups=256) -> int:
    """The tile size, in 32-route fragments, of a wide prefill GEMM (nblk 16: GEMM1, 28: GEMM2)."""
    return plan.plan_wide_tile((ctypes.c_int * len(counts))(*counts), len(counts), nblk, workgroups)


@pytest.fixture(scope="module")
def plan(tmp_path_factory):
    return build_plan(tmp_path_factory.mktemp("plan"))


@pytest.mark.parametrize("T,waves", [
    (960, 4), (961, 8), (1024, 8), (1025, 4), (1536, 4), (1537, 16), (2048, 16), (2049, 4), (2198, 4), (2560, 4), (2561, 8), (3072, 8), (3073, 16), (3222, 16),
    (3520, 16), (3521, 8), (4096, 8), (4097, 4), (5632, 4), (5633, 16), (7104, 16), (7105, 8), (8192, 8), (8193, 4),
    (16384, 16), (16385, 4)])
def test_router_waves_on_256_cus(plan, T, waves):
    """The measured choice either side of each switch: a workgroup of 16 or 8
    waves has a CU to itself, and a token tile's workgroups share an XCD, so the
    rounds are those of the XCD with the most tiles."""
    assert plan.plan_router_waves(T, 256) == waves


@pytest.mark.parametrize("cus", [256, 128, 64, 32, 8, 1])
def test_router_waves_fill_their_rounds(plan, cus):
    """For any size and CU count: more than four waves only where the busiest
    XCD's CUs are at least 7/10 busy over its rounds."""
    per_xcd = max(cus // 8, 1)
    for T in list(range(1, 20000, 37)) + [1 << 15, 1 << 18]:
        waves, parts = plan.plan_router_waves(T, cus), plan.plan_router_k_parts(T)
        assert waves in (4, 8, 16) and (waves == 4 or parts < 14)
        groups = 16 // waves * -(-(-(-T // 64)) // 8) * parts
        if waves > 4:
            assert groups >= 0.7 * per_xcd * -(-groups // per_xcd)


@pytest.mark.parametrize("T,e_local,waves", [
    (1, 32, 4), (64, 16, 4), (65, 16, 1), (128, 16, 1), (65, 13, 4), (65, 14, 1), (128, 18, 1), (128, 19, 4),
    (128, 32, 4), (128, 8, 4), (2, 16, 4)])
def test_stage2_decode_waves_on_256_cus(plan, T, e_local, waves):
    """One wave per decode GEMM2 item where the items fill one round of single
    waves: more than 6 and at most 8 per CU."""
    assert plan.plan_stage2_decode_waves(T, e_local, 256) == waves


@pytest.mark.parametrize("T,e_local,wide", [
    (3071, 32, 0), (3072, 32, 1), (3071, 17, 0), (3072, 17, 1), (3072, 16, 0), (3200, 16, 0), (3455, 16, 0),
    (3456, 16, 1), (16384, 16, 1), (3456, 15, 0), (16384, 8, 0), (129, 32, 0)])
def test_prefill_wide_on_256_cus(plan, T, e_local, wide):
    """The wide kernels' line: later where an item per weight block is at most
    one per CU."""
    assert plan.plan_prefill_wide(T, e_local, 256) == wide


@pytest.mark.parametrize("counts,gemm1,gemm2", [
    ([0] * 16, 8, 8),
    # one busy expert: cut as fine as there are workgroups for
    ([512] + [0] * 15, 2, 2), ([768] + [0] * 15, 2, 3), ([1024] + [0] * 15, 2, 4), ([1536] + [0] * 15, 3, 6),
    ([2048] + [0] * 15, 4, 8), ([3072] + [0] * 15, 6, 6),
    # more items than workgroups with tiles of four fragments: no finer, though three and two fill the last round
    ([96] * 10 + [128] * 10, 8, 8), ([105] * 18, 8, 8),
    ([128] * 32, 8, 8), ([288] * 12 + [256] * 4, 6, 6)])
def test_wide_tile_size(plan, counts, gemm1, gemm2):
    assert (wide_tile(plan, counts, 16), wide_tile(plan, counts, 28)) == (gemm1, gemm2)


@pytest.mark.parametrize("seed", range(24))
def test_wide_items_cover_every_tile_once(plan, seed):
    """The items of the kernels' own arithmetic: for any route counts, each
    (expert, weight block) has its routes dealt to items once, in whole
    fragments, and none holds more than the tile size; an expert's blocks lie
    in quads on different queues."""
    rng = np.random.default_rng(seed)
    e_local = int(rng.integers(1, 33))
    counts = [int(c) for c in rng.choice([0, 1, 31, 32, 33, 255, 256, 257, 513, 2304, 2305, 4096], size=e_local)]
    for nblk in (16, 28):
        for tile in {8, 6, 4, 3, 2, wide_tile(plan, counts, nblk)}:
            room = 2 * nblk * (sum(counts) // 32 + 33)
            buf = np.zeros((room, 5), dtype=np.int32)
            n = plan.plan_wide_items((ctypes.c_int * e_local)(*counts), e_local, nblk, tile,
                                     buf.ctypes.data_as(ctypes.POINTER(ctypes.c_int)), room)
            assert n >= 0
            spans: dict = {}
            for x, e, blk, first, rows in buf[:n].tolist():
                assert 0 <= e < e_local and 0 <= blk < nblk and 0 < rows <= 32 * tile and first % 32 == 0
                spans.setdefault((e, blk), []).append((first, rows, x))
            assert set(spans) == {(e, b) for e in range(e_local) if counts[e] for b in range(nblk)}
            for (e, blk), got in spans.items():
                at = 0
                for first, rows, x in sorted(got):
                    assert first == at and x == got[0][2]
                    at += rows
                assert at == counts[e]
            for e in range(e_local):
                if counts[e]:
                    queue_of = [spans[e, 4 * j][0][2] for j in range(nblk // 4)]
                    assert len(set(queue_of)) == nblk // 4
                    assert all(spans[e, b][0][2] == queue_of[b // 4] for b in range(nblk))
