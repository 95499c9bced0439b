"""The choices of a launch that follow from sizes alone (csrc/plan.h, the code
that the launchers and kernels call), compiled for the CPU."""

from __future__ import annotations

import ctypes
import shutil
import subprocess
from pathlib import Path

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
