"""The cut of the masked backward's dK/dV work (csrc/bwd_plan.h, built for the host): the partial slots that any counts take
fit the workspace, on devices of any size."""
import ctypes as C
import subprocess
from pathlib import Path

import numpy as np
import pytest

ROOT = Path(__file__).resolve().parent.parent


@pytest.fixture(scope="module")
def plan(tmp_path_factory):
    so = tmp_path_factory.mktemp("bwd_plan") / "harness.so"
    subprocess.run(["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-Wall", f"-I{ROOT / 'abridgekv_amd' / 'csrc'}",
                    str(ROOT / "tests" / "bwd_plan_harness.cpp"), "-o", str(so)], check=True)
    lib = C.CDLL(str(so))
    for f in (lib.layout_bytes, lib.layout_cap, lib.slots):
        f.restype = C.c_long
    return lib


@pytest.mark.parametrize("cus", [4, 32, 64, 256, 304])
def test_parts_fit_the_slots(plan, cus):
    rng = np.random.default_rng(cus)
    for _ in range(3000):
        q_tiles, batch = int(rng.integers(1, 200)), int(rng.integers(1, 5))
        kind = rng.integers(3)
        seen = rng.integers(0, q_tiles + 1, q_tiles * batch)
        if kind == 1:                                        # few long tiles among short ones, as codes among content
            seen = np.where(rng.random(seen.size) < 0.2, seen, np.minimum(seen, 8))
        elif kind == 2:                                      # causal
            seen = np.repeat(q_tiles - np.arange(q_tiles), batch)
        seen = np.ascontiguousarray(seen, np.int32)
        n = plan.slots(seen.ctypes.data_as(C.POINTER(C.c_int32)), seen.size, cus)
        assert n <= plan.layout_cap(batch, 64 * q_tiles, cus)


def test_slots_follow_the_device(plan):
    """Long key tiles are split for the workgroups that a device runs at once: an eighth of the CUs, an eighth of the slots."""
    seen = np.full(2000, 100, np.int32)
    seen[:40] = 2000
    at = seen.ctypes.data_as(C.POINTER(C.c_int32))
    assert plan.slots(at, seen.size, 256) == 0 and plan.slots(at, seen.size, 2048) > 0
    assert plan.layout_cap(1, 128000, 32) == plan.layout_cap(1, 128000, 256) // 8
    row_bytes = 256 * 128000
    assert row_bytes < plan.layout_bytes(1, 128000, 256) < row_bytes + (49 << 20)
