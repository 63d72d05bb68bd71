"""The key-tile walk, the per-row key ranges and the per-key query ranges of the masked kernels (csrc/mask_walk.h, built for the host) against the
compression mask: every visible (query, key) pair is covered exactly once, no hidden one ever, over the block layouts,
tails, replay rows, passes, copy rows, prompts and quotas that the kernels take."""
import ctypes as C
import random
import subprocess
from pathlib import Path

import numpy as np
import pytest

from oracle import prefill as op

ROOT = Path(__file__).resolve().parent.parent
POLICIES = ("static", "rolling", "sticky", "raw")
XATTN = ("full", "causal", "none")


@pytest.fixture(scope="module")
def harness(tmp_path_factory):
    so = tmp_path_factory.mktemp("mask_walk") / "harness.so"
    subprocess.run(["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-Wall", f"-I{ROOT / 'abridgekv_amd' / 'csrc'}",
                    str(ROOT / "tests" / "mask_walk_harness.cpp"), "-o", str(so)], check=True)
    lib = C.CDLL(str(so))
    lib.walk_counts.restype = C.c_long
    return lib


def _params(c):
    return (C.c_int32 * 10)(c["C"], c["K"], c["N"], c["L"], c["R"], c["copy"], c["tail"], POLICIES.index(c["policy"]),
                            XATTN.index(c["xattn"]), int(c["rx"]))


def _case(**kw):
    return {**dict(C=128, K=64, N=3, L=1, R=0, copy=0, tail=0, policy="static", xattn="full", rx=False, plen=0,
                   quota=None), **kw}


def _mask(c, quota):
    """bool [4, S, S]: the mask of four query heads."""
    raw = c["policy"] == "raw"
    S = c["N"] * (c["C"] + c["L"] * c["K"] + c["R"]) + c["copy"]
    m = op.arith_mask(c["C"], c["K"], c["N"], [c["plen"]], [quota[u % 4] for u in range(32)],
                      retain_tail=0 if raw else c["tail"], tail_policy="static" if raw else c["policy"],
                      pause_xattn=c["xattn"], passes=c["L"], copy_rows=c["copy"], replay=c["R"],
                      replay_exclude=c["rx"], raw_tail=c["tail"] if raw else 0)
    m = np.asarray(m)
    m = m.reshape(-1, S, S)
    return np.stack([m[u if m.shape[0] > 1 else 0] for u in range(4)])


def _random(rng):
    c = _case(C=rng.choice([8, 33, 64, 100, 128, 200, 256]), K=rng.choice([0, 1, 4, 16, 40, 64, 100, 128]),
              N=rng.randint(1, 5))
    if c["K"]:
        c["K"] = min(c["K"], c["C"])
        c["L"] = rng.choice([1, 1, 1, 2, 3])
        c["xattn"] = rng.choice(["full", "full", "causal", "none"])
        c["copy"] = rng.choice([0, 0, 0, 1, 30, 64, 150, 500])
        if rng.random() < 0.4:
            c["R"] = rng.randint(1, min(c["C"], 70))
            c["rx"] = c["R"] < c["C"] and rng.random() < 0.5
    if not c["R"] and rng.random() < 0.6:
        c["policy"] = rng.choice(POLICIES)
        c["tail"] = rng.randint(0, c["C"] - (c["policy"] != "raw"))
    if rng.random() < 0.5:
        c["plen"] = rng.randint(0, (c["N"] + 1) * c["C"])
    c["quota"] = [rng.randint(0, c["K"] + 1) for _ in range(4)] if rng.random() < 0.5 else None
    return c


CASES = [_case(), _case(C=64, K=0, N=1), _case(C=100, K=0, N=3, plen=130), _case(C=512, K=128, N=2, R=16),
         _case(C=512, K=128, N=2, R=16, rx=True, plen=600), _case(C=200, K=40, N=4, tail=32, policy="rolling"),
         _case(C=200, K=40, N=4, tail=200, policy="raw"), _case(C=128, K=64, N=3, L=2, xattn="causal", copy=100),
         _case(C=8, K=4, N=9, quota=[4, 1, 2, 3], plen=13)]


@pytest.mark.parametrize("rows", [64, 16])                     # query tiles of the bf16 and of the fp32 kernels
@pytest.mark.parametrize("case", CASES + [_random(random.Random(s)) for s in range(140)], ids=str)
def test_walk_covers_the_mask_once(harness, case, rows):
    quota = case["quota"] or [case["K"]] * 4
    S = case["N"] * (case["C"] + case["L"] * case["K"] + case["R"]) + case["copy"]
    counts = np.zeros((4, S, S), np.uint8)
    n = harness.walk_counts(_params(case), case["plen"], (C.c_int32 * 4)(*quota), rows,
                            counts.ctypes.data_as(C.POINTER(C.c_uint8)))
    assert n >= 0
    mask = _mask(case, quota)
    bad = np.argwhere(counts != mask)
    assert bad.size == 0, (bad[:5].tolist(), len(bad))
    if rows != 64:                                           # (the query ranges per key do not depend on it)
        return
    counts[:] = 0
    harness.key_counts(_params(case), case["plen"], (C.c_int32 * 4)(*quota),
                       counts.ctypes.data_as(C.POINTER(C.c_uint8)))
    bad = np.argwhere(counts != mask)
    assert bad.size == 0, (bad[:5].tolist(), len(bad))
