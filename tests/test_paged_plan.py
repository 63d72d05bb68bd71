"""The host plan of a paged multi-query launch: its items cover every key tile of every query tile exactly once."""
import numpy as np
import pytest

from abridgekv_amd import ops


@pytest.mark.parametrize("num_cus", [1, 8, 64, 256])
@pytest.mark.parametrize("seed", range(6))
def test_items_cover_every_tile_once(num_cus, seed):
    rng = np.random.default_rng(seed)
    B = int(rng.integers(1, 12))
    qlen = rng.integers(0, 400, B)
    qs = np.concatenate([[0], np.cumsum(qlen)])
    ks = rng.integers(0, 9000, B)
    causal = rng.integers(0, 2, B)
    kl = np.where(rng.random(B) < 0.2, 0, ks + rng.integers(0, 400, B))
    items, merges, rows = ops.paged_plan(qs, ks, kl, causal, num_cus)
    want = {(r, q0): -(-(min(kl[r], ks[r] + min(q0 + 64, qlen[r])) if causal[r] else kl[r]) // 64)
            for r in range(B) for q0 in range(0, qlen[r], 64)}
    got = {}
    for r, q0, k0, k1, part in items.tolist():
        got.setdefault((r, q0), []).append((k0, k1, part))
    assert set(got) == set(want)
    merged = {int(t): (n, row, parts) for t, n, row, parts in merges.tolist()}
    used = []
    for (r, q0), parts in got.items():
        parts.sort()
        assert parts[0][0] == 0 and parts[-1][1] == want[r, q0]
        assert all(a[1] == b[0] for a, b in zip(parts, parts[1:]))
        token = int(qs[r] + q0)
        if len(parts) == 1:
            assert parts[0][2] == -1 and token not in merged
        else:
            n, row, k = merged.pop(token)
            assert n == min(64, qlen[r] - q0) and k == len(parts)
            assert [p[2] for p in parts] == [row + 64 * i for i in range(k)]
            used += [p[2] for p in parts]
    assert not merged
    assert sorted(used) == list(range(0, rows, 64))
    assert len(used) <= 6 * max(1, num_cus // 8)               # the workspace bound
    lengths = items[:, 3] - items[:, 2]
    assert np.all(np.diff(lengths) <= 0)                       # longest first


def test_empty_batch_and_small_capacity():
    items, merges, rows = ops.paged_plan([0, 0], [5], [5], [1])
    assert len(items) == len(merges) == rows == 0
    from abridgekv_amd._lib import lib
    a = [np.array(x, np.int64) for x in ([0, 256], [9000], [9256], [0])]
    out, sizes = np.empty(9, np.int32), np.zeros(3, np.int32)
    rc = lib().abkv_paged_plan(*(x.ctypes.data for x in a), 1, 256, out.ctypes.data, 1, out.ctypes.data + 20, 1,
                               sizes.ctypes.data)
    assert rc == -5 and sizes[0] > 4
