"""fp32 mode of the attention paths vs the float64 oracle (tolerance: max-abs <= 1e-5 for outputs and LSE)."""
import numpy as np
import pytest
import torch

from oracle import decode as od
from oracle import masks as om
from oracle import prefill as op

pytestmark = pytest.mark.gpu
TOL = 1e-5


def _paged(lens, num_pages, seed):
    rng = np.random.default_rng(seed)
    need = [-(-n // 16) for n in lens]
    perm = rng.permutation(np.arange(1, num_pages))
    tables = np.zeros((len(lens), max(max(need), 1)), np.int32)
    at = 0
    for r, n in enumerate(need):
        tables[r, :n] = perm[at: at + n]
        at += n
    g = torch.Generator().manual_seed(seed)
    cache = torch.randn((num_pages, 2, 16, 8, 128), generator=g, dtype=torch.float32)
    return cache, tables


def test_decode_f32_matches_fp64():
    from abridgekv_amd import ops
    lens = [1, 17, 300, 1068, 2999, 0]
    cache, tables = _paged(lens, 600, 0)
    g = torch.Generator().manual_seed(1)
    q = torch.randn((len(lens), 32, 128), generator=g, dtype=torch.float32)
    dev = torch.device("cuda")
    lse = torch.empty((len(lens), 32), dtype=torch.float32, device=dev)
    out, _ = ops.decode_attention(q.to(dev), cache.to(dev), torch.from_numpy(tables).to(dev),
                                  torch.tensor(lens, dtype=torch.int32, device=dev), 128 ** -0.5, lse=lse)
    torch.cuda.synchronize()
    assert out.dtype == torch.float32
    ref_o, ref_l = od.decode_paged_fp64(q.numpy(), cache.numpy(), tables, lens, 128 ** -0.5)
    got_o, got_l = out.cpu().numpy(), lse.cpu().numpy()
    assert np.abs(got_o - ref_o).max() <= TOL
    live = np.asarray(lens) > 0
    assert np.abs(got_l[live] - ref_l[live]).max() <= TOL
    assert np.all(np.isneginf(got_l[~live])) and np.all(got_o[~live] == 0)


@pytest.mark.parametrize("tail", [0, 40])
def test_paged_multi_query_f32_code_step_and_chunks(tail):
    """fp32 code step (key limit code start + quota; with a static tail, the block's last rows before the codes
    excluded: the reference's mask with its excluded range, compresslm_masks.py:206-213) and causal chunks."""
    from abridgekv_amd import ops
    quota, K = 64, 128
    reqs = [(K, 500 + K, (500, 500 + K)), (90, 90 + 200, None), (1, 777, None)]
    excluded = [(500 - tail, 500) if tail and span else None for _, _, span in reqs]
    cache, tables = _paged([sl for _, sl, _ in reqs], 300, 2)
    qsl = np.concatenate([[0], np.cumsum([r[0] for r in reqs])])
    g = torch.Generator().manual_seed(3)
    q = torch.randn((int(qsl[-1]), 32, 128), generator=g, dtype=torch.float32)
    sls = [r[1] for r in reqs]
    kv_start = [sl - ql for ql, sl, _ in reqs]
    limits = [sl if span is None else span[0] + quota for _, sl, span in reqs]
    causal = [span is None for _, _, span in reqs]
    dev = torch.device("cuda")
    lse = torch.empty((int(qsl[-1]), 32), dtype=torch.float32, device=dev)
    out, _ = ops.paged_prefill_attention(q.to(dev), cache.to(dev), torch.from_numpy(tables).to(dev), qsl, kv_start,
                                         limits, causal, lse=lse, excluded=excluded if tail else None)
    torch.cuda.synchronize()
    got_o, got_l = out.cpu().numpy(), lse.cpu().numpy()
    cf = cache.numpy()
    for r, (ql, sl, span) in enumerate(reqs):
        m = om.request_mask(ql, sl, [span] if span else [], excluded[r], quota, K, causal=span is None)
        ro, rl = om.masked_paged_attention_fp64(q[qsl[r]: qsl[r + 1]].numpy(), cf, tables[r], sl, m, 128 ** -0.5)
        assert np.abs(got_o[qsl[r]: qsl[r + 1]] - ro).max() <= TOL, f"request {r}"
        assert np.abs(got_l[qsl[r]: qsl[r + 1]] - rl).max() <= TOL, f"request {r}"


@pytest.mark.parametrize("prompt_len,quota,tail,policy", [(None, None, 0, "static"), ([40, 150], None, 0, "static"),
                                                           ([0, 70], "mixed", 0, "static"),
                                                           ([40, 0], "mixed", 12, "static"),
                                                           ([40, 0], "mixed", 12, "rolling"),
                                                           ([70, 0], "mixed", 20, "sticky"),
                                                           ([70, 0], "mixed", 20, "causal-codes"),
                                                           ([40, 0], "mixed", 12, "two-passes"),
                                                           (None, "mixed", 0, "copy-region"),
                                                           (None, None, 0, "no-codes"),
                                                           ([40, 0], "mixed", 0, "replay"),
                                                           ([40, 0], "mixed", 12, "raw"),
                                                           ([40, 0], "mixed", 64, "raw")])
def test_masked_prefill_f32_matches_fp64(prompt_len, quota, tail, policy):
    from abridgekv_amd import ops
    xattn = "causal" if policy == "causal-codes" else "full"
    L = 2 if policy in ("two-passes", "copy-region") else 1
    cr = 65 if policy == "copy-region" else 0
    K = 0 if policy == "no-codes" else 16
    R = 12 if policy == "replay" else 0
    policy = "static" if policy in ("causal-codes", "two-passes", "copy-region", "no-codes", "replay") else policy
    C, N, B = 64, 4, 2
    S0 = N * (C + L * K + R) + cr
    head_quota = None if quota is None else [1 + (h * 5) % max(K, 1) for h in range(32)]
    g = torch.Generator().manual_seed(7)
    q = torch.randn((B, S0, 32, 128), generator=g, dtype=torch.float32)
    k = torch.randn((B, S0, 8, 128), generator=g, dtype=torch.float32)
    v = torch.randn((B, S0, 8, 128), generator=g, dtype=torch.float32)
    dev = torch.device("cuda")
    pl = None if prompt_len is None else torch.tensor(prompt_len, dtype=torch.int32, device=dev)
    hq = None if head_quota is None else torch.tensor(head_quota, dtype=torch.int32, device=dev)
    lse = torch.empty((B, 32, S0), dtype=torch.float32, device=dev)
    out, _ = ops.prefill_masked_attention(q.to(dev), k.to(dev), v.to(dev), C, K, N, prompt_len=pl, head_quota=hq,
                                          lse=lse, retain_tail=tail, tail_policy=policy, pause_xattn=xattn,
                                          pause_passes=L, copy_rows=cr, replay_rows=R, replay_exclude=R > 0)
    torch.cuda.synchronize()
    got_o, got_l = out.cpu().numpy(), lse.cpu().numpy()
    for b in range(B):
        raw = policy == "raw"                   # the kernels' raw policy is the oracle's separate raw-tail term
        mask = op.arith_mask(C, K, N, None if prompt_len is None else [prompt_len[b]], head_quota,
                             retain_tail=0 if raw else tail, tail_policy="static" if raw else policy,
                             pause_xattn=xattn, passes=L, copy_rows=cr, replay=R, replay_exclude=R > 0,
                             raw_tail=tail if raw else 0)
        if prompt_len is not None:
            mask = mask[0]
        ro, rl = op.masked_attention_fp64(q[b].numpy(), k[b].numpy(), v[b].numpy(), mask, 128 ** -0.5)
        assert np.abs(got_o[b] - ro).max() <= TOL
        assert np.abs(got_l[b].T - rl).max() <= TOL


def test_decode_f32_page_and_wave_edges():
    """Row counts around one page, the eight pages that the workgroup's waves start with, and their second turn.
    Tolerance: fp32 sums of 128 products and up to 300 weights, under 1e-5 with |out| <= 5."""
    from abridgekv_amd import ops
    lens = [1, 15, 16, 17, 127, 128, 129, 144, 256, 257, 300]
    cache, tables = _paged(lens, 200, 20)
    g = torch.Generator().manual_seed(21)
    q = 2.5 * torch.randn((len(lens), 32, 128), generator=g, dtype=torch.float32)
    dev = torch.device("cuda")
    lse = torch.empty((len(lens), 32), dtype=torch.float32, device=dev)
    out, _ = ops.decode_attention(q.to(dev), cache.to(dev), torch.from_numpy(tables).to(dev),
                                  torch.tensor(lens, dtype=torch.int32, device=dev), 128 ** -0.5, lse=lse)
    ref_o, ref_l = od.decode_paged_fp64(q.numpy(), cache.numpy(), tables, lens, 128 ** -0.5)
    assert np.abs(out.cpu().numpy() - ref_o).max() <= TOL
    assert np.abs(lse.cpu().numpy() - ref_l).max() <= TOL


@pytest.mark.parametrize("causal", [True, False])
def test_paged_f32_tiles_with_rows_of_several_requests(causal):
    """16-row tiles that hold rows of one to six requests, key ranges around the 32-key stages, a request without
    keys. Tolerance as above."""
    from abridgekv_amd import ops
    qlen = [1, 5, 16, 3, 33, 1, 1, 2, 15]
    past = [31, 27, 16, 0, 64, 32, 300, 30, 1]
    sls = [a + b for a, b in zip(qlen, past)]
    limits = [sl if causal else max(0, sl - 1) for sl in sls]
    cache, tables = _paged(sls, 120, 22)
    qsl = np.concatenate([[0], np.cumsum(qlen)])
    if not causal:
        limits[6] = 0
    g = torch.Generator().manual_seed(23)
    q = torch.randn((int(qsl[-1]), 32, 128), generator=g, dtype=torch.float32)
    dev = torch.device("cuda")
    lse = torch.empty((int(qsl[-1]), 32), dtype=torch.float32, device=dev)
    out, _ = ops.paged_prefill_attention(q.to(dev), cache.to(dev), torch.from_numpy(tables).to(dev), qsl, past,
                                         limits, causal, lse=lse)
    got_o, got_l = out.cpu().numpy(), lse.cpu().numpy()
    for r, sl in enumerate(sls):
        a, z = qsl[r], qsl[r + 1]
        if limits[r] == 0:
            assert np.all(got_o[a:z] == 0) and np.all(np.isneginf(got_l[a:z]))
            continue
        k, v = od.paged_rows(cache.numpy(), tables[r], limits[r])
        for i in range(qlen[r]):
            n = min(limits[r], past[r] + i + 1) if causal else limits[r]
            ro, rl = od.decode_fp64(q[a + i].numpy(), k[:n], v[:n], 128 ** -0.5)
            assert np.abs(got_o[a + i] - ro).max() <= TOL, f"request {r} row {i}"
            assert np.abs(got_l[a + i] - rl).max() <= TOL, f"request {r} row {i}"


def _bits(x):
    return x.cpu().numpy().view(np.uint32)


@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
def test_paged_f32_infinite_values_reach_only_the_rows_that_see_them(bad):
    """V elements of one late token of a causal chunk, and of a range hidden by `excluded`, infinite or NaN: rows that do
    not see the token keep every bit, rows that do get it in that head's dims alone (inf with the weight's sign, NaN)."""
    from abridgekv_amd import ops
    dev = torch.device("cuda")
    cache, tables = _paged([200, 90], 60, 30)
    g = torch.Generator().manual_seed(31)
    q = torch.randn((40 + 20, 32, 128), generator=g, dtype=torch.float32).to(dev)
    bt = torch.from_numpy(tables).to(dev)

    def call(c):
        return ops.paged_prefill_attention(q, c.to(dev), bt, [0, 40, 60], [160, 60], [200, 80], [True, False],
                                           excluded=[None, (33, 50)])[0]
    clean = call(cache)
    dirty = cache.clone()
    pos, hid = 160 + 21, 40                                  # row 21's own key; a hidden key of the second request
    dirty[tables[0, pos // 16], 1, pos % 16, 3, [0, 77]] = bad
    dirty[tables[0, 50 // 16], 1, 50 % 16, 6, 5] = -bad       # a key that every row of the chunk sees
    dirty[tables[1, hid // 16], 1, hid % 16] = bad
    got = call(dirty)
    want = clean.clone()
    want[21:40, 12:16, 0] = want[21:40, 12:16, 77] = bad
    want[:40, 24:28, 5] = -bad
    assert torch.equal(torch.isnan(got), torch.isnan(want))
    assert np.array_equal(_bits(got.nan_to_num(nan=7.0)), _bits(want.nan_to_num(nan=7.0)))


@pytest.mark.parametrize("K", [16, 0])
def test_masked_f32_infinite_values_reach_only_the_rows_that_see_them(K):
    """The same under the compression mask: content of block 0 is hidden from later blocks, a row's later keys from it."""
    from abridgekv_amd import ops
    dev = torch.device("cuda")
    C, N = 40, 3
    S = N * (C + K)
    g = torch.Generator().manual_seed(32)
    q, k, v = (torch.randn((1, S, h, 128), generator=g, dtype=torch.float32).to(dev) for h in (32, 8, 8))
    clean = ops.prefill_masked_attention(q, k, v, C, K, N)[0]
    bad = v.clone()
    bad[0, 13, 2, 9] = float("inf")
    got = ops.prefill_masked_attention(q, k, bad, C, K, N)[0]
    sees = torch.from_numpy(np.asarray(op.arith_mask(C, K, N, None, None))).reshape(-1, S, S)[0, :, 13].to(dev)
    want = clean.clone()
    want[0, sees, 8:12, 9] = float("inf")
    assert 0 < int(sees.sum()) < S - 13
    assert np.array_equal(_bits(got), _bits(want))


def test_decode_f32_passes_nan_and_infinities_on():
    """A NaN key makes its head's outputs NaN; an infinite V element of a sequence's last row, whose page is partly
    filled, makes that dim infinite and nothing else."""
    from abridgekv_amd import ops
    dev = torch.device("cuda")
    lens = [37, 200]
    cache, tables = _paged(lens, 40, 33)
    q = torch.randn((2, 32, 128), generator=torch.Generator().manual_seed(34), dtype=torch.float32).to(dev)

    def call(c):
        return ops.decode_attention(q, c.to(dev), torch.from_numpy(tables).to(dev),
                                    torch.tensor(lens, dtype=torch.int32, device=dev), 128 ** -0.5)[0]
    want = call(cache)
    bad = cache.clone()
    bad[tables[0, 36 // 16], 1, 36 % 16, 1, 100] = float("inf")
    bad[tables[1, 150 // 16], 0, 150 % 16, 5, 3] = float("nan")
    got = call(bad)
    want[0, 4:8, 100] = float("inf")
    want[1, 20:24] = float("nan")
    assert torch.equal(torch.isnan(got), torch.isnan(want))
    assert np.array_equal(_bits(got.nan_to_num(nan=7.0)), _bits(want.nan_to_num(nan=7.0)))


@pytest.mark.parametrize("rows", [[1, 2, 3, 4, 5], [1], [4, 17]])
@pytest.mark.parametrize("requests", [9, 210])
def test_paged_f32_many_short_requests(rows, requests):
    """Windows with up to sixteen requests, few of them (a workgroup per request) and many; rows at both sides of the
    four that share a workgroup's columns; excluded ranges. Tolerance as above."""
    from abridgekv_amd import ops
    qlen = [rows[i % len(rows)] for i in range(requests)]
    past = [(11 * i) % 70 for i in range(requests)]
    sls = [a + b for a, b in zip(qlen, past)]
    excluded = [(5, 9) if p > 20 else None for p in past]
    cache, tables = _paged(sls, 2000, 40)
    qsl = np.concatenate([[0], np.cumsum(qlen)])
    q = torch.randn((int(qsl[-1]), 32, 128), generator=torch.Generator().manual_seed(41), dtype=torch.float32)
    dev = torch.device("cuda")
    lse = torch.empty((int(qsl[-1]), 32), dtype=torch.float32, device=dev)
    out, _ = ops.paged_prefill_attention(q.to(dev), cache.to(dev), torch.from_numpy(tables).to(dev), qsl, past, sls, True,
                                         lse=lse, excluded=excluded)
    got_o, got_l = out.cpu().numpy(), lse.cpu().numpy()
    for r, sl in enumerate(sls):
        k, v = od.paged_rows(cache.numpy(), tables[r], sl)
        for i in range(qlen[r]):
            keep = np.arange(past[r] + i + 1)
            if excluded[r]:
                keep = keep[(keep < 5) | (keep >= 9)]
            ro, rl = od.decode_fp64(q[qsl[r] + i].numpy(), k[keep], v[keep], 128 ** -0.5)
            assert np.abs(got_o[qsl[r] + i] - ro).max() <= TOL, f"request {r} row {i}"
            assert np.abs(got_l[qsl[r] + i] - rl).max() <= TOL, f"request {r} row {i}"


def test_paged_f32_infinite_values_in_a_short_chunk():
    """Three rows that share a workgroup's columns, the last one's own V row infinite in one dim: nothing else changes
    but the order of the sums (the tile is walked again, a head per wave)."""
    from abridgekv_amd import ops
    dev = torch.device("cuda")
    cache, tables = _paged([100], 20, 50)
    q = torch.randn((3, 32, 128), generator=torch.Generator().manual_seed(51), dtype=torch.float32).to(dev)
    bt = torch.from_numpy(tables).to(dev)
    clean = ops.paged_prefill_attention(q, cache.to(dev), bt, [0, 3], [97], [100], True)[0]
    cache[tables[0, 99 // 16], 1, 99 % 16, 2, 50] = float("inf")
    got = ops.paged_prefill_attention(q, cache.to(dev), bt, [0, 3], [97], [100], True)[0]
    assert torch.isinf(got[2, 8:12, 50]).all()
    got[2, 8:12, 50] = clean[2, 8:12, 50]
    assert (got - clean).abs().max() <= TOL
