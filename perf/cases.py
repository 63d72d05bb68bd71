"""The performance cases of the abridged-KV attention path: what a serving worker, a trainer or an evaluator calls
per layer, through the public entry points, with inputs made from a seed.

A case is a dict of plain values; ``kind`` names the call:

  decode   one layer of a decode step over the group's paged cache (``ops.decode_attention``), bf16 or fp32
  packed   the same with per-head packed code pages beside the paged rows (``ops.decode_attention_packed``)
  code     a code step: the code rows of closing blocks attend their request's rows (``ops.paged_prefill_attention``)
  step     one layer of a mixed serving step through the attention backend: KV append, decodes, prompt chunks and a
           code step in one batch (``AbridgeAttentionImpl.forward``)
  rope     rotary embedding + KV append of a step's new rows, slots from the page table (``ops.slot_mapping``,
           ``ops.rope_kv_append``)
  moves    the row moves of a compaction step over the shared layer tensors (``worker.launch_moves``)
  masked   teacher-forced attention under the compression mask through the attention function the models register
           (``compress_forward.masked_attention_forward``), forward only or with its gradients, bf16 or fp32

Geometry (32 query heads, 8 KV heads, head size 128, pages of 16 rows) is the kernels' own. Lengths inside a batch
are spread over the case's range in an order fixed by the case, so that every seed has the same amount of work.
"""
from __future__ import annotations

import math
import types

import numpy as np
import torch

from abridgekv_amd import ops, worker, workloads
from abridgekv_amd.backend import NOT_CODE, AbridgeAttentionImpl, AbridgeMetadataBuilder
from abridgekv_amd.compress_forward import CompressMask, masked_attention_forward

HQ, HKV, D, PAGE = 32, 8, 128, 16
G = HQ // HKV
SCALE = 1.0 / math.sqrt(D)

# per-head code quotas with mean 128 of 256 code rows, and a narrow set whose pages hold few rows per head
HEAD_QUOTAS = {"wide": (32, 64, 96, 128, 128, 160, 192, 224), "narrow": (8, 16, 24, 32, 32, 40, 48, 56),
               "even": (128,) * 8}


def listed():
    return [
        # one request decoding alone: 256 prompt rows, four closed blocks of 128 codes, an open block (latency bound)
        {"name": "decode_1", "kind": "decode", "dtype": "bf16", "B": 1, "rows_min": 1068, "rows_max": 1068},
        # full-model decode at batch 64: 512-token prompt, 33 closed blocks of 128 codes, an open block of 1..511 rows
        {"name": "decode_64", "kind": "decode", "dtype": "bf16", "B": 64, "rows_min": 4737, "rows_max": 5247},
        # saturated serving: 256 requests of 2K..32K tokens of context, compacted to 128 rows per closed block
        {"name": "decode_256", "kind": "decode", "dtype": "bf16", "B": 256, "rows_min": 900, "rows_max": 9500},
        # a served model with one quota per head: most of the context lives in packed pages
        {"name": "packed_64", "kind": "packed", "B": 64, "rows_min": 513, "rows_max": 1023, "pages_min": 30,
         "pages_max": 42, "quotas": "wide"},
        # one request closes its block: 256 code rows over its compacted context
        {"name": "code_step_1", "kind": "code", "R": 1, "K": 256, "quota": 128, "before_min": 5200,
         "before_max": 5200, "tail": 0, "dtype": "bf16"},
        # a serving step with arrivals: 24 decodes, two prompt chunks and one code step
        {"name": "step_mixed", "kind": "step", "decodes": 24, "rows_min": 700, "rows_max": 5200, "chunks": 2,
         "chunk_min": 300, "chunk_max": 512, "past_min": 0, "past_max": 1536, "codes": 1, "K": 256, "quota": 128},
        # the new rows of a 256-request decode step
        {"name": "rope_256", "kind": "rope", "T": 256, "per_request": 1, "codes_k": 256, "prompt": False},
        # sixteen requests closed a block in this step; six layer tensors shared by six groups
        {"name": "compact_16", "kind": "moves", "B": 16, "max_prior_blocks": 3},
        # teacher-forced forward: 8192 content tokens a sequence, the first block raw prompt (evaluation, no gradients)
        {"name": "masked_eval", "kind": "masked", "dtype": "bf16", "grad": False, "B": 4, "N": 16, "C": 512, "K": 128,
         "L": 1, "R": 0, "rx": False, "tail": 0, "policy": "static", "xattn": "full", "prompt": 512,
         "head_quota": False},
        # the same attention in float32, as a parity run of a model in float32 uses it
        {"name": "masked_eval_f32", "kind": "masked", "dtype": "f32", "grad": False, "B": 1, "N": 3, "C": 512,
         "K": 128, "L": 1, "R": 0, "rx": False, "tail": 0, "policy": "static", "xattn": "full", "prompt": 200,
         "head_quota": False},
        # a training step's attention on the aligned layout: forward and gradients
        {"name": "train_codes", "kind": "masked", "dtype": "bf16", "grad": True, "B": 2, "N": 12, "C": 512, "K": 128,
         "L": 1, "R": 0, "rx": False, "tail": 0, "policy": "static", "xattn": "full", "prompt": 512,
         "head_quota": False},
        # a training step with the replay tail of 16 rows that the configuration has by default
        {"name": "train_replay", "kind": "masked", "dtype": "bf16", "grad": True, "B": 1, "N": 8, "C": 512, "K": 128,
         "L": 1, "R": 16, "rx": False, "tail": 0, "policy": "static", "xattn": "full", "prompt": 0,
         "head_quota": False},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "packed", "code", "step", "rope", "moves", "masked", "masked", "masked"])
    if kind == "decode":
        B = _log(rng, 1, 256)
        hi = _log(rng, 17, 9500)
        lo = rng.randint(max(1, hi // 10), hi)
        f32 = rng.random() < 0.2
        if f32:
            B = min(B, 32)
        return {"kind": kind, "dtype": "f32" if f32 else "bf16", "B": B, "rows_min": lo, "rows_max": hi}
    if kind == "packed":
        lo, hi = sorted((rng.randint(17, 1100), rng.randint(17, 1100)))
        p0, p1 = sorted((rng.randint(0, 42), rng.randint(1, 42)))
        return {"kind": kind, "B": _log(rng, 1, 128), "rows_min": lo, "rows_max": hi, "pages_min": p0,
                "pages_max": p1, "quotas": rng.choice(sorted(HEAD_QUOTAS))}
    if kind == "code":
        K = rng.choice([32, 64, 128, 256, 256])
        lo, hi = sorted((_log(rng, 513, 12000), _log(rng, 513, 12000)))
        f32 = rng.random() < 0.15
        return {"kind": kind, "R": 1 if f32 else rng.choice([1, 1, 2, 3, 4]), "K": K,
                "quota": rng.choice([q for q in (16, 32, 64, 128, 256) if q <= K]), "before_min": min(lo, 4000) if f32
                else lo, "before_max": min(hi, 4000) if f32 else hi, "tail": rng.choice([0, 0, 16, 32]),
                "dtype": "f32" if f32 else "bf16"}
    if kind == "step":
        lo, hi = sorted((_log(rng, 33, 9000), _log(rng, 33, 9000)))
        c0, c1 = sorted((rng.randint(2, 512), rng.randint(2, 512)))
        return {"kind": kind, "decodes": rng.randint(0, 64), "rows_min": lo, "rows_max": hi,
                "chunks": rng.randint(1, 4), "chunk_min": c0, "chunk_max": c1, "past_min": 0,
                "past_max": rng.choice([0, 512, 3000]), "codes": rng.randint(0, 2), "K": 256,
                "quota": rng.choice([64, 128, 256])}
    if kind == "rope":
        per = rng.choice([1, 1, _log(rng, 2, 512)])
        return {"kind": kind, "T": _log(rng, max(1, per), 4096), "per_request": per, "codes_k": rng.choice([128, 256]),
                "prompt": rng.random() < 0.3}
    if kind == "moves":
        return {"kind": kind, "B": _log(rng, 1, 32), "max_prior_blocks": rng.randint(0, 4)}
    c = {"kind": kind, "dtype": "bf16", "grad": rng.random() < 0.6, "B": rng.choice([1, 1, 2, 3]), "N": 1, "C": 512,
         "K": 128, "L": 1, "R": 0, "rx": False, "tail": 0, "policy": "static", "xattn": "full", "prompt": 0,
         "head_quota": rng.random() < 0.4}
    c["C"], c["K"] = rng.choice([(512, 128), (512, 128), (512, 256), (512, 64), (256, 64), (200, 40), (128, 64)])
    if rng.random() < 0.5:
        c["prompt"] = rng.randint(1, 2 * c["C"])
    how = rng.choice(["plain", "plain", "tail", "replay", "replay", "passes", "xattn", "causal"])
    if how == "tail":
        c["tail"], c["policy"] = rng.choice([16, 32, 100]), rng.choice(["static", "rolling", "sticky", "raw"])
    elif how == "replay":
        c["R"], c["rx"] = rng.choice([16, 16, 16, 32, 64]), rng.random() < 0.3
    elif how == "passes":
        c["L"] = 2
    elif how == "xattn":
        c["xattn"] = rng.choice(["causal", "none"])
    elif how == "causal":                                   # the model's plain forward: no codes
        c["K"], c["prompt"], c["head_quota"] = 0, 0, False
        c["C"] = rng.choice([_log(rng, 65, 4096), 512, 2048])
    if rng.random() < 0.15:
        c["dtype"], c["grad"], c["B"] = "f32", False, 1
    per = c["C"] + c["L"] * c["K"] + c["R"]
    most = 2000 if c["dtype"] == "f32" else 4096 if c["K"] == 0 else 7200 // c["B"]
    if c["dtype"] == "f32" and c["K"] == 0:
        c["C"] = per = min(c["C"], 1500)
    c["N"] = 1 if c["K"] == 0 else rng.randint(1, max(1, most // per))
    return c


# -- inputs ----------------------------------------------------------------------------------------------------------
def _spread(n, lo, hi, key):
    """n whole numbers evenly over [lo, hi], in an order fixed by ``key``."""
    v = np.rint(np.linspace(lo, hi, n)).astype(np.int64) if n > 1 else np.full(n, hi, np.int64)
    return np.random.RandomState(key).permutation(v)


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed) * 7919 + 17)


def _randn(gen, shape, dtype=torch.bfloat16, gain=1.0):
    t = torch.empty(shape, dtype=dtype, device="cuda").normal_(generator=gen)
    return t if gain == 1.0 else t.mul_(gain)


def _queries(gen, lead, dtype=torch.bfloat16):
    """Queries whose heads have different score scales (1 to 2.5: the logits of a normalised q.k differ by head)."""
    q = _randn(gen, (*lead, HQ, D), torch.float32)
    return q.mul_(torch.linspace(1.0, 2.5, HQ, device="cuda")[:, None]).to(dtype)


def _pages(rows):
    return -(-np.asarray(rows, np.int64) // PAGE)


def _tables(gen, rows, slack=2):
    """A page table [B, W] of pages scattered over a pool ``slack`` times the pages in use, and the pool's size."""
    n = _pages(rows)
    pool = int(n.sum()) * slack + 8
    W = int(n.max())
    ids = torch.randperm(pool, generator=gen, device="cuda").to(torch.int32).cpu().numpy()
    tab = np.zeros((len(rows), W), np.int32)
    at = 0
    for b, k in enumerate(n.tolist()):
        tab[b, :k] = ids[at: at + k]
        at += k
    return tab, pool


def _dtype(case):
    return torch.float32 if case.get("dtype") == "f32" else torch.bfloat16


def _rows(case):
    return _spread(case["B"], case["rows_min"], case["rows_max"], case["B"])


def _code_before(case):
    return _spread(case["R"], case["before_min"], case["before_max"], case["R"])


def _step_sizes(case):
    dec = _spread(case["decodes"], case["rows_min"], case["rows_max"], 3)
    chunk = _spread(case["chunks"], case["chunk_min"], case["chunk_max"], 4)
    past = _spread(case["chunks"], case["past_min"], case["past_max"], 5)
    before = _spread(case["codes"], case["rows_min"] + 512, case["rows_max"] + 512, 6)
    qlen = np.concatenate([np.ones(len(dec), np.int64), chunk, np.full(len(before), case["K"], np.int64)])
    seq = np.concatenate([dec, past + chunk, before + case["K"]])
    return dec, chunk, past, before, qlen, seq


def _quota_of_heads(case):
    """Code rows visible per query head (equal within a KV head), or None."""
    if not case["head_quota"]:
        return None
    share = np.array([1.0, 0.5, 0.75, 0.25, 0.1, 0.4, 1.0, 0.6])
    return np.repeat(np.maximum(1, (share * case["K"]).astype(np.int64)), G)


def _prompt_lens(case):
    if not case["prompt"]:
        return None
    return _spread(case["B"], max(1, case["prompt"] // 2), case["prompt"], 7)


def _masked_rows(case):
    return case["N"] * (case["C"] + case["L"] * case["K"] + case["R"])


def prepare(case, seed):
    gen = _gen(seed)
    kind = case["kind"]
    s = types.SimpleNamespace(case=case)
    if kind == "decode":
        rows = _rows(case)
        dt = _dtype(case)
        tab, pool = _tables(gen, rows)
        s.cache = _randn(gen, ops.kv_cache_shape(pool), dt)
        s.q = _queries(gen, (case["B"],), dt)
        s.table = torch.from_numpy(tab).cuda()
        s.lens = torch.from_numpy(rows.astype(np.int32)).cuda()
        s.out, s.lse = torch.empty_like(s.q), torch.empty((case["B"], HQ), dtype=torch.float32, device="cuda")
        s.split = ops.auto_split_pages(rows)
        s.ws = ops.decode_workspace(case["B"], tab.shape[1], s.split, device="cuda") if dt == torch.bfloat16 else None
    elif kind == "packed":
        rows = _rows(case)
        quotas = HEAD_QUOTAS[case["quotas"]]
        n = _spread(case["B"], case["pages_min"], case["pages_max"], 2)
        tab, pool = _tables(gen, rows)
        s.cache = _randn(gen, ops.kv_cache_shape(pool))
        side = int(n.sum()) * 2 + 4
        s.pool = _randn(gen, (side, 2, sum(quotas), D))
        ids = torch.randperm(side, generator=gen, device="cuda").to(torch.int32).cpu().numpy()
        pt = np.zeros((case["B"], case["pages_max"]), np.int32)
        at = 0
        for b, k in enumerate(n.tolist()):
            pt[b, :k] = ids[at: at + k]
            at += k
        s.quotas, s.ptab, s.pcount = quotas, torch.from_numpy(pt).cuda(), torch.from_numpy(n.astype(np.int32)).cuda()
        s.q = _queries(gen, (case["B"],))
        s.table = torch.from_numpy(tab).cuda()
        s.lens = torch.from_numpy(rows.astype(np.int32)).cuda()
        s.out, s.lse = torch.empty_like(s.q), torch.empty((case["B"], HQ), dtype=torch.float32, device="cuda")
        s.split = ops.auto_split_pages(rows)
    elif kind == "code":
        before = _code_before(case)
        K, dt = case["K"], _dtype(case)
        tab, pool = _tables(gen, before + K)
        s.cache = _randn(gen, ops.kv_cache_shape(pool), dt)
        s.q = _queries(gen, (case["R"] * K,), dt)
        s.table = torch.from_numpy(tab).cuda()
        s.starts, s.limits = before, before + case["quota"]
        s.q_start = np.arange(case["R"] + 1, dtype=np.int64) * K
        s.excluded = [(int(b) - case["tail"], int(b)) for b in before] if case["tail"] else None
        s.out = torch.empty_like(s.q)
    elif kind == "step":
        dec, chunk, past, before, qlen, seq = _step_sizes(case)
        tab, pool = _tables(gen, seq)
        T = int(qlen.sum())
        s.cache = _randn(gen, ops.kv_cache_shape(pool))
        s.q = _queries(gen, (T,)).view(T, HQ * D)
        s.k, s.v = _randn(gen, (T, HKV * D)), _randn(gen, (T, HKV * D))
        s.table = torch.from_numpy(tab).cuda()
        qsl = np.concatenate([[0], np.cumsum(qlen)])
        limits = np.full(len(seq), NOT_CODE, np.int64)
        limits[len(dec) + len(chunk):] = before + case["quota"]
        pos = np.concatenate([np.arange(n - m, n) for n, m in zip(seq, qlen)])
        builder = AbridgeMetadataBuilder(max_num_seqs=len(seq), max_pages=tab.shape[1])
        s.md = builder.build(qsl, seq, s.table, positions=torch.from_numpy(pos).cuda(), code_key_limit=limits)
        s.impl, s.layer, s.out = AbridgeAttentionImpl(), object(), torch.empty_like(s.q)
    elif kind == "rope":
        T, per = case["T"], case["per_request"]
        R = -(-T // per)
        idx = np.arange(T) // per
        base = _spread(R, 600, 30000 if not case["prompt"] else 600, 8)
        pos = base[idx] + np.arange(T) % per                 # logical positions of the abridged layout
        removed = np.maximum(base - 400, 0)                  # rows the group has compacted away so far
        tab, pool = _tables(gen, np.full(R, 400 + per + PAGE))
        s.cache = _randn(gen, ops.kv_cache_shape(pool))
        s.q, s.k, s.v = _queries(gen, (T,)), _randn(gen, (T, HKV, D)), _randn(gen, (T, HKV, D))
        s.table = torch.from_numpy(tab).cuda()
        s.idx = torch.from_numpy(idx.astype(np.int32)).cuda()
        s.pos = torch.from_numpy(pos.astype(np.int64)).cuda()
        s.removed = torch.from_numpy(removed.astype(np.int32)).cuda()
        s.cos_sin = ops.rope_cos_sin_cache(32768, device="cuda")
        s.max_pos = int(pos.max())
    elif kind == "moves":
        st = workloads.build_compaction_state(case["B"], seed=case["B"] + 100 * case["max_prior_blocks"],
                                              max_prior_blocks=case["max_prior_blocks"], slack_pages=64, op_rows=False)
        st.planner.apply_events(st.pending)
        _, buf, parts = st.planner.take_step_moves()
        n = max(len(g) for g in st.groups)
        s.caches = [_randn(gen, ops.kv_cache_shape(st.num_pages)) for _ in range(n)]
        s.by_group = [s.caches[: len(g)] for g in st.groups]
        s.moves = worker.device_move_lists(torch.from_numpy(buf.copy()).cuda(), parts)
    else:
        B, S, dt = case["B"], _masked_rows(case), _dtype(case)
        s.q = _queries(gen, (B, S), dt).transpose(1, 2)      # [B, heads, S, 128] views, as a model's layers hand them
        s.k = _randn(gen, (B, S, HKV, D), dt).transpose(1, 2)
        s.v = _randn(gen, (B, S, HKV, D), dt).transpose(1, 2)
        pl, hq = _prompt_lens(case), _quota_of_heads(case)
        s.mask = CompressMask(case["C"], case["K"], case["N"],
                              None if pl is None else torch.from_numpy(pl.astype(np.int32)).cuda(),
                              None if hq is None else torch.from_numpy(hq.astype(np.int32)).cuda()[None].contiguous(),
                              case["tail"], case["policy"], case["xattn"], case["L"], 0, case["R"], case["rx"])
        s.module = types.SimpleNamespace(layer_idx=0)
        if case["grad"]:
            for t in (s.q, s.k, s.v):
                t.requires_grad_(True)
            s.dout = _randn(gen, (B, S, HQ, D))
    return s


def run(s):
    case = s.case
    kind = case["kind"]
    if kind == "decode":
        out, lse = ops.decode_attention(s.q, s.cache, s.table, s.lens, SCALE, max_pages=s.table.shape[1], out=s.out,
                                        lse=s.lse, split_pages=s.split, workspace=s.ws)
        return {"out": out, "lse": lse}
    if kind == "packed":
        out, lse = ops.decode_attention_packed(s.q, s.cache, s.table, s.lens, s.pool, s.quotas, s.ptab, s.pcount,
                                               SCALE, out=s.out, lse=s.lse, split_pages=s.split)
        return {"out": out, "lse": lse}
    if kind == "code":
        out, _ = ops.paged_prefill_attention(s.q, s.cache, s.table, s.q_start, s.starts, s.limits, False, SCALE,
                                             out=s.out, excluded=s.excluded)
        return {"out": out}
    if kind == "step":
        return {"out": s.impl.forward(s.layer, s.q, s.k, s.v, s.cache, s.md, s.out)}
    if kind == "rope":
        slots = ops.slot_mapping(s.idx, s.pos, s.table, compacted=s.removed)
        ops.rope_kv_append(s.q, s.k, s.v, s.pos, s.cos_sin, slot_mapping=slots, kv_cache=s.cache,
                           block_c=0 if case["prompt"] else 512, codes_k=0 if case["prompt"] else case["codes_k"],
                           max_position=s.max_pos)
        return {"slots": slots, "q": s.q, "k": s.k, "cache": s.cache}
    if kind == "moves":
        worker.launch_moves(s.moves, s.by_group)
        return s.caches
    out, _ = masked_attention_forward(s.module, s.q, s.k, s.v, s.mask, scaling=SCALE)
    if not case["grad"]:
        return {"out": out}
    dq, dk, dv = torch.autograd.grad(out, (s.q, s.k, s.v), s.dout)
    return {"out": out, "dq": dq, "dk": dk, "dv": dv}


# -- the compression mask, stated plainly ----------------------------------------------------------------------------
def _visible(case, rows, plen, quota, device):
    """Bool [len(rows), S]: which key rows the query rows see (blocks of [C content | L passes of K codes | R replayed
    rows]; plen raw-prompt content tokens; quota code rows of each pass)."""
    C, K, L, R, S = case["C"], case["K"], case["L"], case["R"], _masked_rows(case)
    per, code_end = C + L * K + R, C + L * K
    tail, policy = case["tail"], case["policy"]
    hidden = R if case["rx"] else 0 if policy == "raw" else tail

    def facts(i):
        b, w = i // per, i % per
        content, replay = w < C, w >= code_end
        return b, w, content, ~content & ~replay, replay, (w - C) // max(K, 1) + 1

    q = torch.as_tensor(rows, device=device)[:, None]
    k = torch.arange(S, device=device)[None, :]
    qb, qw, qc, qcode, qrep, qp = facts(q)
    kb, kw, kc, kcode, krep, kp = facts(k)
    same, final = qb == kb, kcode & (kp == L)
    v = (kc & same) | (final & (kb < qb)) | (kc & (kb * C + kw < plen))
    if tail:
        is_tail = kc & (kw >= C - tail)
        if policy == "static":
            v |= is_tail & (kb < qb)
        else:
            near = is_tail & qc & (kb + 1 == qb)
            v |= near if policy == "sticky" else near & (kw - (C - tail) >= qw)
    if R:
        v |= qrep & same & (krep | final)
        v |= qc & krep & (kb + 1 == qb) & (kw - code_end >= qw)
    v &= k <= q
    own = qcode & kcode & same
    v |= own & (kp + 1 == qp)
    if case["xattn"] != "none":
        v |= own & (kp == qp) & ((k <= q) if case["xattn"] == "causal" else True)
    if hidden:
        v &= ~(qcode & same & kc & (kw >= C - hidden))
    return v & (~kcode | (kw - C - (kp - 1) * K < quota)) if K else v


def _masked_pairs(case):
    """Visible (query, key) pairs over all heads and sequences."""
    S = _masked_rows(case)
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    pl = _prompt_lens(case)
    hq = _quota_of_heads(case)
    n, known = 0, {}
    for b in range(case["B"]):
        for h in range(HKV):
            key = (int(pl[b]) if pl is not None else 0, int(hq[G * h]) if hq is not None else case["K"])
            if key not in known:
                known[key] = sum(int(_visible(case, np.arange(r, min(S, r + 1024)), *key, dev).sum())
                                 for r in range(0, S, 1024))
            n += G * known[key]
    return n


def work(case):
    kind = case["kind"]
    e = 4 if case.get("dtype") == "f32" else 2
    row = 2 * HKV * D * e                                     # K and V of one row
    if kind == "decode":
        n = int(_rows(case).sum())
        return {"bytes": n * row + case["B"] * HQ * (2 * D * e + 4), "flops": 4 * D * HQ * n}
    if kind == "packed":
        n, q = int(_rows(case).sum()), sum(HEAD_QUOTAS[case["quotas"]])
        side = int(_spread(case["B"], case["pages_min"], case["pages_max"], 2).sum()) * q
        return {"bytes": n * row + side * 4 * D + case["B"] * HQ * (4 * D + 4), "flops": 4 * D * (HQ * n + G * side)}
    if kind == "code":
        n = int((_code_before(case) + case["quota"] - case["tail"]).sum())
        return {"bytes": n * row + case["R"] * case["K"] * HQ * D * 2 * e, "flops": 4 * D * HQ * case["K"] * n}
    if kind == "step":
        dec, chunk, past, before, qlen, seq = _step_sizes(case)
        pairs = int(dec.sum() + (chunk * past + chunk * (chunk + 1) // 2).sum()
                    + case["K"] * (before + case["quota"]).sum())
        T = int(qlen.sum())
        keys = int(dec.sum() + (past + chunk).sum() + (before + case["quota"]).sum())
        return {"bytes": keys * row + T * (HQ * D * 4 + 2 * row), "flops": 4 * D * HQ * pairs}
    if kind == "rope":
        T = case["T"]
        return {"bytes": T * (2 * HQ * D * 2 + 2 * HKV * D * 2 + HKV * D * 2 + row + D * 4 + 20),
                "flops": T * (HQ + HKV) * D * 3}
    if kind == "moves":
        st = workloads.build_compaction_state(case["B"], seed=case["B"] + 100 * case["max_prior_blocks"],
                                              max_prior_blocks=case["max_prior_blocks"], slack_pages=64, op_rows=False)
        st.planner.apply_events(st.pending)
        parts = st.planner.take_step_moves()[2]
        n = sum(p[2] * len(st.groups[p[0]]) for p in parts)
        return {"bytes": n * 2 * row, "flops": 0}
    S, B = _masked_rows(case), case["B"]
    fwd = B * S * (2 * HQ + 2 * HKV) * D * e
    pairs = _masked_pairs(case)
    if not case["grad"]:
        return {"bytes": fwd, "flops": 4 * D * pairs}
    return {"bytes": fwd + B * S * (2 * HQ + 2 * HKV) * D * e, "flops": 14 * D * pairs}


def tolerance(case):
    kind = case["kind"]
    if kind == "moves":
        return "exact"
    if case.get("dtype") == "f32":
        return {"rel": 1e-5, "max": 1e-3}
    if kind == "rope":
        return {"rel": 7e-3, "max": 0.05}
    if kind == "masked" and case["grad"]:
        return {"rel": 1.6e-2, "max": 0.5}
    return {"rel": 1e-2, "max": 0.2}


# -- the same results in 64 bits -------------------------------------------------------------------------------------
def _attend(q, k, v, vis=None):
    """Attention of q [G, n, D] over k, v [m, D], all float64; vis [n, m] bool or None. (out [G, n, D], lse [G, n])"""
    sc = (q @ k.T) * SCALE
    if vis is not None:
        sc.masked_fill_(~vis, -math.inf)
    lse = torch.logsumexp(sc, -1)
    p = torch.exp(sc - torch.where(torch.isfinite(lse), lse, 0.0)[..., None])
    return p @ v, lse


def _gather(cache, table, n):
    """Rows 0 .. n - 1 of a sequence: K and V [8, n, 128] float64."""
    kv = cache[table[: -(-n // PAGE)].long()]
    k, v = (kv[:, i].reshape(-1, HKV, D)[:n].double().transpose(0, 1).contiguous() for i in (0, 1))
    return k, v


def exact(case, seed):
    kind = case["kind"]
    if kind == "moves":
        return None
    s = prepare(case, seed)
    if kind in ("decode", "packed"):
        out = torch.empty((case["B"], HQ, D), dtype=torch.float64, device="cuda")
        lse = torch.empty((case["B"], HQ), dtype=torch.float64, device="cuda")
        lens = s.lens.tolist()
        for b in range(case["B"]):
            k, v = _gather(s.cache, s.table[b], lens[b])
            side = None
            if kind == "packed":
                side = s.pool[s.ptab[b, : int(s.pcount[b])].long()].double()      # [pages, 2, rows, D]
            at = 0
            for h in range(HKV):
                kh, vh = k[h], v[h]
                if side is not None:
                    n = s.quotas[h]
                    kh = torch.cat([kh, side[:, 0, at: at + n].reshape(-1, D)])
                    vh = torch.cat([vh, side[:, 1, at: at + n].reshape(-1, D)])
                    at += n
                o, z = _attend(s.q[b, G * h: G * h + G].double()[:, None], kh, vh)
                out[b, G * h: G * h + G], lse[b, G * h: G * h + G] = o[:, 0], z[:, 0]
        return {"out": out, "lse": lse}
    if kind in ("code", "step"):
        if kind == "code":
            requests = [(int(a), int(a) + case["K"], int(st), int(lim), False)
                        for a, st, lim in zip(s.q_start, s.starts, s.limits)]
        else:
            slots, n = s.md.slot_mapping, s.md.num_actual_tokens
            for i, new in ((0, s.k), (1, s.v)):
                s.cache[slots // PAGE, i, slots % PAGE] = new.view(n, HKV, D)
            qsl, sl, lims = s.md.query_start_loc, s.md.seq_lens, s.md.code_key_limit
            requests = [(int(qsl[r]), int(qsl[r + 1]), int(sl[r] - (qsl[r + 1] - qsl[r])),
                         int(sl[r]) if lims[r] == NOT_CODE else int(lims[r]), lims[r] == NOT_CODE)
                        for r in range(len(sl))]
        T = s.q.shape[0]
        q = s.q.view(T, HQ, D)
        out = torch.empty((T, HQ, D), dtype=torch.float64, device="cuda")
        for r, (a, z, start, limit, causal) in enumerate(requests):
            k, v = _gather(s.cache, s.table[r], limit)
            keys = torch.arange(limit, device="cuda")[None, :]
            vis = keys <= start + torch.arange(z - a, device="cuda")[:, None] if causal else None
            if kind == "code" and s.excluded:
                lo, hi = s.excluded[r]
                vis = ((keys < lo) | (keys >= hi)).expand(z - a, limit)
            for h in range(HKV):
                o, _ = _attend(q[a:z, G * h: G * h + G].double().transpose(0, 1), k[h], v[h], vis)
                out[a:z, G * h: G * h + G] = o.transpose(0, 1)
        return {"out": out.view(s.q.shape)}
    if kind == "rope":
        pos = s.pos.clone()
        if not case["prompt"]:
            K = case["codes_k"]
            blk, w = pos // (512 + K), pos % (512 + K)
            rev = torch.zeros_like(w)
            for i in range(int(math.log2(K))):
                rev |= ((torch.clamp(w - 512, min=0) >> i) & 1) << (int(math.log2(K)) - 1 - i)
            pos = blk * 512 + torch.where(w < 512, w, rev * 512 // K)
        cs = s.cos_sin[pos].double()[:, None]
        cos, sin = cs[..., :64], cs[..., 64:]

        def turn(x):
            a, b = x.double()[..., :64], x.double()[..., 64:]
            return torch.cat([a * cos - b * sin, b * cos + a * sin], -1)

        q, k = turn(s.q), turn(s.k)
        p = s.pos - s.removed[s.idx.long()]
        slots = s.table[s.idx.long(), p // PAGE].long() * PAGE + p % PAGE
        cache = s.cache.double()
        cache[slots // PAGE, 0, slots % PAGE] = k
        cache[slots // PAGE, 1, slots % PAGE] = s.v.double()
        return {"slots": None, "q": q, "k": k, "cache": cache}
    B, S = case["B"], _masked_rows(case)
    pl, hq = _prompt_lens(case), _quota_of_heads(case)
    q, k, v = (t.detach() for t in (s.q, s.k, s.v))
    out = torch.empty((B, S, HQ, D), dtype=torch.float64, device="cuda")
    grads = [torch.zeros(t.shape, dtype=torch.float64, device="cuda") for t in (q, k, v)] if case["grad"] else None
    step = 2048
    for b in range(B):
        last, vis = None, None
        for h in range(HKV):
            key = (int(pl[b]) if pl is not None else 0, int(hq[G * h]) if hq is not None else case["K"])
            if key != last:
                vis = torch.cat([_visible(case, np.arange(r, min(S, r + 1024)), *key, "cuda")
                                 for r in range(0, S, 1024)])
                last = key
            kh, vh = k[b, h].double(), v[b, h].double()
            for u in range(G * h, G * h + G):
                for r in range(0, S, step):
                    e = min(S, r + step)
                    qh, m = q[b, u, r:e].double(), vis[r:e]
                    sc = (qh @ kh.T).mul_(SCALE).masked_fill_(~m, -math.inf)
                    p = torch.softmax(sc, -1)
                    del sc
                    o = p @ vh
                    out[b, r:e, u] = o
                    if case["grad"]:
                        g = s.dout[b, r:e, u].double()
                        grads[2][b, h] += p.T @ g
                        ds = (g @ vh.T).sub_((g * o).sum(-1, keepdim=True)).mul_(p)
                        grads[0][b, u, r:e] = (ds @ kh) * SCALE
                        grads[1][b, h] += (ds.T @ qh) * SCALE
                        del ds
                    del p
    if not case["grad"]:
        return {"out": out}
    return {"out": out, "dq": grads[0], "dk": grads[1], "dv": grads[2]}
