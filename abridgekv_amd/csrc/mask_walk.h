// The compression mask as key ranges: which key tiles a 64-row query tile reads and which keys of a tile one query row
// sees. Plain integer code without GPU types, so a host build can check it against the mask's definition.
#pragma once

#if defined(__HIP__) || defined(__HIPCC__)
#define ABKV_HD __host__ __device__ __forceinline__
#else
#define ABKV_HD inline
#endif

namespace abkv {

constexpr int kBM = 64;                  // query rows per tile
constexpr int kBN = 64;                  // keys per tile

// Retained-tail policies (retain_tail_policy): which later rows see an earlier block's last T content rows.
constexpr int kTailStatic = 0;   // every later row
constexpr int kTailRolling = 1;  // the next block's i-th content row sees the tail's rows i .. T-1
constexpr int kTailSticky = 2;   // every content row of the next block
constexpr int kTailRaw = 3;      // the rolling window of raw_tail (compress_forward.py:89-96): the codes see the whole
                                 // block, their own tail included (code_excluded_tail = 0, :309-311)

// pause_xattn: which code rows of its own pass and block a code row sees (compress_forward.py:313-314, 622-625).
constexpr int kXattnFull = 0;     // all of them (bidirectional)
constexpr int kXattnCausal = 1;   // those at or before its own position
constexpr int kXattnNone = 2;     // none, itself included

constexpr int kNoKey = 0x7fffffff;       // a range start past every key

struct TileMask {
  int mode;        // 0 none, 1 key < this lane's limit, 2 key < limit[u] (this wave's head u), 3 this lane's span of
                   // the segment part (lane_span: seg, kb, limit = {segment start, part end}),
                   // 4 key < this lane's limit and outside the excluded range [limit[0], limit[1]),
                   // 5 key < limit[0] or key >= this lane's limit + limit[1] (a band that moves with the query row)
  int limit[2];
  int seg, kb;     // mode 3: segment (kSeg* or a pause pass 1 .. L) of block kb
};

constexpr int kSegContent = 0;
constexpr int kSegReplay = -1;
constexpr int kSegCopy = -2;

// Sequence layout: N blocks of [C content | L passes of K codes | R replay rows] (per rows each), then copy rows.
struct MaskShape {
  int S0, C, K, L, R, copy, per, N;
  int tail, policy, xattn;
  bool rx;
  ABKV_HD int block_rows() const { return S0 - copy; }
  ABKV_HD int code_end() const { return C + L * K; }
  // the own-block content rows hidden from the codes
  ABKV_HD int hidden() const { return rx ? R : policy == kTailRaw ? 0 : tail; }
};

ABKV_HD int imin(int a, int b) { return a < b ? a : b; }
ABKV_HD int imax(int a, int b) { return a > b ? a : b; }
ABKV_HD int iclamp(int x, int lo, int hi) { return imax(lo, imin(x, hi)); }

// What the mask asks about one query row.
struct RowFacts {
  int q, qb, qw;   // row, block, in-block offset
  int seg;         // kSegContent, a pause pass 1 .. L, kSegReplay, kSegCopy
  bool valid;      // inside the S0 rows
};
ABKV_HD RowFacts row_facts(const MaskShape& g, int q) {
  RowFacts r;
  r.q = q;
  r.valid = q < g.S0;
  r.qb = q / g.per;
  r.qw = q - r.qb * g.per;
  r.seg = q >= g.block_rows()  ? kSegCopy
          : r.qw < g.C         ? kSegContent
          : r.qw >= g.code_end() ? kSegReplay
                                 : (r.qw - g.C) / g.K + 1;
  return r;
}

// Keys of one segment part that a query row sees: key < a, or b <= key < end (a <= end; keys at or past the part's end
// belong to other tiles). The part lies in segment `seg` of block kb, whose first key is base.
ABKV_HD void lane_span(const MaskShape& g, const RowFacts& r, int seg, int kb, int base, int end, int plen, int quota,
                       int& a, int& b) {
  a = base;
  b = kNoKey;
  const bool own = kb == r.qb && r.seg != kSegCopy;
  if (seg == kSegContent) {
    if (own) {
      a = r.seg == kSegContent ? r.q + 1 : base + g.C - (r.seg > 0 ? g.hidden() : 0);
    } else if (r.seg != kSegCopy && kb < r.qb) {
      a = base + iclamp(plen - kb * g.C, 0, g.C);
      if (g.tail > 0) {
        const bool next = r.seg == kSegContent && kb + 1 == r.qb;
        if (g.policy == kTailStatic || (next && g.policy == kTailSticky)) b = base + g.C - g.tail;
        else if (next) b = base + g.C - g.tail + r.qw;
      }
    }
  } else if (seg > 0) {
    const int seen = base + iclamp(quota, 0, g.K);
    if (r.seg == kSegCopy) {
      if (seg == g.L && kb == g.N - 1) a = seen;
    } else if (kb < r.qb) {
      if (seg == g.L) a = seen;
    } else if (own) {
      if (r.seg > 0) {
        if (seg + 1 == r.seg) a = seen;
        else if (seg == r.seg && g.xattn != kXattnNone) a = g.xattn == kXattnFull ? seen : imin(seen, r.q + 1);
      } else if (r.seg == kSegReplay && seg == g.L) {
        a = seen;
      }
    }
  } else if (seg == kSegReplay) {
    if (own) {
      if (r.seg == kSegReplay) a = r.q + 1;
    } else if (r.seg == kSegContent && kb + 1 == r.qb) {
      b = base + r.qw;
    }
  } else if (r.seg == kSegCopy) {
    a = r.q + 1;
  }
  if (!r.valid) {
    a = base;
    b = kNoKey;
  }
  a = imin(a, end);
}

// Walk over the key tiles that the query rows q0 .. q_last (at most 64) read, segment by segment: a tile holds up to 64
// keys of one segment, starting at any row, so a block's K codes cost ceil(K / 64) tiles wherever the block starts and
// the hidden content of earlier blocks costs none. Every key a row of the tile sees lies in exactly one tile.
//   blocks before the tile's first block (far): the raw-prompt prefix, a static tail, the final pass's codes; all
//     rows see the same keys (modes 0 and 2)
//   the block before it: also a window tail or replay rows (mode 3)
//   the tile's own blocks (near): the segments up to the last row. A tile inside one block's content takes modes 0 and
//     1, a tile inside one code pass 0 and 2; what is left (rows of several segments) takes the row's span (mode 3).
// The state is wave-uniform.
struct SegWalk {
  static constexpr bool kHole = false;
  static constexpr bool kBand = false;
  static constexpr bool kSpan = true;
  MaskShape g;
  int q0, q_last, plen, qmin, qmax, wq0, wq1;
  int qb_lo, qb_hi;                  // blocks of the tile's rows (copy rows alone: N, with no own block)
  int kb_end;                        // blocks to walk
  int lim;                           // no key at or past it is seen in the tile's last block
  int full;                          // in the tile's block every row sees the content keys below it
  int one_pass;                      // the pass all rows belong to (one block), or 0
  int first_pass;                    // earliest pass of block qb_lo that the tile reads
  int qw0;                           // in-block offset of row q0
  bool has_rows, has_copy, one_block, content;
  int kb, part, pos, base, end, seg;

  ABKV_HD SegWalk(const MaskShape& g_, int q0_, int q_last_, int plen_, int qmin_, int qmax_, int wq0_, int wq1_)
      : g(g_), q0(q0_), q_last(q_last_), plen(plen_), qmin(qmin_), qmax(qmax_), wq0(wq0_), wq1(wq1_) {
    const int rows = g.block_rows();
    has_rows = q0 < rows;
    has_copy = q_last >= rows;
    const int ql = imin(q_last, rows - 1);
    qb_lo = has_rows ? q0 / g.per : g.N;
    qb_hi = has_rows ? ql / g.per : g.N - 1;
    kb_end = qb_hi + 1;
    one_block = has_rows && !has_copy && qb_lo == qb_hi;
    qw0 = q0 - qb_lo * g.per;
    const int wl = ql - qb_hi * g.per;
    const int ce = g.code_end();
    const int pl = wl < g.C || wl >= ce ? 0 : (wl - g.C) / g.K + 1;        // pass of the last row
    const int pf = qw0 < g.C || qw0 >= ce ? 0 : (qw0 - g.C) / g.K + 1;     // pass of the first row
    lim = has_copy ? rows : pl > 0 ? qb_hi * g.per + g.C + pl * g.K : ql + 1;
    content = one_block && wl < g.C;
    one_pass = one_block && pf == pl ? pl : 0;
    full = one_block ? imin(q0 + 1, qb_lo * g.per + g.C - g.hidden()) : 0;
    if (content) full = q0 + 1;
    first_pass = has_rows && qw0 >= g.C ? (pf > 0 ? imax(pf - 1, 1) : g.L) : 1;
    kb = has_rows ? 0 : g.N - 1;
    part = -1;
    pos = -kBN;
    end = 0;
    base = 0;
    seg = 0;
  }

  // the next non-empty part: base, pos (its first key), end, seg, kb; false when none is left
  ABKV_HD bool advance() {
    for (;;) {
      ++part;
      if (kb >= kb_end) {                                     // after the blocks: the copy rows
        if (!has_copy || part > 0) return false;
        seg = kSegCopy;
        base = pos = g.block_rows();
        end = q_last + 1;
        return true;
      }
      const int b0 = kb * g.per;
      if (part == 0) {                                        // content: all of an own block's, else the raw prompt
        base = pos = b0;
        seg = kSegContent;
        if (!has_rows) {
          part = g.L;                                         // copy rows read the last block's final pass alone
          continue;
        }
        end = kb >= qb_lo ? imin(b0 + g.C, lim) : b0 + iclamp(plen - kb * g.C, 0, g.C);
        if (pos < end) return true;
      } else if (part == 1) {                                 // an earlier block's retained tail
        if (kb >= qb_lo) {
          if (kb == qb_lo) part = first_pass;                 // (the next part is pass first_pass)
          if (g.K == 0) part = g.L + 1;
          continue;
        }
        int start = g.C;
        if (g.policy == kTailStatic) start = g.C - g.tail;
        else if (kb + 1 == qb_lo && qw0 < g.C) start = g.C - g.tail + (g.policy == kTailSticky ? 0 : qw0);
        const int from = b0 + imax(start, iclamp(plen - kb * g.C, 0, g.C));
        part = g.L;                                           // earlier passes of an earlier block are hidden
        if (g.tail > 0 && from < b0 + g.C) {
          base = b0;
          pos = from;
          end = b0 + g.C;
          return true;
        }
      } else if (part <= g.L + 1) {                           // pass part - 1
        base = pos = b0 + g.C + (part - 2) * g.K;
        seg = part - 1;
        end = base + iclamp(qmax, 0, g.K);
        if (kb >= qb_lo) end = imin(end, lim);
        if (pos < end) return true;
      } else {                                                // replay rows, then the next block
        base = pos = b0 + g.code_end();
        seg = kSegReplay;
        end = base;
        if (g.R > 0 && has_rows) {
          if (kb >= qb_lo) end = imin(base + g.R, lim);
          else if (kb + 1 == qb_lo && qw0 < g.R) {
            pos = base + qw0;
            end = base + g.R;
          }
        }
        if (pos < end) {
          ++kb;                                               // (tile masks of the part use kb - 1: see next)
          part = -1;
          return true;
        }
        ++kb;
        part = -1;
      }
    }
  }

  // next tile (k0: its first key) and its mask; false when the walk is done
  ABKV_HD bool next(int& k0, TileMask& tm, bool) {
    pos += kBN;
    if (pos >= end && !advance()) return false;
    k0 = pos;
    const int blk = seg == kSegReplay ? kb - 1 : kb;
    const bool far = blk < qb_lo && !has_copy;
    tm.seg = seg;
    tm.kb = blk;
    tm.mode = 3;
    tm.limit[0] = base;
    tm.limit[1] = end;
    if (seg == kSegContent) {
      if (far) {
        if (pos < base + iclamp(plen - blk * g.C, 0, g.C) || g.policy == kTailStatic) {
          tm.mode = pos + kBN <= end ? 0 : 2;                 // a range that every row sees: keys below its end
          tm.limit[0] = tm.limit[1] = end;
        }
      } else if (one_block && pos + kBN <= imin(full, end)) {
        tm.mode = 0;
      } else if (content && blk == qb_lo) {
        tm.mode = 1;
      }
    } else if (seg > 0) {
      const bool own_full = one_pass > 0 && blk == qb_lo &&
                            (seg + 1 == one_pass || (seg == one_pass && g.xattn == kXattnFull));
      if (far || own_full) {
        tm.mode = pos + kBN <= base + iclamp(qmin, 0, g.K) ? 0 : 2;
        tm.limit[0] = base + iclamp(wq0, 0, g.K);
        tm.limit[1] = base + iclamp(wq1, 0, g.K);
      }
    }
    return true;
  }
};

// The query rows that see one key: [a1, e1) and [a2, e2) (empty ranges are [0, 0)); a code key only for heads whose
// quota exceeds its slot.
struct KeySpan {
  int a1, e1, a2, e2;
  int slot;          // index within its pass, -1 for a key that is no code
};
ABKV_HD KeySpan key_span(const MaskShape& g, int key, int plen) {
  KeySpan s{0, 0, 0, 0, -1};
  if (key >= g.S0) return s;
  const int rows = g.block_rows();
  if (key >= rows) {                                          // copy rows: themselves, causally
    s.a1 = key;
    s.e1 = g.S0;
    return s;
  }
  const int kb = key / g.per, kw = key - kb * g.per;
  const int b0 = kb * g.per, b1 = b0 + g.per, ce = b0 + g.code_end();
  if (kw < g.C) {
    const bool hidden = kw >= g.C - g.hidden();               // from its own block's codes
    s.a1 = key;
    s.e1 = hidden ? b0 + g.C : b1;
    s.a2 = hidden ? ce : b1;
    s.e2 = b1;                                                // then the own block's replay rows
    const int t = kw - (g.C - g.tail);                        // index in the retained tail
    if (kb * g.C + kw < plen) s.e2 = rows;
    else if (g.tail > 0 && t >= 0)
      s.e2 = imin(rows, g.policy == kTailStatic ? rows : b1 + (g.policy == kTailSticky ? g.C : t + 1));
  } else if (b0 + kw < ce) {
    const int p = (kw - g.C) / g.K, p0 = b0 + g.C + p * g.K, p1 = p0 + g.K;
    s.slot = kw - g.C - p * g.K;
    s.a1 = g.xattn == kXattnFull ? p0 : g.xattn == kXattnCausal ? key : p1;
    s.e1 = p1;
    s.a2 = p1;
    s.e2 = p + 1 < g.L ? p1 + g.K : kb == g.N - 1 ? g.S0 : rows;
  } else {                                                    // replay row r: its block's later ones, and content rows
    s.a1 = key;                                               // 0 .. r of the next block
    s.e1 = imin(rows, b1 + (b0 + kw - ce) + 1);
    if (kb == g.N - 1) s.e1 = b1;
  }
  if (s.e1 >= s.a2 && s.a2 < s.e2) {                          // adjoining ranges: one
    s.e1 = imax(s.e1, s.e2);
    s.a2 = s.e2 = 0;
  }
  if (s.a1 >= s.e1) s.a1 = s.e1 = 0;
  if (s.a2 >= s.e2) s.a2 = s.e2 = 0;
  return s;
}

}  // namespace abkv
