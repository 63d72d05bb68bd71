// Host build of the compression mask's key ranges (csrc/mask_walk.h): how often each (query, key) pair of one KV head's
// four query heads is visited as visible by the walk over key tiles.
#include <stdint.h>

#include "mask_walk.h"

using namespace abkv;

static MaskShape shape(const int32_t* p) {
  MaskShape g;
  g.C = p[0]; g.K = p[1]; g.N = p[2]; g.L = p[3]; g.R = p[4]; g.copy = p[5];
  g.tail = p[6]; g.policy = p[7]; g.xattn = p[8]; g.rx = p[9] != 0;
  g.per = g.C + g.L * g.K + g.R;
  g.S0 = g.N * g.per + g.copy;
  return g;
}

static bool visible(const MaskShape& g, const TileMask& tm, const RowFacts& r, int key, int plen, int quota, int u) {
  switch (tm.mode) {
    case 0: return true;
    case 1: return key < r.q + 1;
    case 2: return key < tm.limit[u];
    default: {
      int a, b;
      lane_span(g, r, tm.seg, tm.kb, tm.limit[0], tm.limit[1], plen, quota, a, b);
      return key < a || (key >= b && key < tm.limit[1]);
    }
  }
}

extern "C" {

// counts [4][S0][S0] over query tiles of `rows` rows; returns the number of key tiles walked, or -1 for a tile whose first
// key is out of range.
long walk_counts(const int32_t* params, int plen, const int32_t* quota, int rows, uint8_t* counts) {
  const MaskShape g = shape(params);
  const long S = g.S0;
  int qmin = quota[0], qmax = quota[0];
  for (int u = 1; u < 4; ++u) {
    qmin = imin(qmin, quota[u]);
    qmax = imax(qmax, quota[u]);
  }
  long tiles = 0;
  for (int hb = 0; hb < 4; hb += 2)
    for (int q0 = 0; q0 < g.S0; q0 += rows) {
      SegWalk walk(g, q0, imin(q0 + rows, g.S0) - 1, plen, qmin, qmax, quota[hb], quota[hb + 1]);
      int k0 = 0;
      TileMask tm;
      for (bool first = true; walk.next(k0, tm, first); first = false) {
        if (k0 < 0 || k0 >= g.S0) return -1;
        ++tiles;
        for (int q = q0; q < imin(q0 + rows, g.S0); ++q) {
          const RowFacts r = row_facts(g, q);
          for (int u = 0; u < 2; ++u)
            for (int key = k0; key < k0 + kBN; ++key) {
              if (!visible(g, tm, r, key, plen, quota[hb + u], u)) continue;
              if (key >= g.S0) return -2;
              ++counts[((hb + u) * S + q) * S + key];
            }
        }
      }
    }
  return tiles;
}

// counts [4][S0][S0] from the query ranges of every key.
void key_counts(const int32_t* params, int plen, const int32_t* quota, uint8_t* counts) {
  const MaskShape g = shape(params);
  const long S = g.S0;
  for (int key = 0; key < g.S0; ++key) {
    const KeySpan k = key_span(g, key, plen);
    for (int u = 0; u < 4; ++u) {
      if (k.slot >= quota[u]) continue;
      for (int q = k.a1; q < k.e1; ++q) ++counts[(u * S + q) * S + key];
      for (int q = k.a2; q < k.e2; ++q) ++counts[(u * S + q) * S + key];
    }
  }
}

}
