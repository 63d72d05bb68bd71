// Host plan of a multi-query attention launch over the paged cache (paged_prefill.hip): which workgroup takes which key
// tiles of which query tile. Pure host code: no HIP call is made from this file.
//
// A batch's query tiles differ by orders of magnitude in their key ranges (a code step over its whole compacted context
// beside a prompt's first chunk), and a launch ends with its longest workgroup. Query tiles whose range exceeds a length
// L are split along the keys into equal parts of at most L tiles, whose partial results a second kernel merges; L is the
// candidate with the smallest makespan on num_cus / 8 slots (a workgroup fills a CU; the 8 KV heads take the same items),
// items handed out longest first, as the grid does.
//
// Measured against equal splits of every tile or none (us a call, uploads included): two chunks of 300 / 512 rows and a
// code step over 5800 keys 240 -> 129 (none: 136 workgroups, the code step's 90 tiles in a row), with two code steps
// and four chunks 354 -> 170; code steps of four requests over 3000 .. 12000 keys 256 -> 222, of two 184 -> 146;
// four chunks of 200 .. 512 rows, which are not split, 120 -> 117.
#include "abridgekv_amd.h"

#include <stdint.h>

#include <algorithm>
#include <functional>
#include <queue>
#include <vector>

namespace {

constexpr int kTileRows = 64, kTileKeys = 64, kHeads = 8;
// Costs in key tiles (about 2.1 us each): a workgroup's start (queries, first tiles) and end, the merge launch.
constexpr int kItemCost = 6, kMergeCost = 3;

struct Tile {
  int req, q0, keys;         // keys: key tiles of its range
};

// First key tile of part p of n.
int part_of(int keys, int p, int n) { return (int)((int64_t)keys * p / n); }

// Time until the last slot is free when the items (longest first) go to the slot that is free first.
int makespan(const std::vector<int>& lengths, int slots) {
  std::priority_queue<int, std::vector<int>, std::greater<int>> free_at;
  int end = 0;
  for (int n : lengths) {
    int t = n + kItemCost;
    if ((int)free_at.size() >= slots) {
      t += free_at.top();
      free_at.pop();
    }
    free_at.push(t);
    end = std::max(end, t);
  }
  return end;
}

}  // namespace

extern "C" {

int abkv_paged_plan(const int64_t* q_start, const int64_t* kv_start, const int64_t* kv_limit, const int64_t* causal,
                    int num_reqs, int num_cus, int32_t* items, long items_cap, int32_t* merges, long merges_cap,
                    int32_t* sizes) {
  if (num_reqs < 0 || (num_reqs > 0 && (q_start == nullptr || kv_start == nullptr || kv_limit == nullptr ||
                                        causal == nullptr)) || sizes == nullptr || num_cus <= 0)
    return ABKV_ERR_ARG;
  try {
    std::vector<Tile> tiles;
    int64_t total = 0;
    int longest = 0;
    for (int r = 0; r < num_reqs; ++r) {
      const int64_t nq = q_start[r + 1] - q_start[r];
      for (int64_t q0 = 0; q0 < nq; q0 += kTileRows) {
        const int64_t last = std::min<int64_t>(q0 + kTileRows, nq) - 1;
        const int64_t keys = causal[r] ? std::min(kv_limit[r], kv_start[r] + last + 1) : kv_limit[r];
        const int n = (int)((std::max<int64_t>(keys, 0) + kTileKeys - 1) / kTileKeys);
        tiles.push_back({r, (int)q0, n});
        total += n;
        longest = std::max(longest, n);
      }
    }
    const int slots = std::max(1, num_cus / kHeads);
    const int n_tiles = (int)tiles.size();
    // candidates: the longest range in k parts; at most three more items a slot than there are tiles
    int best_len = std::max(longest, 1), best = 0x7fffffff, tried = 0;
    std::vector<int> lengths;
    for (int k = 1; k <= 64; k += k < 8 ? 1 : k < 16 ? 2 : 8) {
      const int len = (longest + k - 1) / k;
      if (k > 1 && (len == tried || len < 2)) continue;
      tried = len;
      lengths.clear();
      bool split = false;
      for (const Tile& t : tiles) {
        const int parts = t.keys > len ? (t.keys + len - 1) / len : 1;
        split |= parts > 1;
        for (int p = 0; p < parts; ++p) lengths.push_back(part_of(t.keys, p + 1, parts) - part_of(t.keys, p, parts));
      }
      const int64_t n = (int64_t)lengths.size();
      if (k > 1 && n > n_tiles + 3L * slots) break;
      const int64_t bound = (total + n * kItemCost) / slots + (split ? kMergeCost : 0);
      if (bound >= best) break;
      std::sort(lengths.begin(), lengths.end(), std::greater<int>());
      const int end = makespan(lengths, slots) + (split ? kMergeCost : 0);
      if (end < best) {
        best = end;
        best_len = std::max(len, 1);
      }
    }
    struct Item {
      int length;
      int32_t v[5];
    };
    std::vector<Item> out;
    long n_merges = 0, rows = 0;
    for (const Tile& t : tiles) {
      const int parts = t.keys > best_len ? (t.keys + best_len - 1) / best_len : 1;
      const long row = parts > 1 ? rows : -1;
      for (int p = 0; p < parts; ++p) {
        const int k0 = part_of(t.keys, p, parts), k1 = part_of(t.keys, p + 1, parts);
        out.push_back({k1 - k0, {t.req, t.q0, k0, k1, parts > 1 ? (int32_t)(row + (long)p * kTileRows) : -1}});
      }
      if (parts > 1) {
        if (n_merges < merges_cap && merges != nullptr) {
          int32_t* m = merges + 4 * n_merges;
          m[0] = (int32_t)(q_start[t.req] + t.q0);
          m[1] = (int32_t)std::min<int64_t>(kTileRows, q_start[t.req + 1] - q_start[t.req] - t.q0);
          m[2] = (int32_t)row;
          m[3] = parts;
        }
        ++n_merges;
        rows += (long)parts * kTileRows;
      }
    }
    sizes[0] = (int32_t)out.size();
    sizes[1] = (int32_t)n_merges;
    sizes[2] = (int32_t)rows;
    if ((long)out.size() > items_cap || n_merges > merges_cap || rows > 0x7fffffffL) return ABKV_ERR_CAPACITY;
    std::stable_sort(out.begin(), out.end(), [](const Item& a, const Item& b) { return a.length > b.length; });
    for (size_t i = 0; i < out.size(); ++i) std::copy(out[i].v, out[i].v + 5, items + 5 * i);
    return ABKV_OK;
  } catch (...) {
    return ABKV_ERR_ARG;
  }
}

}  // extern "C"
