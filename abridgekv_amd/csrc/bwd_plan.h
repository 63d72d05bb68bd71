// How the masked backward cuts its dK/dV work, and the workspace that this takes. Plain integer code without GPU types, so
// a host build can check the bounds.
#pragma once
#include <stddef.h>

#include "mask_walk.h"

namespace abkv {

constexpr int kDkvMinPart = 12;                 // query tiles (x 4 heads) a part is worth starting for
constexpr int kSlotFloats = 2 * kBN * 128;      // dK and dV of a key tile, of one KV head

// Even share of a launch: `total` query tiles seen by all key tiles over the workgroups that run at once per KV head.
ABKV_HD int dkv_share(int total, int workers) { return imax(kDkvMinPart, (total + workers - 1) / workers); }

// Parts of a key tile that `seen` query tiles see.
ABKV_HD int dkv_parts(int seen, int share) {
  if (2 * seen <= 3 * share) return 1;                      // (at most 3/2 seen / share parts otherwise)
  return (seen + share - 1) / share;
}

// Workspace offsets in bytes: lse2 at 0, dvec; from seen on relative to the next 16-byte boundary.
struct BwdLayout {
  size_t rows;                                  // lse2 and dvec: the least workspace; without the rest nothing is split
  size_t dvec, seen, done, slots, bytes;
  int workers, cap;                             // cap: partial slots per KV head (parts of split tiles)
};
inline BwdLayout bwd_layout(int batch, int seq_len, int cus) {
  constexpr size_t kHeadsQ_ = 32, kHeadsKV_ = 8;
  const size_t q_tiles = ((size_t)(seq_len > 0 ? seq_len : 0) + kBN - 1) / kBN;
  const size_t tiles = q_tiles * (size_t)(batch > 0 ? batch : 0);
  auto up = [](size_t n) { return (n + 255) / 256 * 256; };
  BwdLayout l;
  l.workers = imax(1, 2 * cus / (int)kHeadsKV_);            // two workgroups a CU
  // parts (dkv_parts): at most 3/2 * workers in all (48 MiB of slots on 256 CUs), and a tile's are under
  // q_tiles / kDkvMinPart + 1
  const size_t few = tiles * (q_tiles / kDkvMinPart + 1), most = (size_t)(3 * l.workers / 2);
  l.cap = (int)(few < most ? few : most);
  if (2 * q_tiles <= 3 * kDkvMinPart) l.cap = 0;            // nothing is split
  l.dvec = tiles * kBN * kHeadsQ_ * sizeof(float);
  l.rows = 2 * l.dvec;
  l.seen = l.rows;
  l.done = l.seen + up(tiles * sizeof(int));
  l.slots = l.done + up((size_t)l.cap * kHeadsKV_ * sizeof(int));
  l.bytes = l.slots + (size_t)l.cap * kHeadsKV_ * kSlotFloats * sizeof(float) + 16;   // + the alignment
  return l;
}

}  // namespace abkv
