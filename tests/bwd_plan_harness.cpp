// Host build of the masked backward's dK/dV cut (csrc/bwd_plan.h).
#include <stdint.h>

#include "bwd_plan.h"

using namespace abkv;

extern "C" {

long layout_bytes(int batch, int seq_len, int cus) { return (long)bwd_layout(batch, seq_len, cus).bytes; }
long layout_cap(int batch, int seq_len, int cus) { return bwd_layout(batch, seq_len, cus).cap; }

// Slots per KV head that key tiles seen by seen[i] query tiles take.
long slots(const int32_t* seen, int tiles, int cus) {
  const int workers = bwd_layout(1, 64, cus).workers;
  int total = 0;
  for (int i = 0; i < tiles; ++i) total += seen[i];
  long n = 0;
  for (int i = 0; i < tiles; ++i) {
    const int parts = dkv_parts(seen[i], dkv_share(total, workers));
    n += parts > 1 ? parts : 0;
  }
  return n;
}

}
