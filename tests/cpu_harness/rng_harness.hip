// The packet stream taken several words at a time (PacketRng::take) against the
// same stream word by word, on the host.
#include <stdint.h>

#include "philox.h"

using namespace mcm;

// Follows packet `id` through nCalls draws; n[k] in 0..4 words at call k by
// take(), n[k] < 0: -n[k] words one at a time.  Returns the number of the first
// call that differs from the word-by-word stream, or -1.
extern "C" int rng_take_compare(uint32_t k0, uint32_t k1, uint32_t stream, uint64_t id, const int* n, int nCalls) {
  PacketRng a, b;
  for (PacketRng* r : {&a, &b}) {
    r->key0 = k0;
    r->key1 = k1;
    r->stream = stream;
    r->start(id);
  }
  for (int k = 0; k < nCalls; ++k) {
    uint32_t w[4] = {0, 0, 0, 0};
    const int m = n[k] < 0 ? -n[k] : n[k];
    if (n[k] >= 0) a.take(w, m);
    for (int q = 0; q < m; ++q) {
      if (n[k] < 0) w[0] = a.next_word();
      if (b.next_word() != w[n[k] < 0 ? 0 : q]) return k;
    }
    // at most three words wait, as a launch record holds
    if (a.have < 0 || a.have > 3) return k;
  }
  return -1;
}
