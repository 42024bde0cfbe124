// Prints the plan of `fwd|hbf16|hf32 BH NT K V` lines on stdin (256 CUs):
// out per len, and the workspace in bytes beyond the records.
#include <cstdio>
#include <cstring>

#include "seg_plan.h"

int main() {
  char what[16];
  long BH, NT, K, V;
  while (std::scanf("%15s %ld %ld %ld %ld", what, &BH, &NT, &K, &V) == 5) {
    using namespace thm::seg;
    const Plan p = !std::strcmp(what, "fwd") ? plan_fwd(BH, NT, K, V, 256) : plan_h(BH, NT, K, V, !std::strcmp(what, "hf32"), 256);
    const long ws = (long)(p_bytes(p, BH, NT, K) + s_bytes(p, BH, NT, K, V) + redo_bytes(p, BH, V));
    std::printf("%ld %ld %ld %ld\n", (long)p.out, (long)p.per, (long)p.len, ws);
  }
  return 0;
}
