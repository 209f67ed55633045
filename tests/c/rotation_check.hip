// Host check of which launches start their tasks at different reduction steps.
#include <cstdio>

#include "tile_list.hpp"

using namespace moe_i8;

int main() {
  int wrong = 0;
  auto check = [&](int experts, int k, int inter, bool rotates) {  // gate_up
    if ((rotation(k, (int64_t)experts * 2 * inter * k, experts) != 0) != rotates) ++wrong, printf("%d experts of %d x %d\n", experts, k, inter);
  };
  check(32, 8192, 1024, true);    // 0.5 GiB: 15 and 27 % faster with narrow and deep tiles
  check(64, 8192, 768, true);     // 0.75 GiB
  check(64, 8192, 1024, false);   // 1 GiB: 10 % slower with narrow tiles
  check(64, 8192, 2048, false);   // 2 GiB: 8 and 15 % slower
  check(64, 4096, 1024, true);
  check(256, 4096, 2048, true);   // 4 GiB
  check(64, 2048, 1024, false);   // no multiple of 4096 bytes
  check(64, 7168, 1024, false);
  // the starts of up to 32 experts: all different, and as far apart as they can be
  for (int experts = 1; experts <= 300; ++experts) {
    const int r = rotation(4096, 0, experts);
    bool used[kStartSteps] = {};
    for (int e = 0; e < experts; ++e) {
      const int s = start_step(e, r);
      if (s < 0 || s >= kStartSteps || (experts <= kStartSteps && (used[s] || s < e * (kStartSteps / experts)))) ++wrong, printf("start of %d of %d\n", e, experts);
      else used[s] = true;
    }
  }
  if (!wrong) printf("ok\n");
  return wrong != 0;
}
