// Host check of the words that tasks reach workgroups in: every pair of an expert and a channel tile that a launch can have comes
// back as it went in and is told from the end of the list.
#include <cstdio>

#include "tile_list.hpp"

using namespace moe_i8;

int main() {
  if (task_expert(kNoTask) >= 0) return printf("the end of the list reads as a task\n"), 1;
  const uint32_t tiles = ((1ull << 32) / 256 - 16 + 255) / 256;  // of the longest matrix of rows of 256 bytes
  for (uint32_t e : {0u, 1u, (uint32_t)kMaxExperts - 1})
    for (uint32_t nt = 0; nt < tiles; ++nt) {
      const uint32_t w = task_word(e, nt);
      if (task_expert(w) != (int)e || task_channel_tile(w) != (int)nt) return printf("expert %u, channel tile %u\n", e, nt), 1;
    }
  printf("ok\n");
  return 0;
}
