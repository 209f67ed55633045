// A masked store inside a branch that only some lanes take.
#include "lds_loads.hpp"

__global__ void store_by_some_lanes(uint4* out, const uint4* in, int limit) {
  const int t = threadIdx.x;
  if (in[t].x & 1) {
    const uint4 v = in[t + 64];
    moe_i8::store16_through(out + t, v, __ballot(t < limit));
    out[t + 64] = v;
  }
}
