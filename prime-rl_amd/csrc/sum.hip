// Top-k combine for gfx950: out[m, :] = sum_j in[m, j, :] over bf16 rows.
//
// One lane owns 8 consecutive columns (one 16-byte load per routed row, one 16-byte store).
// For k in {2, 3, 4} the adds round to bf16 after every step; any other k accumulates in fp32
// in ascending j and rounds once.  Traffic is the minimum (k + 1) * M * H * 2 bytes: HBM-bound for a
// prefill, one memory latency for a handful of tokens, which is why all loads of a lane are issued before
// the first add (KMAX at a time; a loop over a runtime k makes them a chain of k latencies: 3.9 us for one
// token of 8 rows).
#include "common.hpp"

namespace moe_i8 {
namespace {

constexpr int kThreads = 256;

__device__ __forceinline__ void add8(float (&acc)[8], const v4i& v, bool round_each) {
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const float lo = __uint_as_float((uint32_t)v[e] << 16);
    const float hi = __uint_as_float((uint32_t)v[e] & 0xffff0000u);
    acc[2 * e] += lo;
    acc[2 * e + 1] += hi;
    if (round_each) {
      acc[2 * e] = round_to_bf16(acc[2 * e]);
      acc[2 * e + 1] = round_to_bf16(acc[2 * e + 1]);
    }
  }
}

// KMAX: rows fetched at a time; exactly top_k of them when kExact.
template <bool kRoundEachAdd, int KMAX, bool kExact>
__global__ __launch_bounds__(kThreads) void moe_sum_kernel(const v4i* __restrict__ in, uint4* __restrict__ out, int64_t total,
                                                           int top_k, int vec_per_row) {
  const int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x;
  if (i >= total) return;
  const int64_t m = total >> 32 ? i / vec_per_row : (int64_t)((uint32_t)i / (uint32_t)vec_per_row);
  const int c = (int)(i - m * vec_per_row);
  const int k = kExact ? KMAX : top_k;
  const v4i* src = in + m * (int64_t)k * vec_per_row + c;
  float acc[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) acc[e] = 0.0f;
  for (int j0 = 0; j0 < k; j0 += KMAX) {
    v4i v[KMAX];
#pragma unroll
    for (int j = 0; j < KMAX; ++j) {
      // past the last row: the last one again, not added
      const int row = kExact || j0 + j < k ? j0 + j : k - 1;
      v[j] = __builtin_nontemporal_load(src + (int64_t)row * vec_per_row);
    }
#pragma unroll
    for (int j = 0; j < KMAX; ++j)
      if (kExact || j0 + j < k) add8(acc, v[j], kRoundEachAdd && j > 0);
  }
  uint32_t o[4];
#pragma unroll
  for (int e = 0; e < 4; ++e)
    o[e] = f32_to_bf16_bits(acc[2 * e]) | (f32_to_bf16_bits(acc[2 * e + 1]) << 16);
  out[i] = make_uint4(o[0], o[1], o[2], o[3]);
}

}  // namespace

hipError_t launch_moe_sum(const uint16_t* in, uint16_t* out, int64_t m, int top_k, int hidden,
                          hipStream_t stream) {
  const int vec_per_row = hidden / 8;
  const int64_t total = m * vec_per_row;
  if (total == 0) return hipSuccess;
  const dim3 grid((unsigned)((total + kThreads - 1) / kThreads));
#define MOE_I8_SUM(ROUND, KMAX, EXACT)                                                             \
  hipLaunchKernelGGL((moe_sum_kernel<ROUND, KMAX, EXACT>), grid, dim3(kThreads), 0, stream,        \
                     reinterpret_cast<const v4i*>(in), reinterpret_cast<uint4*>(out), total, top_k, vec_per_row)
  switch (top_k) {
    case 1: MOE_I8_SUM(false, 1, true); break;
    case 2: MOE_I8_SUM(true, 2, true); break;
    case 3: MOE_I8_SUM(true, 3, true); break;
    case 4: MOE_I8_SUM(true, 4, true); break;
    case 6: MOE_I8_SUM(false, 6, true); break;
    case 8: MOE_I8_SUM(false, 8, true); break;
    case 9: MOE_I8_SUM(false, 9, true); break;
    default: MOE_I8_SUM(false, 4, false); break;
  }
#undef MOE_I8_SUM
  return hipGetLastError();
}

}  // namespace moe_i8
