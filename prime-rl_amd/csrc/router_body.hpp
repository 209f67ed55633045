// Routing of one token by one 64-lane wavefront, shared by the router launch and by the launch that routes a single token
// and starts its layer.
//
// Lane l holds experts [l*C, (l+1)*C) in registers (C = 1, 2, 4, 8 or 16, so up to 1024 experts), which makes every
// expert group a run of whole lanes: group reductions are xor-butterflies over that run.  Selection is k rounds of a
// wave-wide arg-max: the maximum by lane permutes on the VALU, then a ballot of the lanes that hold it; the
// lowest such lane wins, and inside a lane the lowest slot, so equal values resolve to the lowest
// expert index and the result comes out in descending order.
//
// Arithmetic is fp32 throughout.  score: softmax over all experts, sigmoid, or the raw logit
// (softmax over the selected k afterwards).  A selection bias is added for choosing only; the
// returned weights come from the unbiased scores, optionally divided by (their sum + 1e-20) and
// multiplied by a scale.
#pragma once

#include "common.hpp"

namespace moe_i8 {

template <int C>
__device__ __forceinline__ void route_logits(const RouteArgs& a, int64_t tok, float (&logits)[C]) {
  const float* row = a.logits + tok * (int64_t)a.num_experts;
#pragma unroll
  for (int j = 0; j < C; ++j) logits[j] = row[lane_id() * C + j < a.num_experts ? lane_id() * C + j : 0];
}

constexpr float kNegInf = -__builtin_huge_valf();

// Lowest lane whose value equals the wave-wide maximum of `v` (lanes with `live` false never win
// unless no lane is live, which the callers exclude).
__device__ __forceinline__ int wave_argmax_lane(float v, bool live) {
  const float top = wave_reduce_max(live ? v : kNegInf);
  const uint64_t holders = __ballot(live && v == top);
  return __ffsll((unsigned long long)holders) - 1;
}

// One token by one wavefront; logits(j): logit of expert lane * C + j.  Returns in lane j < k the j-th expert and its
// score; only the first `rounds` of them.
template <int C>
__device__ __forceinline__ void route_select(const RouteArgs& a, const float (&logits)[C], int rounds, int& my_id, float& my_w) {
  const int lane = lane_id();
  const int E = a.num_experts;
  const int e0 = lane * C;

  float s[C];  // unbiased score (the source of the returned weights)
  float v[C];  // selection value
#pragma unroll
  for (int j = 0; j < C; ++j) s[j] = e0 + j < E ? logits[j] : kNegInf;

  if (a.score_func == kScoreSoftmax) {
    float mx = kNegInf;
#pragma unroll
    for (int j = 0; j < C; ++j) mx = fmaxf(mx, s[j]);
    mx = wave_reduce_max(mx);
    float sum = 0.0f;
#pragma unroll
    for (int j = 0; j < C; ++j) {
      s[j] = e0 + j < E ? expf(s[j] - mx) : 0.0f;
      sum += s[j];
    }
    sum = wave_reduce_sum(sum);
#pragma unroll
    for (int j = 0; j < C; ++j) s[j] = s[j] / sum;
  } else if (a.score_func == kScoreSigmoid) {
#pragma unroll
    for (int j = 0; j < C; ++j) s[j] = 1.0f / (1.0f + expf(-s[j]));
  }
#pragma unroll
  for (int j = 0; j < C; ++j) {
    v[j] = kNegInf;
    if (e0 + j < E) v[j] = a.bias ? s[j] + a.bias[e0 + j] : s[j];
  }

  if (a.num_groups > 1) {
    // group score = largest (or sum of the two largest) selection values of the group
    const int lanes_per_group = E / a.num_groups / C;
    float t1 = kNegInf, t2 = kNegInf;
#pragma unroll
    for (int j = 0; j < C; ++j) {
      t2 = fmaxf(t2, fminf(t1, v[j]));
      t1 = fmaxf(t1, v[j]);
    }
    for (int d = 1; d < lanes_per_group; d <<= 1) {
      const float o1 = __shfl_xor(t1, d), o2 = __shfl_xor(t2, d);
      t2 = fmaxf(fminf(t1, o1), fmaxf(t2, o2));
      t1 = fmaxf(t1, o1);
    }
    const float group_score = a.group_top2 ? t1 + t2 : t1;
    const int group = lane / lanes_per_group;
    bool chosen = false;
    for (int it = 0; it < a.topk_groups; ++it) {
      const int win = wave_argmax_lane(group_score, !chosen && group < a.num_groups) / lanes_per_group;
      if (group == win) chosen = true;
    }
#pragma unroll
    for (int j = 0; j < C; ++j) v[j] = chosen ? v[j] : kNegInf;
  }

  uint32_t taken = 0u;
  my_w = 0.0f;
  my_id = 0;
  for (int it = 0; it < rounds; ++it) {
    float best_v = kNegInf, best_s = 0.0f;
    int best_j = -1;
#pragma unroll
    for (int j = 0; j < C; ++j) {
      const bool open = e0 + j < E && !((taken >> j) & 1u);
      if (open && (best_j < 0 || v[j] > best_v)) {
        best_v = v[j];
        best_s = s[j];
        best_j = j;
      }
    }
    const int owner = wave_argmax_lane(best_v, best_j >= 0);
    const int e = __builtin_amdgcn_readlane(e0 + best_j, owner);
    const float w = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(best_s), owner));
    if (lane == owner) taken |= 1u << best_j;
    if (lane == it) {
      my_w = w;
      my_id = e;
    }
  }
}

// The weights of the k selected experts, and everything written where it belongs.
__device__ __forceinline__ void route_write(const RouteArgs& a, int64_t tok, int my_id, float my_w) {
  const int lane = lane_id(), k = a.top_k;
  const bool mine = lane < k;
  if (a.score_func == kScoreTopkSoftmax) {
    const float mx = wave_reduce_max(mine ? my_w : kNegInf);
    const float ex = mine ? expf(my_w - mx) : 0.0f;
    my_w = ex / wave_reduce_sum(ex);
  }
  if (a.renormalize) my_w = my_w / (wave_reduce_sum(mine ? my_w : 0.0f) + 1e-20f);
  my_w *= a.route_scale;
  if (mine) {
    a.weights[tok * k + lane] = my_w;
    a.ids[tok * k + lane] = my_id;
    const int64_t at = tok * a.capture_stride + a.capture_offset + lane;
    if (a.capture_bytes == 1) static_cast<uint8_t*>(a.capture)[at] = (uint8_t)my_id;
    if (a.capture_bytes == 2) static_cast<uint16_t*>(a.capture)[at] = (uint16_t)my_id;
  }
}

}  // namespace moe_i8
