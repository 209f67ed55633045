// The whole MoE layer of one to a few tokens in two launches, for gfx950.
//
// With so few tokens the layer's kernels are shorter than what lies between them: of the 20 us of a layer of one
// token (8 experts of 1536 x 2048 and 2048 x 768) 38 MB of weights need 6.  Here no rows are gathered per expert and
// nothing is quantised ahead; a routed pair (token, expert) is a matrix-vector product, and an expert that several
// tokens chose is read once, by the first of its pairs:
//
//  * gate_up: a workgroup of four wavefronts takes a handful of channels of one expert in use.  It quantises the rows of
//    the tokens that chose it itself, the first one while the weights are on their way;
//  * down: a workgroup takes eight channels of all tokens, its wavefronts the experts in use.  They quantise the
//    pairs' activations themselves; the results, each rounded as the separate kernels round it, meet in LDS and
//    are added up in ascending order of a token's experts: no alignment, no quantisation launches, no combine launch.
//
// A lane holds 16 consecutive reduction bytes of every row (v_dot4_i32_i8 on registers, sums across the wavefront by
// lane permutes: int32, exact in any order); all of a wavefront's weights, up to 16 KB, are requested before the first
// is used.  What bounds it: one memory latency and the bytes at one token of a small layer, the bytes alone
// where experts are large.
#include "quant_body.hpp"
#include "router_body.hpp"

namespace moe_i8 {
namespace {

constexpr int kGateWaves = 4;
constexpr int down_rows(int c) { return c <= 2 ? 8 : 4; }     // channels of a down workgroup
constexpr int down_waves(int c) { return c == 1 ? 16 : 8; }  // its wavefronts at most

// C: 1 KB pieces of a row (hidden <= 1024 * C)
// kOne: one token, so no expert has two pairs.  kRoute > 0: of one token, which every wavefront routes itself (kRoute
// experts per lane), as far as its pair; the first one writes the routing for the down launch and the caller.
template <int C, bool kOne, int kRoute = 0>
__global__ __launch_bounds__(64 * kGateWaves) void gate_up_few_kernel(FewTokensArgs p, RouteArgs route) {
  constexpr int kThreads = 64 * kGateWaves;
  constexpr int R = C <= 2 ? 8 : C <= 4 ? 4 : 2;  // weight rows of a wavefront: half gate, half up
  constexpr int kVec = (C * 1024 / kQuantVec + kThreads - 1) / kThreads;
  __shared__ __align__(16) int8_t xq[C * 1024];
  __shared__ float part[kGateWaves];
  const int tid = threadIdx.x, lane = lane_id();
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int pairs = p.tokens * p.top_k, K = p.hidden;
  int pair = blockIdx.y;
  // the pairs of this pair's expert: the first one's workgroups take them all
  // the token's row and logits first: their loads are waited for first
  uint4 v[kVec];
  auto fetch = [&] {
    const uint4* x = reinterpret_cast<const uint4*>(p.x + (int64_t)(pair / p.top_k) * K);
#pragma unroll
    for (int i = 0; i < kVec; ++i) v[i] = i * kThreads + tid < K / kQuantVec ? x[i * kThreads + tid] : make_uint4(0u, 0u, 0u, 0u);
  };
  fetch();
  float logits[kRoute > 0 ? kRoute : 1];
  if constexpr (kRoute > 0) route_logits<kRoute>(route, 0, logits);

  int e;
  uint64_t same = 0;
  if constexpr (kRoute > 0) {
    const bool writes = blockIdx.x == 0 && pair == 0 && wave == 0;
    int id;
    float w;
    route_select<kRoute>(route, logits, writes ? p.top_k : pair + 1, id, w);
    if (writes) route_write(route, 0, id, w);
    e = __builtin_amdgcn_readlane(id, pair);
  } else if constexpr (kOne) {
    e = p.topk_ids[pair];
  } else {
    const int id = lane < pairs ? p.topk_ids[lane] : -1;
    e = __builtin_amdgcn_readlane(id, pair);
    same = __ballot(id == e);
    if (__builtin_ctzll(same) != pair) return;
  }
  if (e < 0 || e >= p.num_experts) return;

  const int ch0 = (blockIdx.x * kGateWaves + wave) * (R / 2);
  v4i w[R][C];
  const int8_t* base = p.w1 + (int64_t)e * 2 * p.inter * K;
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int ch = ch0 + r % (R / 2) < p.inter ? ch0 + r % (R / 2) : p.inter - 1;
    const v4i* row = reinterpret_cast<const v4i*>(base + (int64_t)(r < R / 2 ? ch : p.inter + ch) * K);
#pragma unroll
    for (int c = 0; c < C; ++c) w[r][c] = __builtin_nontemporal_load(row + (c * kWave + lane < K / 16 ? c * kWave + lane : 0));
  }
  // lane r < R / 2: scales of channel ch0 + r
  const int mine = ch0 + lane < p.inter ? ch0 + lane : p.inter - 1;
  const float* scales = p.w1_scale + (int64_t)e * 2 * p.inter;
  const float wg = scales[mine], wu = scales[p.inter + mine];

  while (true) {
    float m = 0.0f;
#pragma unroll
    for (int i = 0; i < kVec; ++i) m = fmaxf(m, absmax8(v[i]));
    m = wave_max(m);
    if (lane == 0) part[wave] = m;
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kGateWaves; ++i) m = fmaxf(m, part[i]);
    const float absmax = fmaxf(m, 1e-10f);
    const float inv = 127.0f / absmax, a_scale = absmax / 127.0f;
#pragma unroll
    for (int i = 0; i < kVec; ++i)  // (zeros behind the row)
      if (i * kThreads + tid < C * 1024 / kQuantVec) *reinterpret_cast<uint2*>(xq + (i * kThreads + tid) * kQuantVec) = quant8(v[i], inv);
    __syncthreads();

    const int64_t out = (int64_t)pair * p.inter + ch0 + lane;
    if constexpr (!kOne) same &= same - 1;
    if (same) {  // the next token's row, behind the products of this one's
      pair = __builtin_ctzll(same);
      fetch();
    }
    v4i q[C];
#pragma unroll
    for (int c = 0; c < C; ++c) q[c] = *reinterpret_cast<const v4i*>(xq + (c * kWave + lane) * 16);
    int acc[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
      acc[r] = 0;
#pragma unroll
      for (int c = 0; c < C; ++c) acc[r] = dot16(w[r][c], q[c], acc[r]);
    }
    const int g = wave_totals<R>(acc);
    const int u = dpp_shift_down<R / 2>(g);
    if (lane < R / 2 && ch0 + lane < p.inter) p.act[out] = (uint16_t)silu_mul_epilogue1(g, u, a_scale, wg, wu);
    if (!same) return;
  }
}

// C: 1 KB pieces of a row (inter <= 1024 * C)
// kOne: one token and a wavefront for each of its experts
template <int C, bool kOne>
__global__ __launch_bounds__(64 * (kOne ? 16 : down_waves(C))) void down_few_kernel(FewTokensArgs p) {
  constexpr int R = down_rows(C);
  __shared__ float rows[kFewTokensMaxPairs][R];
  const int lane = lane_id();
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), waves = blockDim.x / kWave;
  const int pairs = p.tokens * p.top_k, K = p.inter;
  const int n0 = blockIdx.x * R;
  const int id = lane < pairs ? p.topk_ids[lane] : -1;
  const float routed = lane < pairs ? p.topk_weights[lane] : 0.0f;

  // the wave-th, (wave + waves)-th, ... expert in use, in the order of their first pairs
  uint64_t left = __ballot(id >= 0 && id < p.num_experts);
  const uint64_t used = left;
  for (int nth = 0; left; ++nth) {
    int e;
    uint64_t same;
    if constexpr (kOne) {
      left = 0;
      e = __builtin_amdgcn_readfirstlane(p.topk_ids[wave]);
      if (e < 0 || e >= p.num_experts) break;
      same = 1ull << wave;
    } else {
      e = __builtin_amdgcn_readlane(id, __builtin_ctzll(left));
      same = __ballot(id == e);
      left &= ~same;
      if (nth % waves != wave) continue;
    }
    uint4 v[2 * C];
    int pair;
    auto fetch = [&] {  // activations of the next pair
      pair = __builtin_ctzll(same);
      same &= same - 1;
      const uint4* x = reinterpret_cast<const uint4*>(p.act + (int64_t)pair * K);
#pragma unroll
      for (int c = 0; c < C; ++c) {
        const bool in = c * kWave + lane < K / 16;
        v[2 * c] = in ? x[2 * (c * kWave + lane)] : make_uint4(0u, 0u, 0u, 0u);
        v[2 * c + 1] = in ? x[2 * (c * kWave + lane) + 1] : make_uint4(0u, 0u, 0u, 0u);
      }
    };
    fetch();
    v4i w[R][C];
    const int8_t* base = p.w2 + (int64_t)e * p.hidden * K;
#pragma unroll
    for (int r = 0; r < R; ++r) {  // hidden is a multiple of 8
      const v4i* row = reinterpret_cast<const v4i*>(base + (int64_t)(n0 + r) * K);
#pragma unroll
      for (int c = 0; c < C; ++c) w[r][c] = __builtin_nontemporal_load(row + (c * kWave + lane < K / 16 ? c * kWave + lane : 0));
    }
    const float ws = p.w2_scale[(int64_t)e * p.hidden + n0 + (lane & (R - 1))];
    while (true) {
      const int at = pair;
      float m = 0.0f;  // (with absmax8 131 registers at C = 2, not 115: 4 tokens on 256 experts of 7168 x 2048 193.5 us, not 188)
#pragma unroll
      for (int c = 0; c < 2 * C; ++c) m = fmaxf(m, absmax8_skip_nan(v[c]));
      const float absmax = fmaxf(wave_max(m), 1e-10f);
      const float inv = 127.0f / absmax, a_scale = absmax / 127.0f;
      v4i q[C];
#pragma unroll
      for (int c = 0; c < C; ++c) {
        const uint2 lo = quant8(v[2 * c], inv), hi = quant8(v[2 * c + 1], inv);
        q[c] = v4i{(int)lo.x, (int)lo.y, (int)hi.x, (int)hi.y};
      }
      const bool more = !kOne && same != 0;
      if (more) fetch();
      int acc[R];
#pragma unroll
      for (int r = 0; r < R; ++r) {
        acc[r] = 0;
#pragma unroll
        for (int c = 0; c < C; ++c) acc[r] = dot16(w[r][c], q[c], acc[r]);
      }
      const int mine = wave_totals<R>(acc);
      const float rw = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(routed), at));
      if (lane < R) rows[at][lane] = bf16_bits_to_f32(down_epilogue1(mine, a_scale, ws, rw) & 0xffffu);
      if (!more) break;
    }
  }
  __syncthreads();
  for (int i = threadIdx.x; i < p.tokens * R; i += blockDim.x) {
    const int token = i / R, c = i % R;
    // the adds round as the stand-alone combine's do; pairs without an expert add nothing
    const bool round_each = p.top_k >= 2 && p.top_k <= 4;
    auto row = [&](int j) { return (used >> (token * p.top_k + j)) & 1 ? rows[token * p.top_k + j][c] : 0.0f; };
    float s = row(0);
    for (int j = 1; j < p.top_k; ++j) {
      s += row(j);
      if (round_each) s = round_to_bf16(s);
    }
    p.out[(int64_t)token * p.hidden + n0 + c] = (uint16_t)f32_to_bf16_bits(s);
  }
}

template <int C>
hipError_t launch_gate_up(const FewTokensArgs& a, const RouteArgs* route, hipStream_t stream) {
  constexpr int kChannels = (C <= 2 ? 8 : C <= 4 ? 4 : 2) / 2 * kGateWaves;
  const dim3 grid((unsigned)((a.inter + kChannels - 1) / kChannels), (unsigned)(a.tokens * a.top_k)), block(64 * kGateWaves);
  const RouteArgs r = route ? *route : RouteArgs{};
  if (route && route_experts_per_lane(a.num_experts) <= 2)
    hipLaunchKernelGGL((gate_up_few_kernel<C, true, 2>), grid, block, 0, stream, a, r);
  else if (route)
    hipLaunchKernelGGL((gate_up_few_kernel<C, true, 4>), grid, block, 0, stream, a, r);
  else if (a.tokens == 1)
    hipLaunchKernelGGL((gate_up_few_kernel<C, true>), grid, block, 0, stream, a, r);
  else
    hipLaunchKernelGGL((gate_up_few_kernel<C, false>), grid, block, 0, stream, a, r);
  return hipGetLastError();
}
template <int C>
hipError_t launch_down(const FewTokensArgs& a, hipStream_t stream) {
  const int pairs = a.tokens * a.top_k;
  const bool one = a.tokens == 1 && pairs <= 16;
  const int most = one ? 16 : down_waves(C);
  const dim3 grid((unsigned)(a.hidden / down_rows(C))), block((unsigned)(64 * (pairs < most ? pairs : most)));
  if (one)
    hipLaunchKernelGGL((down_few_kernel<C, true>), grid, block, 0, stream, a);
  else
    hipLaunchKernelGGL((down_few_kernel<C, false>), grid, block, 0, stream, a);
  return hipGetLastError();
}

}  // namespace

// Layer us, blocks of rows per expert -> this, at 1 / 2 / 3 / 4 / 8 tokens: 20.4 / 25.9 / 30.7 / 35.3 / 55.3 -> 10.9 / 16.7 /
// 22.4 / 27.4 / 47.6 (128 experts of 2048 x 768, 8 per token), 67.3 / 127.3 / 157.3 / 197.5 / 305 -> 55.4 / 107.4 / 141.4 /
// 179.6 / 308 (256 experts of 7168 x 2048).
//
// An expert is taken row after row here, so what decides is how many tokens share one.  An expert that every token
// visits (one of 129 of 4096 x 1408, skewed routing; 17 MB of weights) is the longest chain of the launch: 60.5 / 45.7,
// 63.7 / 54.1, 72.8 / 68.2, 72.9 / 72.6, 78.4 / 85.6 there / here at 2 to 6 tokens.  With small experts that chain is short
// against the launches saved.  The line at 8 MB is on the safe side: evenly routed, 8 tokens on 128 experts of 2880 x
// 960 (7.9 MB) take 98.3 / 74.2, but on ones of 4096 x 1024 (12 MB), which go there, 126.3 / 101.5.
// Where more than seven tokens share every expert the chain of launches is shorter at any size: 8 tokens on one expert of
// 2048 x 1024 17.1 / 18.0, on eight of 2048 x 1280 that all visit 31.6 / 34.5 (7 tokens: 16.9 / 16.5, 31.8 / 31.4).
bool few_tokens_takes(int64_t tokens, int top_k, int num_experts, int hidden, int inter) {
  const bool small_experts = 3ll * hidden * inter <= (8ll << 20);
  return tokens <= (small_experts ? 8 : 4) && tokens * top_k <= kFewTokensMaxPairs && tokens * top_k <= 7ll * num_experts &&
         hidden % 16 == 0 && inter % 16 == 0 && hidden <= 8 * 1024 && inter <= 4 * 1024;
}

bool few_tokens_routes(int64_t tokens, int num_experts) {
  // an expert group is a run of whole lanes: with other numbers of experts per lane than these two a launch of its own
  return tokens == 1 && (route_experts_per_lane(num_experts) == 2 || route_experts_per_lane(num_experts) == 4);
}

hipError_t launch_few_tokens(const FewTokensArgs& a, const RouteArgs* route, hipStream_t stream) {
  hipError_t err;
  switch ((a.hidden + 1023) / 1024) {
    case 1: err = launch_gate_up<1>(a, route, stream); break;
    case 2: err = launch_gate_up<2>(a, route, stream); break;
    case 3: err = launch_gate_up<3>(a, route, stream); break;
    case 4: err = launch_gate_up<4>(a, route, stream); break;
    case 5: err = launch_gate_up<5>(a, route, stream); break;
    case 6: err = launch_gate_up<6>(a, route, stream); break;
    case 7: err = launch_gate_up<7>(a, route, stream); break;
    default: err = launch_gate_up<8>(a, route, stream); break;
  }
  if (err != hipSuccess) return err;
  switch ((a.inter + 1023) / 1024) {
    case 1: return launch_down<1>(a, stream);
    case 2: return launch_down<2>(a, stream);
    case 3: return launch_down<3>(a, stream);
    default: return launch_down<4>(a, stream);
  }
}

}  // namespace moe_i8
