// Shared device helpers and launcher declarations for the gfx950 INT8 MoE kernels.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <atomic>

namespace moe_i8 {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));

constexpr int kWave = 64;
constexpr int kMaxExperts = 1024;  // == MOE_I8_MAX_EXPERTS

__device__ __forceinline__ int lane_id() { return threadIdx.x & (kWave - 1); }

// Compute units of the current device (asked once per process; 256 if the runtime will not say).
inline int device_cu_count() {
  static const int count = [] {
    int dev = 0, n = 0;
    if (hipGetDevice(&dev) != hipSuccess) return 256;
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n < 8) return 256;
    return n;
  }();
  return count;
}

// A kernel's limit of dynamic LDS, raised on each device the first time a launch goes there (one object per kernel).
class DynamicLds {
 public:
  hipError_t allow(const void* kernel, int bytes) {
    int dev = 0;
    hipError_t err = hipGetDevice(&dev);
    if (err != hipSuccess) return err;
    const uint64_t bit = 1ull << (dev & 63);
    if (dev < 64 && (done_.load(std::memory_order_acquire) & bit)) return hipSuccess;
    err = hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
    if (err == hipSuccess) done_.fetch_or(bit, std::memory_order_release);
    return err;
  }

 private:
  std::atomic<uint64_t> done_{0};
};

__device__ __forceinline__ float bf16_bits_to_f32(uint32_t b) { return __uint_as_float(b << 16); }

// fp32 -> bf16 bits, round to nearest even; NaN stays a quiet NaN.
__device__ __forceinline__ uint32_t f32_to_bf16_bits(float f) {
  uint32_t u = __float_as_uint(f);
  if ((u & 0x7fffffffu) > 0x7f800000u) return (u >> 16) | 0x40u;
  u += 0x7fffu + ((u >> 16) & 1u);
  return u >> 16;
}

__device__ __forceinline__ float round_to_bf16(float f) {
  return bf16_bits_to_f32(f32_to_bf16_bits(f));
}

// Wave-wide reductions on the VALU's data-parallel-primitive lane permutes (no LDS traffic, a few
// cycles per step): quads, half rows and rows of 16 by mirror permutes, then row 15 -> next row and
// row 31 -> upper half broadcasts leave the total in lane 63, which is read back as a scalar.
template <int kCtrl, int kRowMask>
__device__ __forceinline__ float dpp_move(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(v), __float_as_int(v), kCtrl, kRowMask, 0xf, false));
}
__device__ __forceinline__ float wave_reduce_max(float v) {
  v = fmaxf(v, dpp_move<0xb1, 0xf>(v));   // quad_perm [1,0,3,2]
  v = fmaxf(v, dpp_move<0x4e, 0xf>(v));   // quad_perm [2,3,0,1]
  v = fmaxf(v, dpp_move<0x141, 0xf>(v));  // row_half_mirror
  v = fmaxf(v, dpp_move<0x140, 0xf>(v));  // row_mirror
  v = fmaxf(v, dpp_move<0x142, 0xa>(v));  // row_bcast:15 into rows 1 and 3
  v = fmaxf(v, dpp_move<0x143, 0xc>(v));  // row_bcast:31 into rows 2 and 3
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 63));
}
__device__ __forceinline__ float wave_reduce_sum(float v) {
  v += dpp_move<0xb1, 0xf>(v);
  v += dpp_move<0x4e, 0xf>(v);
  v += dpp_move<0x141, 0xf>(v);
  v += dpp_move<0x140, 0xf>(v);
  // the broadcasts must add only into the rows they target: elsewhere the permute returns the
  // lane's own value and would double it
  const float b15 = dpp_move<0x142, 0xa>(v);
  v += (lane_id() & 16) ? b15 : 0.0f;
  const float b31 = dpp_move<0x143, 0xc>(v);
  v += (lane_id() & 32) ? b31 : 0.0f;
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 63));
}

// Inclusive add-scan over the 64 lanes on the same lane permutes: shifts by 1, 2, 4 and 8 inside rows
// of 16 (a lane without a source adds 0), then the total of row 0 / 2 into every lane of row 1 / 3 and
// the total of the lower half into the upper half.
__device__ __forceinline__ int wave_inclusive_scan_add(int v) {
  v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, false);  // row_shr:1
  v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, false);  // row_shr:2
  v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, false);  // row_shr:4
  v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, false);  // row_shr:8
  v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);  // row_bcast:15 into rows 1 and 3
  v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);  // row_bcast:31 into rows 2 and 3
  return v;
}

// Sums of R values over the wavefront, R = 2, 4 or 8: value l % R's in lane l.  Two values are folded into one by every
// lane keeping the one it will end with and handing the other to its partner: 28 operations for eight values where
// eight reductions of their own take 56.
template <int R>
__device__ __forceinline__ int wave_totals(const int (&v)[R]) {
  const int lane = lane_id();
  // partner at distance 1, 2 (quads), 4 (a shift up or down by half of eight lanes), 8 (rotation of a row of sixteen)
  auto partner1 = [](int x) { return __builtin_amdgcn_update_dpp(0, x, 0xb1, 0xf, 0xf, false); };
  auto partner2 = [](int x) { return __builtin_amdgcn_update_dpp(0, x, 0x4e, 0xf, 0xf, false); };
  auto partner4 = [](int x) {
    const int up = __builtin_amdgcn_update_dpp(0, x, 0x104, 0xf, 0x5, false);   // row_shl:4 into lanes 0-3 and 8-11 of a row
    return __builtin_amdgcn_update_dpp(up, x, 0x114, 0xf, 0xa, false);          // row_shr:4 into the others
  };
  auto fold = [&](int a, int b, int bit, auto partner) { return (lane & bit ? b : a) + partner(lane & bit ? a : b); };
  int x;
  if constexpr (R == 2) {
    x = fold(v[0], v[1], 1, partner1);
    x += partner2(x);
    x += partner4(x);
  } else if constexpr (R == 4) {
    x = fold(fold(v[0], v[1], 1, partner1), fold(v[2], v[3], 1, partner1), 2, partner2);
    x += partner4(x);
  } else {
    static_assert(R == 8, "2, 4 or 8 values");
    x = fold(fold(fold(v[0], v[1], 1, partner1), fold(v[2], v[3], 1, partner1), 2, partner2),
             fold(fold(v[4], v[5], 1, partner1), fold(v[6], v[7], 1, partner1), 2, partner2), 4, partner4);
  }
  x += __builtin_amdgcn_update_dpp(0, x, 0x128, 0xf, 0xf, false);  // row_ror:8
  const auto rows = __builtin_amdgcn_permlane16_swap(x, x, false, false);
  x = (int)rows[0] + (int)rows[1];
  const auto halves = __builtin_amdgcn_permlane32_swap(x, x, false, false);
  return (int)halves[0] + (int)halves[1];
}

// lane l: the value of lane l + kBy of its row of sixteen (0 past its end)
template <int kBy>
__device__ __forceinline__ int dpp_shift_down(int v) {
  return __builtin_amdgcn_update_dpp(0, v, 0x100 + kBy, 0xf, 0xf, true);
}

// acc + the products of 16 int8 pairs (v_dot4_i32_i8)
__device__ __forceinline__ int dot16(const v4i& a, const v4i& b, int acc) {
#pragma unroll
  for (int i = 0; i < 4; ++i) acc = __builtin_amdgcn_sdot4(a[i], b[i], acc, false);
  return acc;
}

typedef float f2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf2 __attribute__((ext_vector_type(2)));

// Two fp32 -> packed bf16 (v_cvt_pk_bf16_f32, round to nearest even); lo in bits 15:0.
__device__ __forceinline__ uint32_t pack_bf16(float lo, float hi) {
  const bf2 b = __builtin_convertvector(f2{lo, hi}, bf2);
  return *reinterpret_cast<const uint32_t*>(&b);
}

// SiLU with the hardware exp2 / reciprocal approximations (a few fp32 ulp); every GEMM family uses
// this one definition so that the result does not depend on which kernel ran.
__device__ __forceinline__ float fast_silu(float g) {
  return g * __builtin_amdgcn_rcpf(1.0f + __expf(-g));
}

// Four (gate, up) accumulator pairs -> four bf16 outputs with the rounding points of an unfused
// pipeline: gate and up rounded to bf16, silu(gate) rounded to bf16, product rounded to bf16.
__device__ __forceinline__ uint2 silu_mul_epilogue4(const int (&g)[4], const int (&u)[4], float a_scale,
                                                    const float4& wg, const float4& wu) {
  const float wgv[4] = {wg.x, wg.y, wg.z, wg.w};
  const float wuv[4] = {wu.x, wu.y, wu.z, wu.w};
  float h[4];
#pragma unroll
  for (int r = 0; r < 4; r += 2) {
    const uint32_t g2 = pack_bf16((float)g[r] * a_scale * wgv[r], (float)g[r + 1] * a_scale * wgv[r + 1]);
    const uint32_t u2 = pack_bf16((float)u[r] * a_scale * wuv[r], (float)u[r + 1] * a_scale * wuv[r + 1]);
    const uint32_t s2 =
        pack_bf16(fast_silu(__uint_as_float(g2 << 16)), fast_silu(__uint_as_float(g2 & 0xffff0000u)));
    h[r] = __uint_as_float(s2 << 16) * __uint_as_float(u2 << 16);
    h[r + 1] = __uint_as_float(s2 & 0xffff0000u) * __uint_as_float(u2 & 0xffff0000u);
  }
  return make_uint2(pack_bf16(h[0], h[1]), pack_bf16(h[2], h[3]));
}

// The same of one pair; the result in the low 16 bits.
__device__ __forceinline__ uint32_t silu_mul_epilogue1(int g, int u, float a_scale, float wg, float wu) {
  const uint32_t gu = pack_bf16((float)g * a_scale * wg, (float)u * a_scale * wu);
  const uint32_t s = pack_bf16(fast_silu(__uint_as_float(gu << 16)), 0.0f);
  return pack_bf16(__uint_as_float(s << 16) * __uint_as_float(gu & 0xffff0000u), 0.0f);
}
__device__ __forceinline__ uint32_t down_epilogue1(int acc, float a_scale, float ws, float rw) {
  return pack_bf16((float)acc * a_scale * ws * rw, 0.0f);
}

// Four down-projection accumulators -> four bf16 outputs: acc * a_scale * w_scale * routed weight.
__device__ __forceinline__ uint2 down_epilogue4(const int (&acc)[4], float a_scale, const float4& ws, float rw) {
  return make_uint2(pack_bf16((float)acc[0] * a_scale * ws.x * rw, (float)acc[1] * a_scale * ws.y * rw),
                    pack_bf16((float)acc[2] * a_scale * ws.z * rw, (float)acc[3] * a_scale * ws.w * rw));
}

// ---- launchers (defined one per .hip file; all asynchronous on `stream`) ----

struct AlignArgs {
  const int32_t* topk_ids;
  int64_t num_pairs;
  int num_experts;
  int block_size;
  int32_t* sorted_token_ids;
  int64_t sorted_cap;
  int32_t* expert_ids;
  int64_t expert_cap;
  int32_t* num_tokens_post_padded;
  int32_t* workspace;
};
int64_t align_workspace_ints(int64_t num_pairs, int num_experts);
hipError_t launch_align(const AlignArgs& a, hipStream_t stream);
int align_launches(const AlignArgs& a);  // 1, 2 or 3 by the number of pairs

struct QuantArgs {
  const uint16_t* x;  // bf16 bits
  int64_t src_rows;
  int cols;
  int64_t row_stride;
  const int32_t* gather;
  int gather_div;
  int64_t rows;
  int8_t* q;
  float* scale;
  // Output row of input row r is (r / rows_per_group) * out_rows_per_group + out_row_offset +
  // r % rows_per_group; rows_per_group == 0 means out row == r.  Lets one call drop the gate or
  // the up projection of every expert into its half of a stacked [E, 2I, H] tensor.
  int64_t rows_per_group = 0;
  int64_t out_rows_per_group = 0;
  int64_t out_row_offset = 0;
  int round_even = 0;  // activations: ties to even instead of away from zero
  int q_stride = 0;    // row quantiser only: bytes from one row of q to the next, zero-filled behind cols; 0 = cols
  // Row quantiser only: also write the routing of a dense layer seen as one expert that every row
  // visits (rows in order, padded to whole blocks with the sentinel, used blocks owned by expert
  // 0, the rest of both arrays marked unused) — one launch less in front of a dense GEMM.
  int32_t* route_sorted = nullptr;  // null: no routing
  int32_t* route_expert_ids = nullptr;
  int32_t* route_npp = nullptr;
  int route_block = 0;
  int64_t route_cap = 0;
};
hipError_t launch_quant_rows(const QuantArgs& a, hipStream_t stream);
// Router: scores -> (grouped) top-k -> weights, one wavefront per token.
enum ScoreFunc { kScoreSoftmax = 0, kScoreSigmoid = 1, kScoreTopkSoftmax = 2 };
struct RouteArgs {
  const float* logits;  // [m, num_experts]
  int64_t m;
  int num_experts;
  int top_k;
  int score_func;
  const float* bias;  // [num_experts] or null; added for selection only
  int num_groups;     // 1 = no group pre-selection
  int topk_groups;
  int group_top2;  // group score: 1 = sum of the two largest selection values, 0 = the largest
  int renormalize;
  float route_scale;
  float* weights;  // [m, top_k]
  int32_t* ids;    // [m, top_k]
  void* capture;   // compact copy of ids at capture[tok * capture_stride + capture_offset + j]
  int capture_bytes;  // 0 = none, 1 = uint8, 2 = uint16
  int64_t capture_stride;
  int64_t capture_offset;
};
int route_experts_per_lane(int num_experts);
hipError_t launch_route_topk(const RouteArgs& a, hipStream_t stream);

// Per-output-channel weight quantisation (round to nearest even of w / scale, scale = absmax / 127) of 1 to
// 3 matrices; the first two of three have the same row length.
hipError_t launch_quant_weights(const QuantArgs* a, int count, hipStream_t stream);
// moe_align and the quantisation of `q` in one launch; only when align_quant_fusable() says so.
bool align_quant_fusable(const AlignArgs& a, const QuantArgs& q);
hipError_t launch_align_quant(const AlignArgs& a, const QuantArgs& q, hipStream_t stream);

enum GemmMode { kGateUpSilu = 0, kDown = 1, kAccI32 = 2 };

struct GemmArgs {
  int mode;
  const uint16_t* a_bf16 = nullptr;  // down, streaming family only: bf16 activations [P, K] quantised in the kernel
  bool a_round_even = false;         // ... rounding ties to even (dense path) instead of away from zero (MoE path)
  const int8_t* a_q;      // [*, K] activations (int8)
  const float* a_scale;   // per activation row
  const int8_t* w;        // [E, N, K]
  const float* w_scale;   // [E, N]
  const float* row_weight;  // [P] routed weights (down); null = 1
  const int32_t* sorted_token_ids;
  const int32_t* expert_ids;
  const int32_t* num_tokens_post_padded;
  int64_t num_pairs;
  int row_div;  // activation row of pair t is t / row_div
  int num_experts;
  int n;  // weight rows per expert (2I for gate_up, H for down)
  int k;  // reduction length
  int block_size;
  int64_t sorted_cap;
  void* out;  // bf16 [P, I] | bf16 [P, H] | int32 [P, N]
  int64_t max_rows_per_expert = 0;  // upper bound if the caller knows one (the token count), else 0
  bool expert_ids_ascend = false;   // expert_ids is known to come from moe_align (non-decreasing over the used blocks)
  bool identity = false;            // ... and one expert owns all of them, every block is used: a dense layer
  int tile_geometry = 0;            // LDS-tiled family: kTileAuto, kTileWide (256-row tiles), kTileDeep (128-row tiles) or kTileRing (256-row tiles, four-stage ring; on demand only)
};
constexpr int kTileAuto = 0, kTileWide = 1, kTileDeep = 2, kTileRing = 3;
// The LDS-tiled family picks its deep geometry up to this many routed rows per expert (launches with 2 GB of weights and more: fewer).
constexpr int kTileDeepRowsPerExpert = 104, kTileDeepRowsLongStream = 80;
constexpr int64_t kLongStreamBytes = 2048ll << 20;  // weights of a launch
hipError_t launch_gemm_stream(const GemmArgs& a, hipStream_t stream);
// register-only int8 MFMA loop (measurement aid): sink holds mfma_probe_sink_bytes(workgroups)
int64_t mfma_probe_sink_bytes(int workgroups);
double mfma_probe_ops(int workgroups, int iters);
hipError_t launch_mfma_probe(bool random_operands, int workgroups, int iters, int32_t* sink, hipStream_t stream);
bool gemm_stream_fuses_quant(const GemmArgs& a);  // the down GEMM of this family can quantise bf16 activations itself
// The streaming family's kernel for a handful of tokens (launch_gemm_stream uses it where it takes the problem).
bool gemm_split_takes(const GemmArgs& a);
bool gemm_split_fuses_quant(int k);
hipError_t launch_gemm_split(const GemmArgs& a, hipStream_t stream);
hipError_t launch_gemm_tile(const GemmArgs& a, hipStream_t stream);
bool gemm_tile_supports(const GemmArgs& a);
bool gemm_tile_prefers_deep(const GemmArgs& a);
int gemm_tile_geometry(const GemmArgs& a);  // kTileWide or kTileDeep (kTileRing on demand): what a launch of the family would use
bool gemm_wide_supports(const GemmArgs& a);
hipError_t launch_gemm_wide(const GemmArgs& a, hipStream_t stream);
bool gemm_deep_supports(const GemmArgs& a);
hipError_t launch_gemm_deep(const GemmArgs& a, hipStream_t stream);
hipError_t launch_gemm_narrow(const GemmArgs& a, hipStream_t stream);
bool gemm_narrow_supports(const GemmArgs& a);

// One weight matrix that every row visits: out = epilogue(a_q[m, k] x w[n, k]^T).
struct DenseArgs {
  int mode;  // kGateUpSilu or kDown
  const int8_t* a_q;  // rows of dense_row_stride(k) bytes, zero from k on
  const float* a_scale;
  const int8_t* w;
  const float* w_scale;
  void* out;
  int64_t m;
  int n;
  int k;
};
int dense_row_stride(int k);
// How a dense GEMM is cut up, chosen once per GEMM and launched with: an entry of the kernel's table of tiles.
struct DensePick {
  int entry;  // -1: the dense kernel is not the one for this problem
  float us;   // what the product is expected to take, by whichever kernel
};
// `wide_allowed`: the 256-row tiles of the LDS-tiled family can run the problem too and are preferred where they are expected to
// be faster.
DensePick gemm_dense_pick(int mode, int64_t m, int n, int k, bool wide_allowed);
struct DenseTile {
  int rows;
  int channels;  // weight rows
};
DenseTile gemm_dense_tile(int entry);
bool gemm_dense_through(int mode, int64_t m, int n);  // results are written through to memory
hipError_t launch_gemm_dense(const DenseArgs& a, int entry, hipStream_t stream);

// The same for a few rows, which the launch quantises itself (ties to even).
struct DenseFewArgs {
  int mode;           // kGateUpSilu or kDown
  const uint16_t* x;  // [m, k] bf16
  const int8_t* w;
  const float* w_scale;
  uint16_t* out;
  int m;
  int n;
  int k;
};
constexpr int kDenseFewRows = 16;
bool dense_few_takes(int64_t m, int n, int k);
float dense_few_estimate(int64_t m, int n, int k);  // us, against the tiles of the kernel below
hipError_t launch_dense_few(const DenseFewArgs& a, hipStream_t stream);
// The dense kernel that quantises its own rows (ties to even): the entry of its table for this problem, -1 if it is not the one.
// `few`: the kernel of a few rows would run it otherwise; if not, `us`: what the quantised product is expected to take.
constexpr int kDenseRowsFrom = 5;  // rows
int dense_rows_pick(int64_t m, int n, int k, bool few, float us);
DenseTile dense_rows_tile(int entry);
hipError_t launch_dense_rows(const DenseFewArgs& a, int entry, hipStream_t stream);

// The whole layer of a few tokens in two launches: act holds tokens * top_k rows of inter bf16.
struct FewTokensArgs {
  const uint16_t* x;  // [tokens, hidden]
  const int8_t* w1;   // [num_experts, 2 * inter, hidden]
  const float* w1_scale;
  const int8_t* w2;   // [num_experts, hidden, inter]
  const float* w2_scale;
  const float* topk_weights;
  const int32_t* topk_ids;
  uint16_t* act;
  uint16_t* out;
  int tokens;
  int top_k;
  int num_experts;
  int hidden;
  int inter;
};
constexpr int kFewTokensMaxPairs = 64;  // one lane per pair
bool few_tokens_takes(int64_t tokens, int top_k, int num_experts, int hidden, int inter);
// `route`: the first launch routes the token too and writes topk_weights and topk_ids; only when few_tokens_routes() says so.
bool few_tokens_routes(int64_t tokens, int num_experts);
hipError_t launch_few_tokens(const FewTokensArgs& a, const RouteArgs* route, hipStream_t stream);

hipError_t launch_moe_sum(const uint16_t* in, uint16_t* out, int64_t m, int top_k, int hidden,
                          hipStream_t stream);

}  // namespace moe_i8
