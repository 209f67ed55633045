// C-ABI of libmoe_i8.so: argument validation, workspace carving and kernel launches.
// Nothing here allocates device memory or synchronises; every launch goes to the caller's stream.
#include <stdarg.h>
#include <stdio.h>

#include <condition_variable>
#include <mutex>
#include <new>

#include "../../include/moe_i8.h"
#include "common.hpp"

namespace {

thread_local char g_error[512] = "";

int fail(int code, const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_error, sizeof(g_error), fmt, ap);
  va_end(ap);
  return code;
}

int check_launch(hipError_t err, const char* what) {
  if (err == hipSuccess) return MOE_I8_OK;
  return fail(MOE_I8_ELAUNCH, "%s: %s", what, hipGetErrorString(err));
}

// A call's turn on its workspace, while it issues its launches.  Calls of several threads on one stream may share a
// workspace, since the stream runs them one after the other, but only if their launches do not interleave.  A thread
// that waits here waits for calls on the same workspace and for nothing else.  The turns taken are a list through the
// calls' own stack frames: nothing is allocated, nothing throws.
class WorkspaceTurn {
 public:
  explicit WorkspaceTurn(const void* workspace) : workspace_(workspace) {
    std::unique_lock<std::mutex> lock(state().mutex);
    while (taken()) state().ended.wait(lock);
    next_ = state().first;
    state().first = this;
  }
  ~WorkspaceTurn() {
    {
      std::lock_guard<std::mutex> lock(state().mutex);
      WorkspaceTurn** at = &state().first;
      while (*at != this) at = &(*at)->next_;
      *at = next_;
    }
    state().ended.notify_all();
  }
  WorkspaceTurn(const WorkspaceTurn&) = delete;

 private:
  struct State {
    std::mutex mutex;
    std::condition_variable ended;
    WorkspaceTurn* first = nullptr;
  };
  static State& state() {
    alignas(State) static char memory[sizeof(State)];
    static State* s = new (memory) State;  // never destroyed: threads may outlive static objects
    return *s;
  }
  bool taken() const {
    for (const WorkspaceTurn* t = state().first; t; t = t->next_)
      if (t->workspace_ == workspace_) return true;
    return false;
  }
  const void* workspace_;
  WorkspaceTurn* next_;
};

bool valid_block_size(int b) { return b == 16 || b == 32 || b == 64 || b == 128; }

int64_t align_up(int64_t v, int64_t a) { return (v + a - 1) / a * a; }

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

int check_gemm_common(const void* a_q, const void* w, const int32_t* sorted, const int32_t* eids,
                      const int32_t* npp, const void* out, int64_t num_pairs, int num_experts,
                      int n, int k, int block_size, int64_t sorted_cap, int variant) {
  if (!a_q || !w || !sorted || !eids || !npp || !out) return fail(MOE_I8_EINVAL, "null pointer");
  if (!aligned16(a_q) || !aligned16(w) || !aligned16(out))
    return fail(MOE_I8_EINVAL, "activation, weight and output pointers must be 16-byte aligned");
  if (num_pairs < 0 || num_pairs > INT32_MAX - 1) return fail(MOE_I8_EINVAL, "num_pairs out of range");
  if (num_experts < 1 || num_experts > MOE_I8_MAX_EXPERTS)
    return fail(MOE_I8_EINVAL, "num_experts must be in [1, %d]", MOE_I8_MAX_EXPERTS);
  if (!valid_block_size(block_size)) return fail(MOE_I8_EINVAL, "block_size must be 16, 32, 64 or 128");
  if (n < 16 || n % 16) return fail(MOE_I8_EINVAL, "output channels (%d) must be a positive multiple of 16", n);
  if (k < 64 || k % 64) return fail(MOE_I8_EINVAL, "reduction length (%d) must be a positive multiple of 64", k);
  if (sorted_cap < moe_i8_sorted_capacity(num_pairs, num_experts, block_size))
    return fail(MOE_I8_EWORKSPACE, "sorted_token_ids capacity %lld too small", (long long)sorted_cap);
  if (variant < MOE_I8_GEMM_AUTO || variant > MOE_I8_GEMM_TILE_RING)
    return fail(MOE_I8_EINVAL, "unknown GEMM variant %d", variant);
  return MOE_I8_OK;
}

// The streaming family reads an expert's weights once per 16 of its rows: it is the fastest kernel
// while every block fits one such pass, and loses badly as soon as a few experts hold more (a
// shared expert that every token visits, skewed routing), which the host cannot see.  It is
// therefore picked where no expert can hold more than 16 rows (it holds at most one per token),
// or where there is at most one routed row per expert on average.  Launches with 2 GB of weights and more run long enough
// for the narrow tiles' slower start not to count, and their deeper prefetch wins earlier: layer us, streaming / narrow, of
// DeepSeek-V3 at 9 / 16 / 32 tokens 338 / 332, 476 / 469, 656 / 642 (0.2-0.4 GB, Qwen3-30B-A3B at 10 / 16: 60 / 62, 75 / 78.5).
// Why not lower: 8 rows from 0.5 GB on would cost evenly spread layers of 0.56 and 1.4 GB 1-2 %, 4 rows from 2 GB on
// layers of 2.5 GB 1-4 %, and which routing a call has the host cannot see.  By how many per cent narrow takes longer, at 5 / 8 /
// 12 / 16 tokens, evenly spread | Zipf routing, by the weight bytes of the gate_up launch:
//   0.4 GB (128 experts of 2048 x 768)  8 / 8 / 2 / 6 | 9 / 6 / 4 / -2        0.56 (96 of 3072 x 1024)  2 / -1 / 1 / -2 | 2 / 3 / 2 / -2
//   1.4 (128 of 4096 x 1408)  1 / 1 / 2 / 2 | -1 / 0 / -5 / -6, with a shared expert -1 / 0 / 1 / 1 | 0 / -1 / -6 / -8
//   1.9 (128 of 5120 x 1536)  -4 / -2 / -2 / -1 | -7 / -5 / -4 / -5           2.5 (128 of 4096 x 2560)  1 / 2 / 0 / -2 | -4 / 4 / -1 / 0
//   2.8 (96 of 6144 x 2560)  -1 / -1 / -1 / 0 | -5 / -4 / -2 / -4             7 (256 of 7168 x 2048)  -2 / -2 / -1 / -1 | -5 / -4 / -4 / -6
// Given away: the negative figures of 0.56 to 1.9 GB at all and of 2.8 and 7 GB at up to 8 tokens.  A launch of 2.5 GB whose down
// GEMM (1.25) keeps streaming is 2 % slower than with both streaming under Zipf routing, up to 2 % faster evenly routed.
constexpr int kStreamMaxRows = 16, kStreamMaxRowsLongStream = 8;
constexpr int kStreamRowsPerExpert = 1;
constexpr int kSelfQuantMaxInter = 1024;  // longest reduction moe_i8_gemm_down_bf16 takes for any routing

int tile_geometry_of(int variant) {
  return variant == MOE_I8_GEMM_TILE_WIDE ? moe_i8::kTileWide
         : variant == MOE_I8_GEMM_TILE_DEEP ? moe_i8::kTileDeep
         : variant == MOE_I8_GEMM_TILE_RING ? moe_i8::kTileRing
                                            : moe_i8::kTileAuto;
}

// Routed rows per expert up to which the narrow tiles beat the deep geometry of the LDS-tiled family.
// The narrow tiles (64 x 128 tasks) start up faster and balance better; the deep tiles stream an
// expert's weights once for up to 128 rows, which counts the more the longer a launch runs and the
// more the routing is skewed.  Where evenly spread and Zipf routing (expert popularity falling with rank^-1.2) disagree, which
// the host cannot see, the line takes the smaller loss.  Measured on launches of 0.16 to 7 GB of 13 layer shapes; us of the
// launch, narrow / deep, at rows per expert, evenly | Zipf:
//   0.38 GB (128 experts of 2048 x 768, gate_up)  32: 66.1 / 68.6 | 57.8 / 60.4   40: 69.6 / 69.7 | 60.4 / 59.0
//   0.56 GB (96 of 3072 x 1024, gate_up)  20: 93.3 / 99.9 | 75.5 / 87.5   28: 96.3 / 101 | 88.0 / 88.8   36: 102 / 102 | 96.6 / 91.9
//   0.69 GB (129 of 4096 x 1408, down)  16: 128 / 131 | 75.3 / 74.0   20: 131 / 132 | 85.0 / 82.9   24: 135 / 133 | 96.9 / 90.4
//   1.4 GB (the same, gate_up)  16: 239 / 244 | 139 / 139   20: 244 / 248 | 155 / 148   24: 243 / 251 | 175 / 164
//   1.9 GB (128 of 5120 x 1536, gate_up)  16: 305 / 305 | 179 / 189   20: 310 / 307 | 212 / 195
//   2.8 GB (96 of 6144 x 2560, gate_up)  10: 442 / 450 | 285 / 296   12: 444 / 452 | 301 / 294   20: 448 / 459 | 369 / 330
//   3.5 GB (256 of 7168 x 2048, down)  8: 575 / 581 | 195 / 186   12: 598 / 600 | 221 / 201   16: 617 / 610 | 274 / 236
//   7.0 GB (the same, gate_up)  8: 1071 / 1072 | 362 / 325   12: 1083 / 1085 | 430 / 357
// Below 0.4 GB the two cross between 26 and more than 44 rows.  From 0.5 to 0.56 GB (four shapes) the deep tiles take 1 to 7 %
// longer at 20-28 rows evenly spread, -8 to +16 %, on average 2, with Zipf routing, and win from 28-36 on; the step from there to 20
// lies between the largest launch measured that wants 28 (0.56 GB) and the smallest that wants 20 (0.69).  Given away: up to 4 %
// of an evenly spread gate_up launch of 1.4-1.5 GB at 20-28 rows (where Zipf routing wins 4-12 %), 2 % of one of 2.8 GB at 10-28.
int narrow_rows_per_expert(const moe_i8::GemmArgs& g) {
  const int64_t weight_bytes = (int64_t)g.num_experts * g.n * g.k;
  return weight_bytes < (512ll << 20) ? 40 : weight_bytes < (640ll << 20) ? 28 : weight_bytes < moe_i8::kLongStreamBytes ? 20 : 10;
}

// Which family a launch goes to (MOE_I8_GEMM_STREAM, _TILE or _NARROW); -1 with the error set if a
// family was demanded for a shape it does not handle.
int picks_family(const moe_i8::GemmArgs& g0, int variant) {
  moe_i8::GemmArgs g = g0;
  g.tile_geometry = tile_geometry_of(variant);
  if (variant == MOE_I8_GEMM_TILE || variant == MOE_I8_GEMM_TILE_WIDE || variant == MOE_I8_GEMM_TILE_DEEP ||
      variant == MOE_I8_GEMM_TILE_RING) {
    if (!moe_i8::gemm_tile_supports(g))
      return fail(MOE_I8_EUNSUPPORTED, "tile GEMM does not support this shape"), -1;
    return MOE_I8_GEMM_TILE;
  }
  if (variant == MOE_I8_GEMM_NARROW) {
    if (!moe_i8::gemm_narrow_supports(g))
      return fail(MOE_I8_EUNSUPPORTED, "narrow-tile GEMM does not support this shape"), -1;
    return MOE_I8_GEMM_NARROW;
  }
  if (variant == MOE_I8_GEMM_STREAM) return MOE_I8_GEMM_STREAM;
  // Measured crossovers, in routed rows per expert.  With evenly spread routing the streaming family
  // would win up to about 4 (by 1-2 % over the narrow tiles); with one expert that every token visits,
  // or Zipf-skewed routing, the narrow tiles win by 18-34 % from 24 tokens on.  Then the narrow tiles
  // while most experts hold a single 64-row block, then the LDS-tiled family (which picks its own
  // geometry).
  const int64_t rows_x_experts = g.num_pairs;
  const int64_t most_rows = g.max_rows_per_expert > 0 && g.max_rows_per_expert < g.num_pairs ? g.max_rows_per_expert
                                                                                             : g.num_pairs;
  const bool long_stream = (int64_t)g.num_experts * g.n * g.k >= moe_i8::kLongStreamBytes && moe_i8::gemm_narrow_supports(g);
  if (long_stream ? most_rows <= kStreamMaxRowsLongStream
                  : most_rows <= kStreamMaxRows || rows_x_experts <= (int64_t)kStreamRowsPerExpert * g.num_experts)
    return MOE_I8_GEMM_STREAM;
  if (rows_x_experts <= (int64_t)narrow_rows_per_expert(g) * g.num_experts && moe_i8::gemm_narrow_supports(g))
    return MOE_I8_GEMM_NARROW;
  if (moe_i8::gemm_tile_supports(g)) return MOE_I8_GEMM_TILE;
  return moe_i8::gemm_narrow_supports(g) ? MOE_I8_GEMM_NARROW : MOE_I8_GEMM_STREAM;
}

int run_gemm(const moe_i8::GemmArgs& g0, int variant, hipStream_t stream) {
  if (g0.num_pairs == 0) return MOE_I8_OK;
  moe_i8::GemmArgs g = g0;
  g.tile_geometry = tile_geometry_of(variant);
  switch (picks_family(g, variant)) {
    case MOE_I8_GEMM_TILE: return check_launch(moe_i8::launch_gemm_tile(g, stream), "gemm_tile");
    case MOE_I8_GEMM_NARROW: return check_launch(moe_i8::launch_gemm_narrow(g, stream), "gemm_narrow");
    case MOE_I8_GEMM_STREAM: return check_launch(moe_i8::launch_gemm_stream(g, stream), "gemm_stream");
    default: return MOE_I8_EUNSUPPORTED;
  }
}

moe_i8::GemmArgs gate_up_args(const int8_t* x_q, const float* a_scale, const int8_t* w1, const float* w1_scale,
                              const int32_t* sorted_token_ids, const int32_t* expert_ids,
                              const int32_t* num_tokens_post_padded, int64_t num_pairs, int top_k, int num_experts,
                              int hidden, int inter, int block_size, int64_t sorted_cap, void* act_out) {
  moe_i8::GemmArgs g{};
  g.mode = moe_i8::kGateUpSilu;
  g.a_q = x_q;
  g.a_scale = a_scale;
  g.w = w1;
  g.w_scale = w1_scale;
  g.row_weight = nullptr;
  g.sorted_token_ids = sorted_token_ids;
  g.expert_ids = expert_ids;
  g.num_tokens_post_padded = num_tokens_post_padded;
  g.num_pairs = num_pairs;
  g.row_div = top_k;
  g.num_experts = num_experts;
  g.n = 2 * inter;
  g.k = hidden;
  g.block_size = block_size;
  g.sorted_cap = sorted_cap;
  g.out = act_out;
  g.max_rows_per_expert = (num_pairs + top_k - 1) / top_k;  // an expert sees a token at most once
  return g;
}

// The family of `picks_family` with the geometry of the LDS-tiled family spelled out
// (MOE_I8_GEMM_STREAM, _NARROW, _TILE_WIDE or _TILE_DEEP; _TILE_RING only when demanded); -1 as there.
int picks_kernel(const moe_i8::GemmArgs& g0, int variant) {
  const int family = picks_family(g0, variant);
  if (family != MOE_I8_GEMM_TILE) return family;
  moe_i8::GemmArgs g = g0;
  g.tile_geometry = tile_geometry_of(variant);
  switch (moe_i8::gemm_tile_geometry(g)) {
    case moe_i8::kTileDeep: return MOE_I8_GEMM_TILE_DEEP;
    case moe_i8::kTileRing: return MOE_I8_GEMM_TILE_RING;
    default: return MOE_I8_GEMM_TILE_WIDE;
  }
}

moe_i8::GemmArgs down_args(const int8_t* h_q, const float* a_scale, const int8_t* w2, const float* w2_scale,
                           const float* topk_weights, const int32_t* sorted_token_ids, const int32_t* expert_ids,
                           const int32_t* num_tokens_post_padded, int64_t num_pairs, int num_experts, int hidden,
                           int inter, int block_size, int64_t sorted_cap, void* out) {
  moe_i8::GemmArgs g{};
  g.mode = moe_i8::kDown;
  g.a_q = h_q;
  g.a_scale = a_scale;
  g.w = w2;
  g.w_scale = w2_scale;
  g.row_weight = topk_weights;
  g.sorted_token_ids = sorted_token_ids;
  g.expert_ids = expert_ids;
  g.num_tokens_post_padded = num_tokens_post_padded;
  g.num_pairs = num_pairs;
  g.row_div = 1;
  g.num_experts = num_experts;
  g.n = hidden;
  g.k = inter;
  g.block_size = block_size;
  g.sorted_cap = sorted_cap;
  g.out = out;
  return g;
}

}  // namespace

extern "C" {

int moe_i8_version(void) { return 1; }

const char* moe_i8_last_error(void) { return g_error; }

int64_t moe_i8_sorted_capacity(int64_t num_pairs, int num_experts, int block_size) {
  if (num_pairs < 0 || num_experts < 1 || block_size < 1) return -1;
  const int64_t full = num_pairs + (int64_t)num_experts * (block_size - 1);
  const int64_t tight = num_pairs * block_size;
  return full < tight ? full : tight;
}

int64_t moe_i8_align_workspace_bytes(int64_t num_pairs, int num_experts, int block_size) {
  (void)block_size;
  if (num_pairs < 0 || num_experts < 1) return -1;
  return moe_i8::align_workspace_ints(num_pairs, num_experts) * (int64_t)sizeof(int32_t);
}

int moe_i8_align_block_size(const int32_t* topk_ids, int64_t num_pairs, int num_experts,
                            int block_size, int32_t* sorted_token_ids, int64_t sorted_cap,
                            int32_t* expert_ids, int64_t expert_cap,
                            int32_t* num_tokens_post_padded, void* workspace,
                            int64_t workspace_bytes, void* stream) {
  if (num_pairs < 0 || num_pairs > INT32_MAX - 1) return fail(MOE_I8_EINVAL, "num_pairs out of range");
  if (num_experts < 1 || num_experts > MOE_I8_MAX_EXPERTS)
    return fail(MOE_I8_EINVAL, "num_experts must be in [1, %d]", MOE_I8_MAX_EXPERTS);
  if (!valid_block_size(block_size)) return fail(MOE_I8_EINVAL, "block_size must be 16, 32, 64 or 128");
  if (!num_tokens_post_padded || (num_pairs > 0 && !topk_ids))
    return fail(MOE_I8_EINVAL, "null pointer");
  const int64_t need = moe_i8_sorted_capacity(num_pairs, num_experts, block_size);
  if (sorted_cap < need)
    return fail(MOE_I8_EWORKSPACE, "sorted_token_ids capacity %lld < %lld", (long long)sorted_cap,
                (long long)need);
  if (expert_cap < (sorted_cap + block_size - 1) / block_size)
    return fail(MOE_I8_EWORKSPACE, "expert_ids capacity %lld too small", (long long)expert_cap);
  if ((sorted_cap > 0 && !sorted_token_ids) || (expert_cap > 0 && !expert_ids))
    return fail(MOE_I8_EINVAL, "null pointer");
  const int64_t ws_need = moe_i8_align_workspace_bytes(num_pairs, num_experts, block_size);
  if (ws_need > 0 && (!workspace || workspace_bytes < ws_need))
    return fail(MOE_I8_EWORKSPACE, "align workspace %lld < %lld bytes", (long long)workspace_bytes,
                (long long)ws_need);
  moe_i8::AlignArgs a;
  a.topk_ids = topk_ids;
  a.num_pairs = num_pairs;
  a.num_experts = num_experts;
  a.block_size = block_size;
  a.sorted_token_ids = sorted_token_ids;
  a.sorted_cap = sorted_cap;
  a.expert_ids = expert_ids;
  a.expert_cap = expert_cap;
  a.num_tokens_post_padded = num_tokens_post_padded;
  a.workspace = static_cast<int32_t*>(workspace);
  return check_launch(moe_i8::launch_align(a, static_cast<hipStream_t>(stream)), "moe_align");
}

static int quant_rows_impl(const void* x, int dtype, int64_t src_rows, int64_t cols, int64_t row_stride,
                           const int32_t* gather, int gather_div, int64_t rows, int8_t* q, float* scale,
                           int round_even, void* stream) {
  if (dtype != MOE_I8_DTYPE_BF16) return fail(MOE_I8_EUNSUPPORTED, "only bf16 activations are supported");
  if (rows < 0 || src_rows < 0) return fail(MOE_I8_EINVAL, "negative row count");
  if (rows == 0) return MOE_I8_OK;
  if (!x || !q || !scale) return fail(MOE_I8_EINVAL, "null pointer");
  if (cols < 8 || cols % 8 || cols > INT32_MAX) return fail(MOE_I8_EINVAL, "cols (%lld) must be a positive multiple of 8", (long long)cols);
  if (row_stride < cols || row_stride % 8) return fail(MOE_I8_EINVAL, "row stride must be >= cols and a multiple of 8");
  if (!aligned16(x) || (reinterpret_cast<uintptr_t>(q) & 7u))
    return fail(MOE_I8_EINVAL, "x must be 16-byte and q 8-byte aligned");
  if (gather && gather_div < 1) return fail(MOE_I8_EINVAL, "gather_div must be >= 1");
  if (!gather && rows > src_rows) return fail(MOE_I8_EINVAL, "rows exceeds src_rows");
  moe_i8::QuantArgs a;
  a.x = static_cast<const uint16_t*>(x);
  a.src_rows = src_rows;
  a.cols = (int)cols;
  a.row_stride = row_stride;
  a.gather = gather;
  a.gather_div = gather ? gather_div : 1;
  a.rows = rows;
  a.q = q;
  a.scale = scale;
  a.round_even = round_even;
  return check_launch(moe_i8::launch_quant_rows(a, static_cast<hipStream_t>(stream)), "quant_rows");
}

int moe_i8_quant_rows(const void* x, int dtype, int64_t src_rows, int64_t cols, int64_t row_stride,
                      const int32_t* gather, int gather_div, int64_t rows, int8_t* q, float* scale,
                      void* stream) {
  return quant_rows_impl(x, dtype, src_rows, cols, row_stride, gather, gather_div, rows, q, scale, 0, stream);
}

int moe_i8_scaled_int8_quant(const void* x, int dtype, int64_t rows, int64_t cols, int64_t row_stride,
                             int8_t* q, float* scale, void* stream) {
  return quant_rows_impl(x, dtype, rows, cols, row_stride, nullptr, 1, rows, q, scale, 1, stream);
}

// The router's arguments, checked; nothing is filled in for zero tokens.
static int route_args(const float* logits, int64_t m, int num_experts, int top_k, int score_func,
                      const float* selection_bias, int num_groups, int topk_groups, int group_score_top2,
                      int renormalize, float route_scale, float* topk_weights, int32_t* topk_ids,
                      void* capture, int capture_dtype, int64_t capture_token_stride, int64_t capture_offset, moe_i8::RouteArgs* out) {
  if (m < 0) return fail(MOE_I8_EINVAL, "negative token count");
  if (num_experts < 1 || num_experts > MOE_I8_MAX_EXPERTS)
    return fail(MOE_I8_EINVAL, "num_experts (%d) must be in [1, %d]", num_experts, MOE_I8_MAX_EXPERTS);
  if (top_k < 1 || top_k > num_experts || top_k > 64)
    return fail(MOE_I8_EINVAL, "top_k (%d) must be in [1, min(num_experts, 64)]", top_k);
  if (score_func != MOE_I8_SCORE_SOFTMAX && score_func != MOE_I8_SCORE_SIGMOID &&
      score_func != MOE_I8_SCORE_TOPK_SOFTMAX)
    return fail(MOE_I8_EINVAL, "unknown score function %d", score_func);
  if (num_groups < 1 || num_experts % num_groups) return fail(MOE_I8_EINVAL, "num_groups must divide num_experts");
  if (num_groups > 1) {
    const int per_lane = moe_i8::route_experts_per_lane(num_experts);
    const int group_size = num_experts / num_groups;
    const int lanes = group_size / per_lane;
    if (group_size % per_lane || lanes < 1 || (lanes & (lanes - 1)))
      return fail(MOE_I8_EUNSUPPORTED, "group size %d must be a power-of-two multiple of %d experts", group_size,
                  per_lane);
    if (topk_groups < 1 || topk_groups > num_groups) return fail(MOE_I8_EINVAL, "topk_groups out of range");
    if (group_score_top2 && group_size < 2) return fail(MOE_I8_EINVAL, "top-2 group score needs groups of >= 2");
    if (top_k > topk_groups * group_size) return fail(MOE_I8_EINVAL, "top_k exceeds the experts of the kept groups");
  }
  if (capture_dtype < 0 || capture_dtype > 2) return fail(MOE_I8_EINVAL, "capture dtype must be 0, 1 (u8) or 2 (u16)");
  if (capture_dtype == 1 && num_experts > 256) return fail(MOE_I8_EINVAL, "uint8 capture holds at most 256 experts");
  if (capture_dtype && (!capture || capture_token_stride < top_k || capture_offset < 0 ||
                        capture_offset + top_k > capture_token_stride))
    return fail(MOE_I8_EINVAL, "capture needs a buffer and offset + top_k <= token stride");
  if (m == 0) return MOE_I8_OK;
  if (!logits || !topk_weights || !topk_ids) return fail(MOE_I8_EINVAL, "null pointer");
  moe_i8::RouteArgs& a = *out;
  a.logits = logits;
  a.m = m;
  a.num_experts = num_experts;
  a.top_k = top_k;
  a.score_func = score_func;
  a.bias = selection_bias;
  a.num_groups = num_groups;
  a.topk_groups = topk_groups;
  a.group_top2 = group_score_top2;
  a.renormalize = renormalize;
  a.route_scale = route_scale;
  a.weights = topk_weights;
  a.ids = topk_ids;
  a.capture = capture_dtype ? capture : nullptr;
  a.capture_bytes = capture_dtype;
  a.capture_stride = capture_token_stride;
  a.capture_offset = capture_offset;
  return MOE_I8_OK;
}

int moe_i8_route_topk(const float* logits, int64_t m, int num_experts, int top_k, int score_func,
                      const float* selection_bias, int num_groups, int topk_groups, int group_score_top2,
                      int renormalize, float route_scale, float* topk_weights, int32_t* topk_ids,
                      void* capture, int capture_dtype, int64_t capture_token_stride,
                      int64_t capture_offset, void* stream) {
  moe_i8::RouteArgs a;
  if (int rc = route_args(logits, m, num_experts, top_k, score_func, selection_bias, num_groups, topk_groups, group_score_top2,
                          renormalize, route_scale, topk_weights, topk_ids, capture, capture_dtype, capture_token_stride,
                          capture_offset, &a))
    return rc;
  if (m == 0) return MOE_I8_OK;
  return check_launch(moe_i8::launch_route_topk(a, static_cast<hipStream_t>(stream)), "route_topk");
}

static int weight_quant_args(const void* w, int dtype, int64_t rows, int64_t cols, int64_t rows_per_group,
                             int64_t out_rows_per_group, int64_t out_row_offset, int8_t* q, float* scale,
                             moe_i8::QuantArgs* out) {
  if (dtype != MOE_I8_DTYPE_BF16) return fail(MOE_I8_EUNSUPPORTED, "only bf16 weights are supported");
  if (rows < 0) return fail(MOE_I8_EINVAL, "negative row count");
  if (rows == 0) return MOE_I8_OK;
  if (!w || !q || !scale) return fail(MOE_I8_EINVAL, "null pointer");
  if (cols < 8 || cols % 8 || cols > INT32_MAX)
    return fail(MOE_I8_EINVAL, "cols (%lld) must be a positive multiple of 8", (long long)cols);
  if (!aligned16(w) || (reinterpret_cast<uintptr_t>(q) & 7u))
    return fail(MOE_I8_EINVAL, "w must be 16-byte and q 8-byte aligned");
  if (rows_per_group < 0 || (rows_per_group > 0 && (rows % rows_per_group || out_row_offset < 0 ||
                                                     out_row_offset + rows_per_group > out_rows_per_group)))
    return fail(MOE_I8_EINVAL, "row groups must tile the input and fit inside the output groups");
  moe_i8::QuantArgs a;
  a.x = static_cast<const uint16_t*>(w);
  a.src_rows = rows;
  a.cols = (int)cols;
  a.row_stride = cols;
  a.gather = nullptr;
  a.gather_div = 1;
  a.rows = rows;
  a.q = q;
  a.scale = scale;
  a.rows_per_group = rows_per_group;
  a.out_rows_per_group = out_rows_per_group;
  a.out_row_offset = out_row_offset;
  *out = a;
  return MOE_I8_OK;
}

int moe_i8_quant_weights(const void* w, int dtype, int64_t rows, int64_t cols, int64_t rows_per_group,
                         int64_t out_rows_per_group, int64_t out_row_offset, int8_t* q, float* scale,
                         void* stream) {
  moe_i8::QuantArgs a;
  if (int rc = weight_quant_args(w, dtype, rows, cols, rows_per_group, out_rows_per_group, out_row_offset, q, scale, &a))
    return rc;
  if (rows == 0) return MOE_I8_OK;
  return check_launch(moe_i8::launch_quant_weights(&a, 1, static_cast<hipStream_t>(stream)), "quant_weights");
}

int moe_i8_quant_expert_weights(const void* gate, const void* up, const void* down, int dtype, int64_t num_experts,
                                int64_t inter, int64_t hidden, int8_t* w13, float* w13_scale, int8_t* w2,
                                float* w2_scale, void* stream) {
  if (num_experts < 0 || inter < 1 || hidden < 1) return fail(MOE_I8_EINVAL, "bad layer shape");
  if (num_experts == 0) return MOE_I8_OK;
  moe_i8::QuantArgs a[3];
  if (int rc = weight_quant_args(gate, dtype, num_experts * inter, hidden, inter, 2 * inter, 0, w13, w13_scale, &a[0])) return rc;
  if (int rc = weight_quant_args(up, dtype, num_experts * inter, hidden, inter, 2 * inter, inter, w13, w13_scale, &a[1]))
    return rc;
  if (int rc = weight_quant_args(down, dtype, num_experts * hidden, inter, 0, 0, 0, w2, w2_scale, &a[2])) return rc;
  return check_launch(moe_i8::launch_quant_weights(a, 3, static_cast<hipStream_t>(stream)), "quant_weights");
}

// The gate_up GEMM behind the entry point; `from_align`: the routing arrays are moe_align's own
// output (the caller of the entry point may pass anything).
static int gemm_gate_up_impl(const int8_t* x_q, const float* a_scale, const int8_t* w1, const float* w1_scale,
                             const int32_t* sorted_token_ids, const int32_t* expert_ids,
                             const int32_t* num_tokens_post_padded, int64_t num_pairs, int top_k, int num_experts,
                             int hidden, int inter, int block_size, int64_t sorted_cap, void* act_out, int variant,
                             bool from_align, void* stream) {
  if (num_pairs == 0) return MOE_I8_OK;
  if (inter < 16 || inter % 16 || inter > (1 << 29)) return fail(MOE_I8_EINVAL, "inter (%d) must be a positive multiple of 16", inter);
  if (int rc = check_gemm_common(x_q, w1, sorted_token_ids, expert_ids, num_tokens_post_padded,
                                 act_out, num_pairs, num_experts, 2 * inter, hidden, block_size,
                                 sorted_cap, variant))
    return rc;
  if (!a_scale || !w1_scale) return fail(MOE_I8_EINVAL, "null scale pointer");
  if (!aligned16(w1_scale)) return fail(MOE_I8_EINVAL, "w1_scale must be 16-byte aligned");
  if (top_k < 1) return fail(MOE_I8_EINVAL, "top_k must be >= 1");
  moe_i8::GemmArgs g = gate_up_args(x_q, a_scale, w1, w1_scale, sorted_token_ids, expert_ids, num_tokens_post_padded,
                                    num_pairs, top_k, num_experts, hidden, inter, block_size, sorted_cap, act_out);
  g.expert_ids_ascend = from_align;
  return run_gemm(g, variant, static_cast<hipStream_t>(stream));
}

int moe_i8_gemm_gate_up_silu(const int8_t* x_q, const float* a_scale, const int8_t* w1,
                             const float* w1_scale, const int32_t* sorted_token_ids,
                             const int32_t* expert_ids, const int32_t* num_tokens_post_padded,
                             int64_t num_pairs, int top_k, int num_experts, int hidden, int inter,
                             int block_size, int64_t sorted_cap, void* act_out, int variant,
                             void* stream) {
  return gemm_gate_up_impl(x_q, a_scale, w1, w1_scale, sorted_token_ids, expert_ids, num_tokens_post_padded, num_pairs,
                           top_k, num_experts, hidden, inter, block_size, sorted_cap, act_out, variant, false, stream);
}

// The down GEMM behind the entry point; `max_rows` bounds the rows any one expert can hold (0: unknown),
// `from_align` as above.
static int gemm_down_impl(const int8_t* h_q, const float* a_scale, const int8_t* w2, const float* w2_scale,
                          const float* topk_weights, const int32_t* sorted_token_ids, const int32_t* expert_ids,
                          const int32_t* num_tokens_post_padded, int64_t num_pairs, int num_experts, int hidden,
                          int inter, int block_size, int64_t sorted_cap, void* out, int variant, int64_t max_rows,
                          bool from_align, void* stream) {
  if (num_pairs == 0) return MOE_I8_OK;
  if (int rc = check_gemm_common(h_q, w2, sorted_token_ids, expert_ids, num_tokens_post_padded, out,
                                 num_pairs, num_experts, hidden, inter, block_size, sorted_cap,
                                 variant))
    return rc;
  if (!a_scale || !w2_scale) return fail(MOE_I8_EINVAL, "null scale pointer");
  if (!aligned16(w2_scale)) return fail(MOE_I8_EINVAL, "w2_scale must be 16-byte aligned");
  moe_i8::GemmArgs g = down_args(h_q, a_scale, w2, w2_scale, topk_weights, sorted_token_ids, expert_ids,
                                 num_tokens_post_padded, num_pairs, num_experts, hidden, inter, block_size,
                                 sorted_cap, out);
  g.max_rows_per_expert = max_rows;
  g.expert_ids_ascend = from_align;
  return run_gemm(g, variant, static_cast<hipStream_t>(stream));
}

int moe_i8_gemm_down(const int8_t* h_q, const float* a_scale, const int8_t* w2,
                     const float* w2_scale, const float* topk_weights,
                     const int32_t* sorted_token_ids, const int32_t* expert_ids,
                     const int32_t* num_tokens_post_padded, int64_t num_pairs, int num_experts,
                     int hidden, int inter, int block_size, int64_t sorted_cap, void* out,
                     int variant, void* stream) {
  return gemm_down_impl(h_q, a_scale, w2, w2_scale, topk_weights, sorted_token_ids, expert_ids,
                        num_tokens_post_padded, num_pairs, num_experts, hidden, inter, block_size, sorted_cap, out,
                        variant, 0, false, stream);
}

// The self-quantising down GEMM behind the entry point; `max_rows` as in gemm_down_impl.
static int gemm_down_bf16_impl(const void* act, const int8_t* w2, const float* w2_scale, const float* topk_weights,
                               const int32_t* sorted_token_ids, const int32_t* expert_ids,
                               const int32_t* num_tokens_post_padded, int64_t num_pairs, int num_experts, int hidden,
                               int inter, int block_size, int64_t sorted_cap, void* out, int64_t max_rows, void* stream) {
  if (num_pairs == 0) return MOE_I8_OK;
  if (int rc = check_gemm_common(act, w2, sorted_token_ids, expert_ids, num_tokens_post_padded, out, num_pairs,
                                 num_experts, hidden, inter, block_size, sorted_cap, MOE_I8_GEMM_STREAM))
    return rc;
  if (!w2_scale) return fail(MOE_I8_EINVAL, "null scale pointer");
  if (!aligned16(w2_scale)) return fail(MOE_I8_EINVAL, "w2_scale must be 16-byte aligned");
  moe_i8::GemmArgs g = down_args(nullptr, nullptr, w2, w2_scale, topk_weights, sorted_token_ids, expert_ids,
                                 num_tokens_post_padded, num_pairs, num_experts, hidden, inter, block_size,
                                 sorted_cap, out);
  g.a_bf16 = static_cast<const uint16_t*>(act);
  g.max_rows_per_expert = max_rows;
  return check_launch(moe_i8::launch_gemm_stream(g, static_cast<hipStream_t>(stream)), "gemm_stream");
}

int moe_i8_gemm_down_bf16(const void* act, const int8_t* w2, const float* w2_scale, const float* topk_weights,
                          const int32_t* sorted_token_ids, const int32_t* expert_ids,
                          const int32_t* num_tokens_post_padded, int64_t num_pairs, int num_experts, int hidden,
                          int inter, int block_size, int64_t sorted_cap, void* out, void* stream) {
  if (num_pairs > 0 && inter > kSelfQuantMaxInter)
    return fail(MOE_I8_EUNSUPPORTED, "inter (%d) is too long for the GEMM that quantises its own activations", inter);
  return gemm_down_bf16_impl(act, w2, w2_scale, topk_weights, sorted_token_ids, expert_ids, num_tokens_post_padded, num_pairs,
                             num_experts, hidden, inter, block_size, sorted_cap, out, 0, stream);
}

int moe_i8_gemm_acc_i32(const int8_t* a_q, const int8_t* w, const int32_t* sorted_token_ids,
                        const int32_t* expert_ids, const int32_t* num_tokens_post_padded,
                        int64_t num_pairs, int row_div, int num_experts, int n, int k,
                        int block_size, int64_t sorted_cap, int32_t* acc_out, int variant,
                        void* stream) {
  if (num_pairs == 0) return MOE_I8_OK;
  if (int rc = check_gemm_common(a_q, w, sorted_token_ids, expert_ids, num_tokens_post_padded,
                                 acc_out, num_pairs, num_experts, n, k, block_size, sorted_cap,
                                 variant))
    return rc;
  if (row_div < 1) return fail(MOE_I8_EINVAL, "row_div must be >= 1");
  moe_i8::GemmArgs g{};
  g.mode = moe_i8::kAccI32;
  g.a_q = a_q;
  g.w = w;
  g.sorted_token_ids = sorted_token_ids;
  g.expert_ids = expert_ids;
  g.num_tokens_post_padded = num_tokens_post_padded;
  g.num_pairs = num_pairs;
  g.row_div = row_div;
  g.num_experts = num_experts;
  g.n = n;
  g.k = k;
  g.block_size = block_size;
  g.sorted_cap = sorted_cap;
  g.out = acc_out;
  return run_gemm(g, variant, static_cast<hipStream_t>(stream));
}

int moe_i8_sum(const void* in, void* out, int64_t m, int top_k, int hidden, void* stream) {
  if (m < 0) return fail(MOE_I8_EINVAL, "negative m");
  if (m == 0) return MOE_I8_OK;
  if (!in || !out) return fail(MOE_I8_EINVAL, "null pointer");
  if (top_k < 1) return fail(MOE_I8_EINVAL, "top_k must be >= 1");
  if (hidden < 8 || hidden % 8) return fail(MOE_I8_EINVAL, "hidden (%d) must be a positive multiple of 8", hidden);
  if (!aligned16(in) || !aligned16(out)) return fail(MOE_I8_EINVAL, "pointers must be 16-byte aligned");
  return check_launch(moe_i8::launch_moe_sum(static_cast<const uint16_t*>(in), static_cast<uint16_t*>(out),
                                             m, top_k, hidden, static_cast<hipStream_t>(stream)),
                      "moe_sum");
}

// Workspace layout of moe_i8_fused_experts (every region 256-byte aligned):
//   x_q i8[M*H] | a1_scale f32[M] | sorted i32[cap] | expert_ids i32[cap/B] | npp i32[1] |
//   align scratch | act bf16[P*I] | act_q i8[P*I] | a2_scale f32[P] | down_out bf16[P*H]
namespace {
struct Carve {
  int64_t x_q, a1, sorted, eids, npp, align_ws, act, act_q, a2, down, total;
  int64_t cap, ecap, align_bytes;
};
Carve carve(int64_t m, int top_k, int num_experts, int hidden, int inter, int block_size) {
  Carve c{};
  const int64_t p = m * top_k;
  c.cap = moe_i8_sorted_capacity(p, num_experts, block_size);
  c.ecap = (c.cap + block_size - 1) / block_size;
  c.align_bytes = moe_i8_align_workspace_bytes(p, num_experts, block_size);
  int64_t off = 0;
  auto take = [&](int64_t bytes) {
    const int64_t at = off;
    off = align_up(off + bytes, 256);
    return at;
  };
  c.x_q = take(m * hidden);
  c.a1 = take(m * 4);
  c.sorted = take(c.cap * 4);
  c.eids = take(c.ecap * 4);
  c.npp = take(4);
  c.align_ws = take(c.align_bytes);
  c.act = take(p * inter * 2);
  c.act_q = take(p * inter);
  c.a2 = take(p * 4);
  c.down = take(p * hidden * 2);
  c.total = off;
  return c;
}

// What moe_i8_fused_experts launches for a layer shape: decided on the host from the sizes alone.
struct LayerPlan {
  int gate_up_kernel;   // MOE_I8_GEMM_STREAM, _NARROW, _TILE_WIDE or _TILE_DEEP; -1 = shape not supported by the demanded family
  int down_kernel;
  bool fuse_align_quant;  // moe_align and the quantisation of the layer input in one launch
  bool down_quantises;    // the streaming down GEMM quantises its own bf16 activations (one launch less)
  int launches;
};

LayerPlan plan_layer(int64_t m, int top_k, int num_experts, int hidden, int inter, int block_size, int variant) {
  const Carve c = carve(m, top_k, num_experts, hidden, inter, block_size);
  const int64_t p = m * top_k;
  LayerPlan plan{};
  moe_i8::GemmArgs gu = gate_up_args(nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, p, top_k, num_experts,
                                     hidden, inter, block_size, c.cap, nullptr);
  gu.expert_ids_ascend = true;
  plan.gate_up_kernel = picks_kernel(gu, variant);
  moe_i8::GemmArgs dg = down_args(nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, p, num_experts,
                                  hidden, inter, block_size, c.cap, nullptr);
  dg.expert_ids_ascend = true;
  dg.max_rows_per_expert = m;
  plan.down_kernel = picks_kernel(dg, variant);
  // Very few rows per expert (decode): the streaming down GEMM quantises its activations itself, one
  // launch less.  Every workgroup of a block repeats that quantisation, so from about four rows
  // per expert on (measured) the separate launch is the cheaper one again.
  plan.down_quantises = plan.down_kernel == MOE_I8_GEMM_STREAM && moe_i8::gemm_stream_fuses_quant(dg) &&
                        p <= (int64_t)3 * num_experts;
  moe_i8::AlignArgs aa{};
  aa.num_pairs = p;
  aa.num_experts = num_experts;
  aa.block_size = block_size;
  aa.sorted_cap = c.cap;
  aa.expert_cap = c.ecap;
  moe_i8::QuantArgs qa{};
  qa.src_rows = m;
  qa.cols = hidden;
  qa.row_stride = hidden;
  qa.gather_div = 1;
  qa.rows = m;
  plan.fuse_align_quant = moe_i8::align_quant_fusable(aa, qa);
  plan.launches = moe_i8::align_launches(aa) + (plan.fuse_align_quant ? 0 : 1) + 1 + (plan.down_quantises ? 1 : 2) + 1;
  return plan;
}

// A few tokens: no rows to gather per expert, the whole layer in two launches instead of that chain.
bool runs_few_tokens(int64_t m, int top_k, int num_experts, int hidden, int inter, int variant) {
  return variant == MOE_I8_GEMM_AUTO && moe_i8::few_tokens_takes(m, top_k, num_experts, hidden, inter);
}
}  // namespace

int64_t moe_i8_workspace_bytes(int64_t m, int top_k, int num_experts, int hidden, int inter,
                               int block_size) {
  if (m < 0 || top_k < 1 || num_experts < 1 || hidden < 1 || inter < 1 || !valid_block_size(block_size))
    return -1;
  return carve(m, top_k, num_experts, hidden, inter, block_size).total;
}

// `route`: the routing is still to be done (topk_weights and topk_ids are written first).
static int fused_experts_impl(const void* hidden, const int8_t* w1, const int8_t* w2,
                         const float* topk_weights, const int32_t* topk_ids,
                         const float* w1_scale, const float* w2_scale, void* out, int64_t m,
                         int top_k, int num_experts, int hidden_size, int inter, int block_size,
                         void* workspace, int64_t workspace_bytes, int variant,
                         const moe_i8::RouteArgs* route, void* stream) {
  if (m < 0) return fail(MOE_I8_EINVAL, "negative m");
  if (m == 0) return MOE_I8_OK;
  if (!hidden || !w1 || !w2 || !topk_weights || !topk_ids || !w1_scale || !w2_scale || !out || !workspace)
    return fail(MOE_I8_EINVAL, "null pointer");
  if (top_k < 1 || m * top_k > INT32_MAX - 1) return fail(MOE_I8_EINVAL, "top_k / num_pairs out of range");
  if (!valid_block_size(block_size)) return fail(MOE_I8_EINVAL, "block_size must be 16, 32, 64 or 128");
  if (hidden_size < 64 || hidden_size % 64 || inter < 64 || inter % 64)
    return fail(MOE_I8_EINVAL, "hidden (%d) and inter (%d) must be positive multiples of 64", hidden_size, inter);
  if (num_experts < 1 || num_experts > MOE_I8_MAX_EXPERTS)
    return fail(MOE_I8_EINVAL, "num_experts must be in [1, %d]", MOE_I8_MAX_EXPERTS);
  if (!aligned16(hidden) || !aligned16(w1) || !aligned16(w2) || !aligned16(out))
    return fail(MOE_I8_EINVAL, "activation, weight and output pointers must be 16-byte aligned");
  if (!aligned16(w1_scale) || !aligned16(w2_scale)) return fail(MOE_I8_EINVAL, "weight scales must be 16-byte aligned");
  if (reinterpret_cast<uintptr_t>(workspace) & 255u) return fail(MOE_I8_EINVAL, "workspace must be 256-byte aligned");
  const Carve c = carve(m, top_k, num_experts, hidden_size, inter, block_size);
  if (workspace_bytes < c.total)
    return fail(MOE_I8_EWORKSPACE, "workspace %lld < %lld bytes", (long long)workspace_bytes, (long long)c.total);
  char* ws = static_cast<char*>(workspace);
  int8_t* x_q = reinterpret_cast<int8_t*>(ws + c.x_q);
  float* a1 = reinterpret_cast<float*>(ws + c.a1);
  int32_t* sorted = reinterpret_cast<int32_t*>(ws + c.sorted);
  int32_t* eids = reinterpret_cast<int32_t*>(ws + c.eids);
  int32_t* npp = reinterpret_cast<int32_t*>(ws + c.npp);
  void* act = ws + c.act;
  int8_t* act_q = reinterpret_cast<int8_t*>(ws + c.act_q);
  float* a2 = reinterpret_cast<float*>(ws + c.a2);
  void* down = ws + c.down;
  const int64_t p = m * top_k;
  const WorkspaceTurn turn(workspace);

  if (runs_few_tokens(m, top_k, num_experts, hidden_size, inter, variant)) {
    moe_i8::FewTokensArgs f;
    f.x = static_cast<const uint16_t*>(hidden);
    f.w1 = w1;
    f.w1_scale = w1_scale;
    f.w2 = w2;
    f.w2_scale = w2_scale;
    f.topk_weights = topk_weights;
    f.topk_ids = topk_ids;
    f.act = static_cast<uint16_t*>(act);
    f.out = static_cast<uint16_t*>(out);
    f.tokens = (int)m;
    f.top_k = top_k;
    f.num_experts = num_experts;
    f.hidden = hidden_size;
    f.inter = inter;
    const bool routes = route && moe_i8::few_tokens_routes(m, num_experts);
    if (route && !routes)
      if (int rc = check_launch(moe_i8::launch_route_topk(*route, static_cast<hipStream_t>(stream)), "route_topk")) return rc;
    return check_launch(moe_i8::launch_few_tokens(f, routes ? route : nullptr, static_cast<hipStream_t>(stream)), "few_tokens");
  }

  const LayerPlan plan = plan_layer(m, top_k, num_experts, hidden_size, inter, block_size, variant);
  if (plan.gate_up_kernel < 0 || plan.down_kernel < 0) return MOE_I8_EUNSUPPORTED;
  if (route)
    if (int rc = check_launch(moe_i8::launch_route_topk(*route, static_cast<hipStream_t>(stream)), "route_topk")) return rc;

  // Small batches: moe_align (one workgroup) and the quantisation of the input share one launch.
  moe_i8::AlignArgs aa;
  aa.topk_ids = topk_ids;
  aa.num_pairs = p;
  aa.num_experts = num_experts;
  aa.block_size = block_size;
  aa.sorted_token_ids = sorted;
  aa.sorted_cap = c.cap;
  aa.expert_ids = eids;
  aa.expert_cap = c.ecap;
  aa.num_tokens_post_padded = npp;
  aa.workspace = reinterpret_cast<int32_t*>(ws + c.align_ws);
  moe_i8::QuantArgs qa;
  qa.x = static_cast<const uint16_t*>(hidden);
  qa.src_rows = m;
  qa.cols = hidden_size;
  qa.row_stride = hidden_size;
  qa.gather = nullptr;
  qa.gather_div = 1;
  qa.rows = m;
  qa.q = x_q;
  qa.scale = a1;
  if (moe_i8::align_quant_fusable(aa, qa)) {
    if (int rc = check_launch(moe_i8::launch_align_quant(aa, qa, static_cast<hipStream_t>(stream)),
                              "align_quant"))
      return rc;
  } else {
    if (int rc = moe_i8_quant_rows(hidden, MOE_I8_DTYPE_BF16, m, hidden_size, hidden_size, nullptr, 1, m,
                                   x_q, a1, stream))
      return rc;
    if (int rc = moe_i8_align_block_size(topk_ids, p, num_experts, block_size, sorted, c.cap, eids, c.ecap,
                                         npp, ws + c.align_ws, c.align_bytes, stream))
      return rc;
  }
  if (int rc = gemm_gate_up_impl(x_q, a1, w1, w1_scale, sorted, eids, npp, p, top_k, num_experts, hidden_size, inter,
                                 block_size, c.cap, act, variant, true, stream))
    return rc;
  if (plan.down_quantises) {
    if (int rc = gemm_down_bf16_impl(act, w2, w2_scale, topk_weights, sorted, eids, npp, p, num_experts,
                                     hidden_size, inter, block_size, c.cap, down, m, stream))
      return rc;
  } else {
    if (int rc = moe_i8_quant_rows(act, MOE_I8_DTYPE_BF16, p, inter, inter, nullptr, 1, p, act_q, a2, stream))
      return rc;
    if (int rc = gemm_down_impl(act_q, a2, w2, w2_scale, topk_weights, sorted, eids, npp, p, num_experts,
                                hidden_size, inter, block_size, c.cap, down, variant, m, true, stream))
      return rc;
  }
  return moe_i8_sum(down, out, m, top_k, hidden_size, stream);
}

int moe_i8_fused_experts(const void* hidden, const int8_t* w1, const int8_t* w2,
                         const float* topk_weights, const int32_t* topk_ids,
                         const float* w1_scale, const float* w2_scale, void* out, int64_t m,
                         int top_k, int num_experts, int hidden_size, int inter, int block_size,
                         void* workspace, int64_t workspace_bytes, int variant, void* stream) {
  return fused_experts_impl(hidden, w1, w2, topk_weights, topk_ids, w1_scale, w2_scale, out, m, top_k, num_experts, hidden_size,
                            inter, block_size, workspace, workspace_bytes, variant, nullptr, stream);
}

int moe_i8_fused_moe(const void* hidden, const float* logits, const int8_t* w1, const int8_t* w2, const float* w1_scale,
                     const float* w2_scale, void* out, int64_t m, int top_k, int num_experts, int hidden_size, int inter,
                     int block_size, int score_func, const float* selection_bias, int num_groups, int topk_groups,
                     int group_score_top2, int renormalize, float route_scale, float* topk_weights, int32_t* topk_ids,
                     void* capture, int capture_dtype, int64_t capture_token_stride, int64_t capture_offset,
                     void* workspace, int64_t workspace_bytes, int variant, void* stream) {
  moe_i8::RouteArgs route;
  if (int rc = route_args(logits, m, num_experts, top_k, score_func, selection_bias, num_groups, topk_groups, group_score_top2,
                          renormalize, route_scale, topk_weights, topk_ids, capture, capture_dtype, capture_token_stride,
                          capture_offset, &route))
    return rc;
  return fused_experts_impl(hidden, w1, w2, topk_weights, topk_ids, w1_scale, w2_scale, out, m, top_k, num_experts, hidden_size,
                            inter, block_size, workspace, workspace_bytes, variant, &route, stream);
}

static int layer_shape_args(int64_t m, int top_k, int num_experts, int hidden_size, int inter, int block_size, int variant) {
  if (m < 1 || top_k < 1 || m * top_k > INT32_MAX - 1) return fail(MOE_I8_EINVAL, "m / top_k out of range");
  if (num_experts < 1 || num_experts > MOE_I8_MAX_EXPERTS)
    return fail(MOE_I8_EINVAL, "num_experts must be in [1, %d]", MOE_I8_MAX_EXPERTS);
  if (!valid_block_size(block_size)) return fail(MOE_I8_EINVAL, "block_size must be 16, 32, 64 or 128");
  if (hidden_size < 64 || hidden_size % 64 || inter < 64 || inter % 64)
    return fail(MOE_I8_EINVAL, "hidden (%d) and inter (%d) must be positive multiples of 64", hidden_size, inter);
  if (variant < MOE_I8_GEMM_AUTO || variant > MOE_I8_GEMM_TILE_RING)
    return fail(MOE_I8_EINVAL, "unknown GEMM variant %d", variant);
  return MOE_I8_OK;
}

int moe_i8_layer_plan(int64_t m, int top_k, int num_experts, int hidden_size, int inter, int block_size,
                      int variant, int* gate_up_kernel, int* down_kernel, int* launches) {
  if (int rc = layer_shape_args(m, top_k, num_experts, hidden_size, inter, block_size, variant)) return rc;
  const LayerPlan plan = plan_layer(m, top_k, num_experts, hidden_size, inter, block_size, variant);
  if (plan.gate_up_kernel < 0 || plan.down_kernel < 0) return MOE_I8_EUNSUPPORTED;
  if (gate_up_kernel) *gate_up_kernel = plan.gate_up_kernel;
  if (down_kernel) *down_kernel = plan.down_kernel;
  if (launches) *launches = plan.launches;
  return MOE_I8_OK;
}

int moe_i8_layer_launches(int64_t m, int top_k, int num_experts, int hidden_size, int inter, int block_size, int variant,
                          int routed, int* launches) {
  if (int rc = layer_shape_args(m, top_k, num_experts, hidden_size, inter, block_size, variant)) return rc;
  if (!launches) return fail(MOE_I8_EINVAL, "null pointer");
  if (runs_few_tokens(m, top_k, num_experts, hidden_size, inter, variant)) {
    *launches = routed && !moe_i8::few_tokens_routes(m, num_experts) ? 3 : 2;
    return MOE_I8_OK;
  }
  const LayerPlan plan = plan_layer(m, top_k, num_experts, hidden_size, inter, block_size, variant);
  if (plan.gate_up_kernel < 0 || plan.down_kernel < 0) return MOE_I8_EUNSUPPORTED;
  *launches = plan.launches + (routed ? 1 : 0);
  return MOE_I8_OK;
}

// ---- the entry point that allocates nothing ----
// The workspace of the layer lives in a file-scope device array instead of caller memory.  The
// array's name is only a host-side handle: the device address is asked from the runtime once per
// device (each device holds its own copy at its own address) and that pointer is what the launches get.
namespace {
static __device__ __attribute__((used)) __align__(256) unsigned char scratch[MOE_I8_STATIC_SCRATCH_BYTES];
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mutex;
void* g_scratch_ptr[kMaxDevices] = {};

int static_scratch(void** out) {
  int dev = -1;
  const hipError_t derr = hipGetDevice(&dev);
  if (derr != hipSuccess) return fail(MOE_I8_ELAUNCH, "hipGetDevice: %s", hipGetErrorString(derr));
  if (dev < 0 || dev >= kMaxDevices) return fail(MOE_I8_EUNSUPPORTED, "device index %d outside [0, %d)", dev, kMaxDevices);
  std::lock_guard<std::mutex> lock(g_scratch_mutex);
  if (!g_scratch_ptr[dev]) {
    void* p = nullptr;
    const hipError_t err = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (err != hipSuccess || !p)
      return fail(MOE_I8_ELAUNCH, "hipGetSymbolAddress(scratch) on device %d: %s", dev, hipGetErrorString(err));
    g_scratch_ptr[dev] = p;
  }
  *out = g_scratch_ptr[dev];
  return MOE_I8_OK;
}
}  // namespace

int moe_i8_fused_experts_static(const void* hidden, const int8_t* w1, const int8_t* w2,
                                const float* topk_weights, const int32_t* topk_ids,
                                const float* w1_scale, const float* w2_scale, void* out, int64_t m,
                                int top_k, int num_experts, int hidden_size, int inter, int block_size,
                                int variant, void* stream) {
  if (m < 0) return fail(MOE_I8_EINVAL, "negative m");
  if (m == 0) return MOE_I8_OK;
  const int64_t need = moe_i8_workspace_bytes(m, top_k, num_experts, hidden_size, inter, block_size);
  if (need < 0) return fail(MOE_I8_EINVAL, "bad layer shape");
  if (need > (int64_t)MOE_I8_STATIC_SCRATCH_BYTES)
    return fail(MOE_I8_EWORKSPACE,
                "this call needs %lld bytes of scratch, the static array holds %lld: use moe_i8_fused_experts "
                "with a caller-owned workspace",
                (long long)need, (long long)MOE_I8_STATIC_SCRATCH_BYTES);
  void* ws = nullptr;
  if (int rc = static_scratch(&ws)) return rc;
  // every region of the workspace is written by the call before it is read: nothing to clear
  return moe_i8_fused_experts(hidden, w1, w2, topk_weights, topk_ids, w1_scale, w2_scale, out, m, top_k,
                              num_experts, hidden_size, inter, block_size, ws, MOE_I8_STATIC_SCRATCH_BYTES, variant,
                              stream);
}

// Workspace of the dense entry points (every region 256-byte aligned; int8 rows are padded to a multiple
// of 128 bytes):
//   x_q i8[M*K] | a1 f32[M] | sorted i32[cap] | expert_ids i32[cap/64] | npp i32[1] |
//   (mlp only) act bf16[M*I] | act_q i8[M*I] | a2 f32[M]
namespace {
constexpr int kDenseBlock = 64;
constexpr int kDenseSelfQuantRows = 16;  // up to this many rows the down GEMM of the MLP quantises its own input
struct DenseCarve {
  int64_t x_q, a1, sorted, eids, npp, act, act_q, a2, total, cap;
};
DenseCarve dense_carve(int64_t m, int k, int inter) {
  DenseCarve c{};
  c.cap = moe_i8_sorted_capacity(m, 1, kDenseBlock);
  int64_t off = 0;
  auto take = [&](int64_t bytes) {
    const int64_t at = off;
    off = align_up(off + bytes, 256);
    return at;
  };
  c.x_q = take(m * moe_i8::dense_row_stride(k));
  c.a1 = take(m * 4);
  c.sorted = take(c.cap * 4);
  c.eids = take((c.cap + kDenseBlock - 1) / kDenseBlock * 4);
  c.npp = take(4);
  if (inter > 0) {
    c.act = take(m * inter * 2);
    c.act_q = take(m * moe_i8::dense_row_stride(inter));
    c.a2 = take(m * 4);
  }
  c.total = off;
  return c;
}

// A dense problem as the grouped families see it: one expert that every row visits.
moe_i8::GemmArgs dense_group(int mode, const DenseCarve& c, char* ws, const int8_t* a_q, const float* a_scale,
                             const int8_t* w, const float* w_scale, void* out, int64_t m, int n, int k) {
  const int32_t* sorted = reinterpret_cast<int32_t*>(ws + c.sorted);
  const int32_t* eids = reinterpret_cast<int32_t*>(ws + c.eids);
  const int32_t* npp = reinterpret_cast<int32_t*>(ws + c.npp);
  moe_i8::GemmArgs g = mode == moe_i8::kGateUpSilu
                           ? gate_up_args(a_q, a_scale, w, w_scale, sorted, eids, npp, m, 1, 1, k, n / 2, kDenseBlock, c.cap, out)
                           : down_args(a_q, a_scale, w, w_scale, nullptr, sorted, eids, npp, m, 1, n, k, kDenseBlock, c.cap, out);
  g.expert_ids_ascend = true;  // one expert
  g.identity = true;
  return g;
}

int check_dense_gemm(const moe_i8::GemmArgs& g, int variant) {
  if (int rc = check_gemm_common(g.a_q, g.w, g.sorted_token_ids, g.expert_ids, g.num_tokens_post_padded, g.out, g.num_pairs,
                                 1, g.n, g.k, g.block_size, g.sorted_cap, variant))
    return rc;
  return aligned16(g.w_scale) ? MOE_I8_OK : fail(MOE_I8_EINVAL, "weight scales must be 16-byte aligned");
}

bool overlap(const void* a, int64_t a_bytes, const void* b, int64_t b_bytes) {
  const uintptr_t a0 = reinterpret_cast<uintptr_t>(a), b0 = reinterpret_cast<uintptr_t>(b);
  return a0 < b0 + (uintptr_t)b_bytes && b0 < a0 + (uintptr_t)a_bytes;
}

// How a GEMM of a dense entry point runs, decided once per GEMM.
enum DenseWay {
  kGrouped,  // quantised by a launch of its own, then the 256-row tiles or a demanded family, which read that launch's routing
  kDense,    // quantised by a launch of its own, then the dense kernel, which needs no routing
  kRows,     // the product's own launch quantises the rows, mostly tens to hundreds of them
  kFew,      // ... a few rows
};
struct DenseChoice {
  DenseWay way;
  int entry;  // tile of the dense kernel or of the one that quantises its rows
};
// `own`: the product's launch may quantise the rows.
DenseChoice dense_choice(moe_i8::GemmArgs g, int variant, bool own) {
  if (variant != MOE_I8_GEMM_AUTO) return {kGrouped, -1};
  const bool few = own && moe_i8::dense_few_takes(g.num_pairs, g.n, g.k);
  if (few && g.num_pairs < moe_i8::kDenseRowsFrom) return {kFew, -1};
  moe_i8::DensePick quantised{-1, 0.0f};
  if (!few) {
    g.tile_geometry = moe_i8::kTileWide;
    quantised = moe_i8::gemm_dense_pick(g.mode, g.num_pairs, g.n, g.k, moe_i8::gemm_tile_supports(g));
  }
  if (own) {
    const int entry = moe_i8::dense_rows_pick(g.num_pairs, g.n, g.k, few, quantised.us);
    if (entry >= 0) return {kRows, entry};
    if (few) return {kFew, -1};
  }
  return {quantised.entry < 0 ? kGrouped : kDense, quantised.entry};
}
// Whether the product's launch may quantise the rows at `x`: not where the output overlaps them, as every workgroup reads rows that
// others need while some already write.  (The other kernels read a copy that a launch of its own has quantised.)
bool may_quantise(const void* x, const moe_i8::GemmArgs& g) {
  const int64_t width = g.mode == moe_i8::kGateUpSilu ? g.n / 2 : g.n;
  return aligned16(x) && aligned16(g.w) && !overlap(x, 2 * g.num_pairs * g.k, g.out, 2 * g.num_pairs * width);
}

struct MlpChoice {
  DenseChoice gate_up, down;
};
// Where a grouped family runs the down GEMM the first quantisation has a launch of its own, which also writes that family's routing.
MlpChoice mlp_choice(const moe_i8::GemmArgs& gu, const moe_i8::GemmArgs& dg, int variant, bool own_gu, bool own_dg) {
  const DenseChoice down = dense_choice(dg, variant, own_dg);
  return {dense_choice(gu, variant, own_gu && down.way != kGrouped), down};
}

// The 256-row tiles of the LDS-tiled family for what the dense kernel leaves to the grouped families, where they can run it.
int grouped_variant(moe_i8::GemmArgs g, int variant) {
  g.tile_geometry = moe_i8::kTileWide;
  return variant == MOE_I8_GEMM_AUTO && moe_i8::gemm_tile_supports(g) ? MOE_I8_GEMM_TILE_WIDE : variant;
}

// The product of a quantised problem.
int run_quantised(const DenseChoice& choice, const moe_i8::GemmArgs& g, int variant, hipStream_t stream) {
  if (int rc = check_dense_gemm(g, variant)) return rc;
  if (choice.way == kDense) {
    const moe_i8::DenseArgs d{g.mode, g.a_q, g.a_scale, g.w, g.w_scale, g.out, g.num_pairs, g.n, g.k};
    return check_launch(moe_i8::launch_gemm_dense(d, choice.entry, stream), "gemm_dense");
  }
  return run_gemm(g, grouped_variant(g, variant), stream);
}
// A problem whose rows the product's launch quantises.
int run_unquantised(const DenseChoice& choice, const void* x, const moe_i8::GemmArgs& g, hipStream_t stream) {
  if (int rc = check_dense_gemm(g, MOE_I8_GEMM_AUTO)) return rc;
  const moe_i8::DenseFewArgs d{g.mode, static_cast<const uint16_t*>(x), g.w, g.w_scale, static_cast<uint16_t*>(g.out), (int)g.num_pairs, g.n, g.k};
  return choice.way == kFew ? check_launch(moe_i8::launch_dense_few(d, stream), "dense_few")
                            : check_launch(moe_i8::launch_dense_rows(d, choice.entry, stream), "dense_rows");
}

int dense_shape_args(int64_t m, int n, int k, int variant) {
  if (m < 1 || m > INT32_MAX - kDenseBlock) return fail(MOE_I8_EINVAL, "m out of range");
  if (n < 16 || n % 16) return fail(MOE_I8_EINVAL, "output channels (%d) must be a positive multiple of 16", n);
  if (k < 64 || k % 64) return fail(MOE_I8_EINVAL, "reduction length (%d) must be a positive multiple of 64", k);
  if (variant < MOE_I8_GEMM_AUTO || variant > MOE_I8_GEMM_TILE_RING) return fail(MOE_I8_EINVAL, "unknown GEMM variant %d", variant);
  return MOE_I8_OK;
}
int dense_plan(const DenseChoice& choice, const moe_i8::GemmArgs& g, int variant, moe_i8_dense_kernel* out) {
  moe_i8_dense_kernel plan{MOE_I8_DENSE_FEW, 0, 0, choice.entry, 0};
  if (choice.way == kGrouped) {
    plan.kernel = picks_kernel(g, grouped_variant(g, variant));
    if (plan.kernel < 0) return MOE_I8_EUNSUPPORTED;
  } else if (choice.way != kFew) {
    const moe_i8::DenseTile tile = choice.way == kDense ? moe_i8::gemm_dense_tile(choice.entry) : moe_i8::dense_rows_tile(choice.entry);
    plan = {choice.way == kDense ? MOE_I8_DENSE_TILES : MOE_I8_DENSE_ROWS, tile.rows, tile.channels, choice.entry,
            choice.way == kRows || moe_i8::gemm_dense_through(g.mode, g.num_pairs, g.n)};
  }
  if (out) *out = plan;
  return MOE_I8_OK;
}

// The ties-to-even row quantiser of the dense path; `padded`: rows for the dense kernel; `route`: its
// threads also write the identity routing the grouped families read (one launch less).
int dense_quant(const void* x, int64_t m, int k, int8_t* q, float* scale, bool padded, bool route, const DenseCarve& c,
                char* ws, hipStream_t stream) {
  moe_i8::QuantArgs a;
  a.x = static_cast<const uint16_t*>(x);
  a.src_rows = m;
  a.cols = k;
  a.row_stride = k;
  a.gather = nullptr;
  a.gather_div = 1;
  a.rows = m;
  a.q = q;
  a.scale = scale;
  a.round_even = 1;
  if (padded) a.q_stride = moe_i8::dense_row_stride(k);
  if (route) {
    a.route_sorted = reinterpret_cast<int32_t*>(ws + c.sorted);
    a.route_expert_ids = reinterpret_cast<int32_t*>(ws + c.eids);
    a.route_npp = reinterpret_cast<int32_t*>(ws + c.npp);
    a.route_block = kDenseBlock;
    a.route_cap = c.cap;
  }
  return check_launch(moe_i8::launch_quant_rows(a, stream), "quant_rows");
}

int check_dense(const void* x, int64_t m, int k, void* workspace, int64_t workspace_bytes, const DenseCarve& c) {
  if (m > INT32_MAX - kDenseBlock) return fail(MOE_I8_EINVAL, "too many rows");
  if (reinterpret_cast<uintptr_t>(workspace) & 255u) return fail(MOE_I8_EINVAL, "workspace must be 256-byte aligned");
  if (workspace_bytes < c.total)
    return fail(MOE_I8_EWORKSPACE, "workspace %lld < %lld bytes", (long long)workspace_bytes, (long long)c.total);
  if (k < 8 || k % 8) return fail(MOE_I8_EINVAL, "k (%d) must be a positive multiple of 8", k);
  if (!aligned16(x)) return fail(MOE_I8_EINVAL, "x must be 16-byte aligned");
  return MOE_I8_OK;
}
}  // namespace

int64_t moe_i8_dense_workspace_bytes(int64_t m, int k, int inter) {
  if (m < 0 || k < 1 || inter < 0) return -1;
  return dense_carve(m, k, inter).total;
}

int moe_i8_w8a8_linear(const void* x, const int8_t* w, const float* w_scale, void* out, int64_t m, int n,
                       int k, void* workspace, int64_t workspace_bytes, int variant, void* stream) {
  if (m < 0) return fail(MOE_I8_EINVAL, "negative m");
  if (m == 0) return MOE_I8_OK;
  if (!x || !w || !w_scale || !out || !workspace) return fail(MOE_I8_EINVAL, "null pointer");
  const DenseCarve c = dense_carve(m, k, 0);
  if (int rc = check_dense(x, m, k, workspace, workspace_bytes, c)) return rc;
  char* ws = static_cast<char*>(workspace);
  hipStream_t s = static_cast<hipStream_t>(stream);
  int8_t* x_q = reinterpret_cast<int8_t*>(ws + c.x_q);
  float* a1 = reinterpret_cast<float*>(ws + c.a1);
  const moe_i8::GemmArgs g = dense_group(moe_i8::kDown, c, ws, x_q, a1, w, w_scale, out, m, n, k);
  const WorkspaceTurn turn(workspace);
  const DenseChoice choice = dense_choice(g, variant, may_quantise(x, g));
  if (choice.way >= kRows) return run_unquantised(choice, x, g, s);
  const bool dense = choice.way == kDense;
  if (int rc = dense_quant(x, m, k, x_q, a1, dense, !dense, c, ws, s)) return rc;
  return run_quantised(choice, g, variant, s);
}

int moe_i8_w8a8_mlp(const void* x, const int8_t* w13, const float* w13_scale, const int8_t* w2,
                    const float* w2_scale, void* out, int64_t m, int hidden, int inter, void* workspace,
                    int64_t workspace_bytes, int variant, void* stream) {
  if (m < 0) return fail(MOE_I8_EINVAL, "negative m");
  if (m == 0) return MOE_I8_OK;
  if (!x || !w13 || !w13_scale || !w2 || !w2_scale || !out || !workspace) return fail(MOE_I8_EINVAL, "null pointer");
  if (inter < 64 || inter % 64) return fail(MOE_I8_EINVAL, "inter (%d) must be a positive multiple of 64", inter);
  const DenseCarve c = dense_carve(m, hidden, inter);
  if (int rc = check_dense(x, m, hidden, workspace, workspace_bytes, c)) return rc;
  char* ws = static_cast<char*>(workspace);
  hipStream_t s = static_cast<hipStream_t>(stream);
  int8_t* x_q = reinterpret_cast<int8_t*>(ws + c.x_q);
  float* a1 = reinterpret_cast<float*>(ws + c.a1);
  int8_t* act_q = reinterpret_cast<int8_t*>(ws + c.act_q);
  float* a2 = reinterpret_cast<float*>(ws + c.a2);
  const moe_i8::GemmArgs gu = dense_group(moe_i8::kGateUpSilu, c, ws, x_q, a1, w13, w13_scale, ws + c.act, m, 2 * inter, hidden);
  moe_i8::GemmArgs dg = dense_group(moe_i8::kDown, c, ws, act_q, a2, w2, w2_scale, out, m, hidden, inter);
  const WorkspaceTurn turn(workspace);
  const auto [choice_gu, choice_dg] = mlp_choice(gu, dg, variant, may_quantise(x, gu), may_quantise(ws + c.act, dg));
  const bool dense_dg = choice_dg.way == kDense;
  if (choice_gu.way >= kRows) {
    if (int rc = check_dense_gemm(dg, variant)) return rc;  // before anything is launched
    if (int rc = run_unquantised(choice_gu, x, gu, s)) return rc;
  } else {
    const bool dense_gu = choice_gu.way == kDense;
    if (int rc = dense_quant(x, m, hidden, x_q, a1, dense_gu, !dense_gu || choice_dg.way == kGrouped, c, ws, s)) return rc;
    if (int rc = run_quantised(choice_gu, gu, variant, s)) return rc;
  }
  if (choice_dg.way >= kRows) return run_unquantised(choice_dg, ws + c.act, dg, s);
  // Few rows on the streaming family: its down GEMM quantises them itself (ties to even here), one
  // launch less.
  if (variant == MOE_I8_GEMM_STREAM && m <= kDenseSelfQuantRows && inter <= kSelfQuantMaxInter) {
    if (int rc = check_gemm_common(ws + c.act, w2, dg.sorted_token_ids, dg.expert_ids, dg.num_tokens_post_padded, out, m, 1,
                                   hidden, inter, kDenseBlock, c.cap, MOE_I8_GEMM_STREAM))
      return rc;
    if (!aligned16(w2_scale)) return fail(MOE_I8_EINVAL, "w2_scale must be 16-byte aligned");
    dg.a_q = nullptr;
    dg.a_scale = nullptr;
    dg.a_bf16 = reinterpret_cast<const uint16_t*>(ws + c.act);
    dg.a_round_even = true;
    return check_launch(moe_i8::launch_gemm_stream(dg, s), "gemm_stream");
  }
  if (int rc = dense_quant(ws + c.act, m, inter, act_q, a2, dense_dg, false, c, ws, s)) return rc;
  return run_quantised(choice_dg, dg, variant, s);
}

int moe_i8_linear_plan(int64_t m, int n, int k, int variant, moe_i8_dense_kernel* product) {
  if (int rc = dense_shape_args(m, n, k, variant)) return rc;
  const DenseCarve c = dense_carve(m, k, 0);
  const moe_i8::GemmArgs g = dense_group(moe_i8::kDown, c, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, m, n, k);
  return dense_plan(dense_choice(g, variant, true), g, variant, product);
}

int moe_i8_mlp_plan(int64_t m, int hidden, int inter, int variant, moe_i8_dense_kernel* gate_up, moe_i8_dense_kernel* down) {
  if (inter < 64 || inter % 64) return fail(MOE_I8_EINVAL, "inter (%d) must be a positive multiple of 64", inter);
  if (int rc = dense_shape_args(m, hidden, hidden, variant)) return rc;
  const DenseCarve c = dense_carve(m, hidden, inter);
  const moe_i8::GemmArgs gu = dense_group(moe_i8::kGateUpSilu, c, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, m, 2 * inter, hidden);
  const moe_i8::GemmArgs dg = dense_group(moe_i8::kDown, c, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, m, hidden, inter);
  const MlpChoice choice = mlp_choice(gu, dg, variant, true, true);
  if (int rc = dense_plan(choice.gate_up, gu, variant, gate_up)) return rc;
  return dense_plan(choice.down, dg, variant, down);
}

}  // extern "C"
