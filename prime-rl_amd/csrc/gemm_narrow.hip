// Grouped int8 GEMM for gfx950, narrow-tile family (tens of rows per expert: small prefill chunks,
// large decode batches).
//
// In this regime every expert is active, a block of 64 rows is all the reuse a weight byte gets,
// and the layer is bound by streaming the weights from HBM once.  What matters is that the stream
// never stops, and that the compute units end together: one workgroup of eight wavefronts per
// compute unit walks its tiles with a ring of six or seven LDS stages, so that five or six reduction
// steps of loads (80-96 KB of weights) are in flight at all times, also across the end of a tile and
// through its epilogue.
//
// A tile's loads and a step's work are kept off the stream's critical path: tasks are looked up 64 at a time,
// token ids travel two tiles ahead, and a step reads its operands before it issues the loads of a later step
// between its multiplications.  What does not change during a step is decided outside the loop over the steps, of which
// there is one per kind of wavefront and of loads: with some twenty branches in it a step cost 0.5 us even where all of its
// rows came from L2, now 0.42; where they come from memory, 0.51-0.55 us a step are 7.6 TB/s of weights.
// Before that -> after, with the starting steps of start_step, the divided last rounds of piece_at and the stores described
// below, in turn on one box, us: the layer of 128 experts of 2048 x 768 at 203 tokens 117.4 -> 115.7, 4096 x 1408 with skewed
// routing at 32 tokens 128 -> 122, 256 experts of 7168 x 2048 at 64 tokens 874 -> 866 (on another box no difference); gate_up +
// down, 64 experts of 4096 x 1408 with 20 / 40 rows each 128.5 + 65.9 / 142 + 78.1 -> 118 + 64.1 / 126 + 69.7, 96 of 3072 x 1024
// 95.0 + 57.0 / 108.9 + 68.3 -> 94.3 + 52.5 / 106.0 + 59.5.
//
// A tile is TOK token rows (32 or 64: part of a moe_align block) x 128 weight rows; the reduction runs
// in steps of 128 bytes and both operands reach LDS by global -> LDS loads (global_load_lds_dwordx4, no
// staging registers).  Wavefront w multiplies weight rows [64 * (w % 2), + 64) of the tile with token rows
// [16 * (w / 2), + 16), used "transposed" (A operand = weight rows), so a lane ends up with runs of 4 consecutive
// channels of one token; after an exchange between lanes a store covers 64 bytes of 16 rows.  For the
// gate_up GEMM the 64 weight rows of a wavefront are 16 gate rows, the 16 matching up rows and once more, which
// puts a gate value and its up value into the same lane.  (32 weight rows x 32 token rows per wavefront read a fifth less
// from LDS, which made steps whose rows come from L2 5 % faster, but their stores were pieces of 32 bytes: 128 experts of
// 2048 x 768 with 14 / 32 / 64 rows each, gate_up + down, 61 + 37.7 / 66 + 43.5 / 79.5 + 54 -> 61 + 36.4 / 64.6 + 41.4 /
// 70.5 + 51.8 us.)
//
// Nothing in the steady state is a compiler-visible vector load: token ids, activation scales,
// routed weights and channel scales of later tiles also travel global -> LDS (4 bytes per lane) while
// the current tile is reduced, into a small triple-buffered area.  The only waits on vector memory are
// therefore the explicit ones of the ring.  They count a wavefront's stage loads only: the few other
// operations (those 4-byte loads, an epilogue's stores) make a wait slightly stricter than needed,
// never weaker.
//
// LDS rows are 128 bytes; the 16-byte chunk index is XOR-swizzled with row bits so that the MFMA
// operand reads spread over all banks; because a load fills LDS linearly the swizzle is applied to the
// global source address of each lane.
#include <type_traits>

#include "lds_loads.hpp"
#include "tile_list.hpp"

namespace moe_i8 {
namespace {

constexpr int kThreads = kTileThreads;
constexpr int kWaves = kThreads / kWave;
constexpr int kCh = 128;    // weight rows per tile
constexpr int kMinSteps = 4;
constexpr int64_t kThroughBytes = 8 << 20;  // results of a launch from which on they are written through (see launch_mode)

template <int TOK>
struct Shape {
  static constexpr int kStages = TOK == 64 ? 6 : 7;
  static constexpr int kStageBytes = (kCh + TOK) * kStepBytes;  // 24 | 20 KB
  static constexpr int kTokWaves = TOK / 8;                     // wavefronts that load token rows (8 rows each)
};

// Inputs of one tile's epilogue (and of the loads of its token rows), filled by 4-byte global -> LDS
// loads while earlier tiles are reduced.  Every wavefront fetches what it reads itself.
struct TileAux {
  int32_t ids[64];    // sorted_token_ids of the tile's rows
  float a_scale[64];  // activation scale of each row (0 index for padding rows)
  float row_w[64];    // routed weight of each row (down GEMM)
  float w_scale[kCh]; // down: scales of the tile's 128 channels; gate_up: 64 gate scales, 64 up scales
};

struct NarrowParams {
  const int8_t* a_q;
  const float* a_scale;
  const int8_t* w;
  const float* w_scale;
  const float* row_weight;  // null = 1
  const int32_t* sorted_ids;
  const int32_t* expert_ids;
  const int32_t* npp;
  int P;
  Divider row_of;
  int E;
  int N;
  int K;
  int B;
  int ntiles;  // channel tiles
  int rotate;  // steps between the starts of two experts that follow each other (rotation)
  bool through;  // results are written through to memory (see launch_mode)
  void* out;
};

__device__ __forceinline__ void load_to_lds_dword(const void* base, uint32_t offset, uint32_t lds_addr) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2"
               :
               : "s"((uint32_t)__builtin_amdgcn_readfirstlane((int)lds_addr)), "v"(offset), "s"(uniform_address(base))
               : "memory", "m0");
}

struct Task {
  int e;          // expert; -1 = no more work
  int n0, n1;     // its channels
  int64_t slot0;  // first slot of the tile in sorted_ids
  bool single;    // nothing else reads the expert's weight rows
};

struct TaskLoads {
  const int8_t* wbase;  // weights of the task's expert (wave-uniform)
  bool stream;          // fetch the weight rows with the non-temporal hint
  int first;            // byte offset of the first reduction step
  uint32_t woff[2];     // per lane: byte offset of its chunk of weight row i from wbase
  uint32_t xoff;        // per lane: byte offset of its chunk of its token row from a_q
};

// FULL: the reduction has at least kStages steps, so that the ring is always full and every wait the same.
template <int MODE, int TOK, bool FULL>
__global__ __launch_bounds__(kThreads, 2) void gemm_narrow_kernel(NarrowParams p) {
  using S = Shape<TOK>;
  using F = Mfma<16>;
  constexpr int kStages = S::kStages;
  constexpr int kStageBytes = S::kStageBytes;
  constexpr int kTokOffset = kCh * kStepBytes;
  constexpr int kOut = MODE == kGateUpSilu ? kCh / 2 : kCh;  // channels of a whole tile
  __shared__ __align__(16) char stages[kStages * kStageBytes];
  __shared__ __align__(16) TileAux aux[3];

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int cg = wave & 1;            // channel half
  const int tok0 = (wave >> 1) * 16;  // first of its 16 token rows
  const int lrow = lane & 15;
  const int lgrp = lane >> 4;
  const int K = p.K;
  const int nk = K / kStepBytes;
  const int inter = p.N / 2;
  const int width = MODE == kGateUpSilu ? inter : p.N;
  const bool loads_tokens = S::kTokWaves == kWaves || wave < S::kTokWaves;
  // Steps the loads run ahead of the multiplication: the ring's depth, less for very short reductions (the
  // rows of the next tile are set up in the first step of the current one).
  const int ahead = FULL ? kStages - 1 : nk - 1;

  // ---- this workgroup's tasks: (block, channel tile), channel tile fastest, split into 8 contiguous
  // ranges, one per XCD (workgroup id % 8), so that workgroups that run side by side share token
  // rows and expert weights in that XCD's L2.  A block of more than TOK rows is walked in as many
  // phases: the first TOK rows of all blocks, then the next (most of those are padding and skipped).
  const int npp = *p.npp;
  const int nblocks = npp / p.B;
  const int sub_per_block = p.B / TOK;
  const int total = nblocks * p.ntiles;
  const int per_xcd = (total + kXcds - 1) / kXcds;
  const int xcd = blockIdx.x % kXcds;
  const int stride = gridDim.x / kXcds;
  const int in_range = total - xcd * per_xcd < per_xcd ? total - xcd * per_xcd : per_xcd;
  const int rounds = (per_xcd + stride - 1) / stride;  // of a phase

  // Candidate tasks of this workgroup: its places in the rounds of its XCD's range, phase by phase (a task of a last round
  // that leaves workgroups idle is cut into pieces of its channels).  Lane i
  // looks up candidate 64 * chunk + i, so that taking the next task is a bit scan and a few lane reads: looked
  // up one by one (two dependent scalar reads, about 1 us) they held up every tile, whose steps are 0.6 us.
  // A task needs a valid expert id and rows that are not all padding (valid rows are a prefix of a block).
  const int candidates = rounds * sub_per_block;
  uint64_t open = 0;  // candidates of the current chunk not handed out yet
  int chunk_base = 0, lane_e = 0, lane_blk = 0, lane_n0 = 0, lane_n1 = 0, lane_flags = 0;
  auto look_up = [&]() {
    const int i = chunk_base + lane;
    const int sub = i / rounds;
    const TaskPiece tp = piece_at((int)(blockIdx.x / kXcds) + (i - sub * rounds) * stride, in_range, stride);
    bool ok = i < candidates && tp.task >= 0;
    const int task = xcd * per_xcd + (ok ? tp.task : 0);
    const int blk = ok ? task / p.ntiles : 0;
    const int64_t slot0 = (int64_t)blk * p.B + (int64_t)(ok ? sub : 0) * TOK;
    const int e = p.expert_ids[blk];
    const int32_t first = p.sorted_ids[slot0];
    // Does the expert hold other tiles?  Its neighbours in the block list, and the next tile of the same block
    // (the next tile's first slot says whether it is in use; any tile but the first has the one in front of it).
    const int before = p.expert_ids[blk > 0 ? blk - 1 : blk];
    const int after = p.expert_ids[blk + 1 < nblocks ? blk + 1 : blk];
    const int32_t other = p.sorted_ids[slot0 + (sub + 1 < sub_per_block && ok ? TOK : 0)];
    // all of them used here, so that the compiler waits for these loads here and not inside the ring's loop
    asm volatile("" ::"v"(e), "v"(first), "v"(before), "v"(after), "v"(other));
    ok = ok && e >= 0 && e < p.E && first >= 0 && first < p.P;
    const bool single = sub == 0 && (blk == 0 || before != e) && (blk + 1 >= nblocks || after != e) &&
                        (sub_per_block == 1 || !(other >= 0 && other < p.P));
    lane_e = e;
    lane_blk = blk;
    const int width = kOut / tp.pieces;
    lane_n0 = (task - blk * p.ntiles) * kOut + tp.piece * width;
    lane_n1 = lane_n0 + width;
    lane_flags = sub * 2 + (single ? 1 : 0);
    open = __ballot(ok);
  };
  auto next_task = [&]() {
    Task tk;
    tk.e = -1;
    tk.n0 = tk.n1 = 0;
    tk.slot0 = 0;
    tk.single = false;
    while (open == 0 && chunk_base + kWave < candidates) {
      chunk_base += kWave;
      look_up();
    }
    if (open != 0) {
      const int i = __ffsll((unsigned long long)open) - 1;
      open &= open - 1;
      const int flags = __builtin_amdgcn_readlane(lane_flags, i);
      tk.e = __builtin_amdgcn_readlane(lane_e, i);
      tk.n0 = __builtin_amdgcn_readlane(lane_n0, i);
      tk.n1 = __builtin_amdgcn_readlane(lane_n1, i);
      tk.slot0 = (int64_t)__builtin_amdgcn_readlane(lane_blk, i) * p.B + (flags >> 1) * TOK;
      tk.single = flags & 1;
    }
    return tk;
  };

  const uint32_t stage0 = lds_address(stages);
  auto in_use = [&](int32_t id) { return (uint32_t)id < (uint32_t)p.P; };

  // ---- global -> LDS loads ----
  // the task's channel c, the last one again behind its end
  auto channel = [&](const Task& tk, int c) { return min(tk.n0 + c, min(tk.n1, width) - 1); };
  // Lane fills LDS slot (lane & 7) of row base + 8 * i + (lane >> 3): it fetches the logical chunk
  // (lane & 7) ^ swizzle(row) of that row.
  auto setup_weight_loads = [&](const Task& tk, TaskLoads& ld) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int row = 16 * wave + 8 * i + (lane >> 3);  // LDS weight row; the wavefronts of channel half row / 64 multiply it
      const int chunk = ((lane & 7) ^ swizzle_of_row(row)) * 16;
      int n;
      if constexpr (MODE == kGateUpSilu) {
        const int j = row & 31;
        n = channel(tk, (row >> 5) * 16 + (j & 15)) + (j >= 16 ? inter : 0);
      } else {
        n = channel(tk, row);
      }
      ld.woff[i] = (uint32_t)n * (uint32_t)K + chunk;
    }
    ld.wbase = p.w + (int64_t)tk.e * p.N * K;
    ld.stream = tk.single;
    ld.first = start_step(tk.e, p.rotate) * kStepBytes;
  };
  auto setup_token_loads = [&](const TileAux& ax, TaskLoads& ld) {
    const int row = (8 * wave + (lane >> 3)) & (TOK - 1);
    const int chunk = ((lane & 7) ^ swizzle_of_row(row)) * 16;
    const int32_t tok = ax.ids[row];
    const uint32_t arow = in_use(tok) ? p.row_of(tok) : 0u;
    ld.xoff = arow * (uint32_t)K + chunk;
  };
  auto issue_weights = [&](const TaskLoads& ld, int stage, int koff) {
    const uint32_t base = stage0 + stage * kStageBytes + wave * 2048;
    if (ld.stream) {
#pragma unroll
      for (int i = 0; i < 2; ++i) load_to_lds_16_stream(ld.wbase + koff, ld.woff[i], base + i * 1024);
    } else {
#pragma unroll
      for (int i = 0; i < 2; ++i) load_to_lds_16(ld.wbase + koff, ld.woff[i], base + i * 1024);
    }
  };
  auto issue_tokens = [&](const TaskLoads& ld, int stage, int koff) {
    if (loads_tokens) load_to_lds_16(p.a_q + koff, ld.xoff, stage0 + stage * kStageBytes + kTokOffset + wave * 1024);
  };
  auto issue_ids = [&](const Task& tk, TileAux& ax) {
    load_to_lds_dword(p.sorted_ids + tk.slot0, (uint32_t)(lane & (TOK - 1)) * 4u, lds_address(ax.ids));
  };
  auto issue_scales = [&](const Task& tk, TileAux& ax) {
    if constexpr (MODE == kAccI32) return;
    const int32_t tok = ax.ids[lane & (TOK - 1)];
    const uint32_t t = in_use(tok) ? (uint32_t)tok : 0u;
    load_to_lds_dword(p.a_scale, p.row_of((int)t) * 4u, lds_address(ax.a_scale));
    const float* wsc = p.w_scale + (int64_t)tk.e * p.N;
    if constexpr (MODE == kDown) {
      // without routed weights the slot is filled with something readable and never used
      if (p.row_weight)
        load_to_lds_dword(p.row_weight, t * 4u, lds_address(ax.row_w));
      else
        load_to_lds_dword(p.a_scale, 0u, lds_address(ax.row_w));
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        load_to_lds_dword(wsc, (uint32_t)channel(tk, 64 * j + lane) * 4u, lds_address(ax.w_scale + 64 * j));
      }
    } else {
      const uint32_t c = (uint32_t)channel(tk, lane);
      load_to_lds_dword(wsc, c * 4u, lds_address(ax.w_scale));
      load_to_lds_dword(wsc, (c + (uint32_t)inter) * 4u, lds_address(ax.w_scale + 64));
    }
  };
  // this wavefront's loads of all but the `steps` most recent steps are in
  auto wait_all_but = [&](int steps) {
    if (loads_tokens)
      wait_groups<3, kStages - 2>(steps);
    else
      wait_groups<2, kStages - 2>(steps);
  };

  // ---- MFMA operand reads ----
  int w_ld[4], chunk[2];
#pragma unroll
  for (int i = 0; i < 4; ++i) w_ld[i] = (64 * cg + 16 * i + lrow) * kStepBytes;
  const int x_ld = kTokOffset + (tok0 + lrow) * kStepBytes;
#pragma unroll
  for (int kk = 0; kk < 2; ++kk) chunk[kk] = ((4 * kk + lgrp) ^ swizzle_of_row(lrow)) * 16;

  // Token row tok0 + lrow of the tile; acc[i][r] is weight row 16 * i + 4 * lgrp + r of this wavefront's 64.
  auto epilogue = [&](const Task& tk, const TileAux& ax, typename F::Acc (&acc)[4]) {
    const int row = tok0 + lrow;
    const int32_t tok = ax.ids[row];
    if (!in_use(tok)) return;
    const int limit = min(tk.n1, width);
    auto piece = [&](int j, int (&v)[4]) {
#pragma unroll
      for (int r = 0; r < 4; ++r) v[r] = acc[j][r];
    };
    // Results of 16 + 16 channels: the lanes of a row trade halves, so that each holds 8 consecutive channels and a store
    // covers 64 bytes of 16 rows.
    auto store = [&](uint16_t* line, int n, const uint2& a, const uint2& b) {
      const auto x = __builtin_amdgcn_permlane16_swap(a.x, b.x, false, false), y = __builtin_amdgcn_permlane16_swap(a.y, b.y, false, false);
      n += 16 * (lgrp & 1) + 8 * (lgrp >> 1);
      if (n < limit) store16(line + n, v4i{(int)x[0], (int)y[0], (int)x[1], (int)y[1]}, p.through);
    };
    if constexpr (MODE == kGateUpSilu) {
      // weight rows 0..15 and 32..47 of the wavefront are gate channels, 16..31 and 48..63 the matching up channels
      const float as = ax.a_scale[row];
      uint2 h[2];
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const int c = 32 * cg + 16 * j + 4 * lgrp;
        int g[4], u[4];
        piece(2 * j, g);
        piece(2 * j + 1, u);
        h[j] = silu_mul_epilogue4(g, u, as, *reinterpret_cast<const float4*>(ax.w_scale + c), *reinterpret_cast<const float4*>(ax.w_scale + 64 + c));
      }
      store(static_cast<uint16_t*>(p.out) + (int64_t)tok * inter, tk.n0 + 32 * cg, h[0], h[1]);
    } else {
      const float as = MODE == kDown ? ax.a_scale[row] : 0.0f;
      const float rw = MODE == kDown && p.row_weight ? ax.row_w[row] : 1.0f;
      uint2 h[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int c = 64 * cg + 16 * j + 4 * lgrp;
        int v[4];
        piece(j, v);
        if constexpr (MODE == kAccI32) {
          if (tk.n0 + c < limit)
            *reinterpret_cast<v4i*>(static_cast<int32_t*>(p.out) + (int64_t)tok * p.N + tk.n0 + c) = v4i{v[0], v[1], v[2], v[3]};
        } else {
          h[j] = down_epilogue4(v, as, *reinterpret_cast<const float4*>(ax.w_scale + c), rw);
        }
      }
      if constexpr (MODE == kDown) {
        uint16_t* line = static_cast<uint16_t*>(p.out) + (int64_t)tok * p.N;
        store(line, tk.n0 + 64 * cg, h[0], h[1]);
        store(line, tk.n0 + 64 * cg + 32, h[2], h[3]);
      }
    }
  };

  // ---- start-up: the first task's weights need nothing but its expert; then what depends on its row ids.
  // Then the rows of the second task (its loads start `ahead` steps before the first one's last).
  if (total == 0) return;
  look_up();
  Task tk = next_task();
  if (tk.e < 0) return;
  TaskLoads ld;
  auto from = [&](const TaskLoads& ld, int s) {
    const int at = ld.first + s * kStepBytes;
    return at < K ? at : at - K;
  };
  constexpr int kEarly = 2;  // steps whose weights are requested before the row ids are in
  issue_ids(tk, aux[0]);
  setup_weight_loads(tk, ld);
#pragma unroll
  for (int s = 0; s < kEarly; ++s) issue_weights(ld, s, from(ld, s));
  Task nx = next_task();
  issue_ids(nx.e >= 0 ? nx : tk, aux[1]);
  Task n2 = next_task();
  // the ids of the first task are the oldest load; every wavefront fetched its own copy, so no barrier is needed
  wait_vmcnt<2 * kEarly>();
  setup_token_loads(aux[0], ld);
#pragma unroll
  for (int s = 0; s < kEarly; ++s) issue_tokens(ld, s, from(ld, s));
  issue_scales(tk, aux[0]);
  for (int s = kEarly; s < ahead; ++s) {
    issue_weights(ld, s, from(ld, s));
    issue_tokens(ld, s, from(ld, s));
  }
  int next_at = from(ld, ahead);  // byte offset of the next step to fetch, of the task that `ld` is set up for
  wait_all_but(ahead - kEarly);  // steps 0 and 1 (their loads are not in the order of the steps)

  int par = 0;                     // aux of the current task; the next ones follow
  int read_at = 0;                 // ring offset of the step being multiplied
  int fill_at = ahead * kStageBytes;  // ... of the step being fetched
  const uint32_t wdst = stage0 + wave * 2048, xdst = stage0 + kTokOffset + wave * 1024;
  // a wavefront whose part of the tile is padding (valid rows are a prefix) only loads
  auto part_in_use = [&](const TileAux& ax) { return tok0 < TOK && in_use(__builtin_amdgcn_readfirstlane(ax.ids[tok0])); };
  bool active = part_in_use(aux[0]), next_active = false;
  while (true) {
    typename F::Acc acc[4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int r = 0; r < F::kRegs; ++r) acc[i][r] = 0;
    TileAux& ax_next = aux[par + 1 < 3 ? par + 1 : par - 2];
    TileAux& ax_n2 = aux[par + 2 < 3 ? par + 2 : par - 1];
    int advance = kStepBytes;
    // Steps [s0, s1), during which the loads are those of one task.  This loop is what the kernel does all the time, and
    // with few rows its instructions, not the memory, are what a step costs as soon as the rows come from L2: everything
    // that does not change inside is decided outside.
    auto steps = [&](auto active_tag, auto stream_tag, int s0, int s1) {
      constexpr bool ACTIVE = decltype(active_tag)::value, STREAM = decltype(stream_tag)::value;
      for (int s = s0; s < s1; ++s) {
        // everybody's loads of step s have landed, and everybody is done reading the stage that is filled next
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        // Operands first, then the loads of the step `ahead` of this one a piece at a time between the
        // multiplications: the address unit takes 16 clocks per load and the whole workgroup's 20-24 of them in front
        // of the operand reads made a step 0.45 us even where every load hit L2.
        const char* st = stages + read_at;
        v4i a[2][4], b[2];
        if constexpr (ACTIVE) {
#pragma unroll
          for (int kk = 0; kk < 2; ++kk) {
            b[kk] = *reinterpret_cast<const v4i*>(st + x_ld + chunk[kk]);
#pragma unroll
            for (int i = 0; i < 4; ++i) a[kk][i] = *reinterpret_cast<const v4i*>(st + w_ld[i] + chunk[kk]);
          }
        }
        const int8_t* wsrc = ld.wbase + next_at;
        const int8_t* xsrc = p.a_q + next_at;
        auto mul = [&](int kk, int half) {
          if constexpr (ACTIVE)
#pragma unroll
            for (int i = 2 * half; i < 2 * half + 2; ++i) acc[i] = F::mul(a[kk][i], b[kk], acc[i]);
        };
        auto one_weight = [&](int i) {
          if constexpr (STREAM)
            load_to_lds_16_stream(wsrc, ld.woff[i], wdst + fill_at + i * 1024);
          else
            load_to_lds_16(wsrc, ld.woff[i], wdst + fill_at + i * 1024);
        };
        mul(0, 0);
        one_weight(0);
        mul(0, 1);
        one_weight(1);
        mul(1, 0);
        if (loads_tokens) load_to_lds_16(xsrc, ld.xoff, xdst + fill_at);
        mul(1, 1);
        if (s == 1) {
          if (nx.e >= 0) issue_scales(nx, ax_next);
          if (n2.e >= 0) issue_ids(n2, ax_n2);
        }
        next_at = next_at + advance < K ? next_at + advance : 0;
        read_at = read_at + kStageBytes < kStages * kStageBytes ? read_at + kStageBytes : 0;
        fill_at = fill_at + kStageBytes < kStages * kStageBytes ? fill_at + kStageBytes : 0;
        // this wavefront's loads of the next step have landed; after a task's last step, before its stores
        if constexpr (FULL) {
          if (loads_tokens)
            wait_vmcnt<3 * (kStages - 2)>();
          else
            wait_vmcnt<2 * (kStages - 2)>();
        } else {
          wait_all_but(ahead - 1);
        }
      }
    };
    // The loads run `ahead` steps in front of the multiplication: into the next task, or (nothing left) this task's last
    // step again and again, which keeps the counts uniform.
    for (int part = 0; part < 2; ++part) {
      const int s0 = part == 0 ? 0 : nk - ahead, s1 = part == 0 ? nk - ahead : nk;
      if (part == 1 && nx.e >= 0) {
        // the next task's rows (their ids were fetched a task ago)
        setup_weight_loads(nx, ld);
        setup_token_loads(ax_next, ld);
        next_at = ld.first;
        next_active = part_in_use(ax_next);
      } else if (part == 1) {
        next_at = (next_at > 0 ? next_at : K) - kStepBytes;
        advance = 0;
      }
      if (active && ld.stream)
        steps(std::true_type{}, std::true_type{}, s0, s1);
      else if (active)
        steps(std::true_type{}, std::false_type{}, s0, s1);
      else if (ld.stream)
        steps(std::false_type{}, std::true_type{}, s0, s1);
      else
        steps(std::false_type{}, std::false_type{}, s0, s1);
    }
    if (active) epilogue(tk, aux[par], acc);
    if (nx.e < 0) break;
    active = next_active;
    tk = nx;
    nx = n2;
    n2 = next_task();
    par = par + 1 < 3 ? par + 1 : 0;
  }
  wait_vmcnt<0>();
}

template <int MODE, int TOK>
hipError_t launch_mode(const GemmArgs& a, hipStream_t stream) {
  NarrowParams p;
  p.a_q = a.a_q;
  p.a_scale = a.a_scale;
  p.w = a.w;
  p.w_scale = a.w_scale;
  p.row_weight = a.row_weight;
  p.sorted_ids = a.sorted_token_ids;
  p.expert_ids = a.expert_ids;
  p.npp = a.num_tokens_post_padded;
  p.P = (int)a.num_pairs;
  p.row_of = divider(a.row_div);
  p.E = a.num_experts;
  p.N = a.n;
  p.K = a.k;
  p.B = a.block_size;
  p.ntiles = MODE == kGateUpSilu ? (a.n / 2 + 63) / 64 : (a.n + kCh - 1) / kCh;
  p.rotate = rotation(a.k, (int64_t)a.num_experts * a.n * a.k, a.num_experts);
  // Results left in the L2s are written back when they are displaced by the weight stream, line by line, and the rest when
  // the launch ends: with few of them that costs less than a write to memory per store, with many more.  Where the two cross
  // depends on the shape, and neither the bytes, the rows per expert nor the weights alone say where; 8 MB is the size from
  // which on writing through won for all shapes but one.  Left / written through, us, at the size where they are even and at 8 MB:
  // gate_up, 32 experts of 4096 x 1536 below 2 MB, at 6 69.9 / 66.2; 128 of 2048 x 512 2.5 MB, 52.2 / 48.9; 96 of 3072 x 1024
  // 3.5 MB, 108.5 / 105.2; 128 of 2048 x 768 4.5 MB, 72.1 / 68.0; 64 of 4096 x 1408 6.5 MB, 131.5 / 129.6; down, 32 of 4096 x 1536
  // 5 MB, 39.6 / 38.0; 64 of 4096 x 1408 5 MB, 64.2 / 62.1; 128 of 2048 x 768 5.5 MB, 39.2 / 38.2; 128 of 2048 x 512 6.5 MB, 31.2 /
  // 30.1; 96 of 3072 x 1024 10 MB, 50.8 / 52.0.  Below 8 MB the line so gives away up to 6 % (128 of 2048 x 512, gate_up), beyond
  // up to 2 (the last one); at 2 to 4 MB writing through would cost a down GEMM 1 to 5 %.
  p.through = a.num_pairs * (MODE == kGateUpSilu ? a.n / 2 : a.n) * 2 >= kThroughBytes;
  p.out = a.out;
  const int grid = device_cu_count() / kXcds * kXcds;
  if (a.k >= Shape<TOK>::kStages * kStepBytes)
    hipLaunchKernelGGL((gemm_narrow_kernel<MODE, TOK, true>), dim3((unsigned)grid), dim3(kThreads), 0, stream, p);
  else
    hipLaunchKernelGGL((gemm_narrow_kernel<MODE, TOK, false>), dim3((unsigned)grid), dim3(kThreads), 0, stream, p);
  return hipGetLastError();
}

// Tiles of 32 token rows where no expert can hold more (a block's second half would be all padding): the
// smaller stage leaves room for a seventh one and a third of the token loads goes away (17 tokens 84.6 -> 81.6 us,
// 40 tokens 109.5 -> 107.0).  Beyond that one expert with more rows would make its weights travel twice (skewed
// routing, 45 tokens: 139.6 -> 151.5).
bool small_tiles(const GemmArgs& a) {
  const int64_t most_rows = a.max_rows_per_expert > 0 && a.max_rows_per_expert < a.num_pairs ? a.max_rows_per_expert : a.num_pairs;
  return most_rows <= 32;
}

}  // namespace

bool gemm_narrow_supports(const GemmArgs& a) {
  // per-lane source offsets are 32-bit: one expert's weights, the activation matrix and the per-pair
  // arrays must each span less than 4 GiB
  const int64_t act_rows = (a.num_pairs + a.row_div - 1) / a.row_div;
  return (a.block_size == 64 || a.block_size == 128) && a.k % kStepBytes == 0 && a.k >= kMinSteps * kStepBytes && a.n % 16 == 0 &&
         (int64_t)a.n * a.k < (1ll << 32) && act_rows * a.k < (1ll << 32) && a.num_pairs < (1ll << 30) &&
         a.sorted_cap / 32 * ((a.n + 63) / 64) < (1ll << 31);
}

hipError_t launch_gemm_narrow(const GemmArgs& a, hipStream_t stream) {
  const bool small = small_tiles(a);
  switch (a.mode) {
    case kGateUpSilu: return small ? launch_mode<kGateUpSilu, 32>(a, stream) : launch_mode<kGateUpSilu, 64>(a, stream);
    case kDown: return small ? launch_mode<kDown, 32>(a, stream) : launch_mode<kDown, 64>(a, stream);
    case kAccI32: return small ? launch_mode<kAccI32, 32>(a, stream) : launch_mode<kAccI32, 64>(a, stream);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace moe_i8
