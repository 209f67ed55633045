// Grouped int8 GEMM for gfx950, deep tiles (some tens to about a hundred routed rows per expert, and skewed routing).
//
// One persistent workgroup of eight wavefronts per compute unit walks tiles of up to 128 token rows (consecutive moe_align
// blocks of one expert) x 256 weight rows (gate_up: 128 gate channels and their up channels); the reduction runs in steps of
// 128 bytes through a ring of three 48 KB LDS stages filled by global -> LDS loads two steps ahead.  The MFMA
// (v_mfma_i32_32x32x32_i8) is used "transposed" (A operand = weight rows): a lane ends up with 4 consecutive channels of a
// token, a wavefront with a quarter of the channels of the 32-row units th and th + 2.  The tasks are cut into ranges of XCDs
// and last rounds into pieces of channels as tile_list.hpp says, and start at the steps of start_step.
//
// What bounds it: the weight stream from memory where an expert has one tile (5.2-5.9e12 bytes per second of weights), the
// path from L2 into LDS (about 1 us a step of 48 KB) where it has several.  Hence:
//  * The step loop holds nothing but the step: a task's steps run in two parts, those whose loads are the task's own and
//    the last two, whose loads are the next task's; what differs by the part, the wavefront's units or the kind of
//    load is a template argument.  Operands are read ahead of the MFMAs and the loads go between them.  Tasks are
//    looked up 64 at a time, token ids travel two tasks ahead and scales one, all global -> LDS; waits count what is in
//    flight, the stores of the last epilogue included.  With scalar decisions in every step, tasks set up by dependent
//    loads and an epilogue that drained everything, 16 experts of 4096 x 1408 with 512 rows each took 114 + 63 us
//    (gate_up + down), 103 + 61 now; 78 experts with 12 to 517 rows 206 + 113, now 173 + 99.
//  * Results are staged in the last step's stage, 4 KB per wavefront, and stored 64 or 128 bytes of a row at a time, through
//    to memory.  64 experts of 4096 x 1408 with 96 rows each: 132 + 79 us; left in the L2s, where the weight stream displaces
//    them, 146 + 88.  With the non-temporal hint instead 133 + 80, and 78 experts with 12 to 517 rows 0.7 % of the layer
//    slower; with it and straight from registers in pieces of 32 bytes 138 + 113.
//  * Weight rows that nothing else reads are fetched with the non-temporal hint, so that they do not displace token rows from
//    L2: 64 experts of 4096 x 1408 with 40 rows each 139 + 84 us without, 132 + 76 with.  It is chosen per task: where only
//    some experts have several tiles the others still profit.
#include <type_traits>

#include "lds_loads.hpp"
#include "tile_list.hpp"

namespace moe_i8 {
namespace {

constexpr int kThreads = kTileThreads;
constexpr int kTok = 128;  // token rows per tile
constexpr int kCh = 256;   // weight rows per tile
constexpr int kUnit = 32;  // token rows of an MFMA
constexpr int kX0 = kCh * kStepBytes;            // token rows of a stage, behind the weight rows
constexpr int kStage = kX0 + kTok * kStepBytes;  // 48 KB
constexpr int kStages = 3;
constexpr int kAhead = kStages - 1;  // steps that the loads run ahead
constexpr int kMinSteps = 3;
constexpr int kMaxTiles = 2048;  // of a launch
constexpr int kTable = 64;       // tasks of a workgroup looked up at a time
constexpr int kLoads = 6;        // of a wavefront and step

struct DeepParams {
  const int8_t* a_q;
  const float* a_scale;
  const int8_t* w;
  const float* w_scale;
  const float* row_weight;  // null = 1
  const int32_t* sorted_ids;
  const int32_t* npp;
  int P;
  Divider row_of;
  int N;
  int K;
  int B;
  TileListArgs tiles;
  int ascend;  // expert_ids is known to ascend over the used blocks (it comes from moe_align)
  int rotate;  // steps between the starts of two experts that follow each other (rotation)
  void* out;
};

// What the loads of a tile's token rows and its epilogue need, filled by 4-byte global -> LDS loads while earlier tiles
// are reduced.
struct TileAux {
  int32_t ids[kTok];    // sorted_token_ids of the tile's rows
  float a_scale[kTok];  // activation scale of each row
  float row_w[kTok];    // routed weight of each row (down GEMM)
  float w_scale[kCh];   // scales of the tile's weight rows
};

struct Task {
  int e;        // expert; -1 = no more work
  int n0, n1;   // its channels (gate_up: gate channels)
  int slot0;    // first slot of the tile in sorted_ids
  int rows;     // slots of the tile
  bool single;  // nothing else reads the expert's weight rows
};

struct TaskLoads {
  const int8_t* wbase;  // weights of the task's expert (wave-uniform)
  bool stream;          // fetch the weight rows with the non-temporal hint
  int first;            // byte offset of the first reduction step
  int units;            // 32-row units up to the last row in use
  uint32_t woff[4];     // per lane: byte offset of its chunk of weight row i from wbase
  uint32_t xoff[2];     // per lane: byte offset of its chunk of token row i from a_q
};

__device__ __forceinline__ int uniform(int v) { return __builtin_amdgcn_readfirstlane(v); }

template <int MODE>
__global__ __launch_bounds__(kThreads, 2) void gemm_deep_kernel(DeepParams p) {
  using F = Mfma<kUnit>;
  __shared__ __align__(16) char stages[kStages * kStage];
  __shared__ __align__(16) TileAux aux[3];
  __shared__ TileList<kMaxTiles> list;
  // tasks it .. of this workgroup: block | blocks << 16 | piece << 20 | log2(pieces) << 22 | single << 31, task_word
  __shared__ uint2 table[kTable];
  constexpr int kOut = MODE == kGateUpSilu ? kCh / 2 : kCh;  // channels of a whole tile
  // counted stores of a wavefront and unit in an epilogue (the int32 results' are the compiler's and not counted)
  constexpr int kUnitStores = MODE == kGateUpSilu ? 2 : MODE == kDown ? 4 : 0;

  const int t = threadIdx.x;
  const int lane = t & 63;
  const int wave = uniform(t >> 6);
  const int cg = wave & 3;   // channel quarter
  const int th = wave >> 2;  // token units th and th + 2
  const int lrow = lane & 31;
  const int lgrp = lane >> 5;
  const int K = p.K;
  const int nk = K / kStepBytes;
  const int inter = p.N / 2;
  const int width = MODE == kGateUpSilu ? inter : p.N;

  const int xcd = blockIdx.x % kXcds;
  TileRange range = p.ascend ? build_ascending(p.tiles, xcd, reinterpret_cast<int*>(stages), list)
                             : build_any_order(p.tiles, uniform(*p.npp) / p.B, xcd, reinterpret_cast<int*>(stages), list);
  // (said to be wave-uniform: everything that follows from them then stays in scalar registers)
  range.lo = uniform(range.lo);
  range.hi = uniform(range.hi);
  range.tiles = uniform(range.tiles);
  const int total = range.tiles * p.tiles.ntiles;
  const int per_xcd = uniform((total + kXcds - 1) / kXcds);
  const int my_tasks = min(per_xcd, max(total - xcd * per_xcd, 0));  // of the XCD
  const int stride = gridDim.x / kXcds;
  int it = 0;  // tasks handed out

  // Looks up tasks n0 .. n0 + kTable - 1 of this workgroup.
  auto fill_table = [&](int n0) {
    if (t >= kTable) return;
    const TaskPiece tp = piece_at(blockIdx.x / kXcds + (n0 + t) * stride, my_tasks, stride);
    uint2 d = make_uint2(0u, kNoTask);
    if (tp.task >= 0) {
      d = look_up_task(p.tiles, list, range, xcd * per_xcd + tp.task);
      const bool single = (d.x >> 20) == (1u << 4);  // rank 0 of a group of one
      d.x = (d.x & 0xfffffu) | (uint32_t)tp.piece << 20 | (uint32_t)(tp.pieces >> 1) << 22 | (single ? 0x80000000u : 0u);
    }
    table[t] = d;
  };
  auto next_task = [&]() {
    const uint2 d = table[it % kTable];
    const uint32_t d0 = (uint32_t)uniform((int)d.x);
    const uint32_t d1 = (uint32_t)uniform((int)d.y);
    const int shift = (int)(d0 >> 22) & 3;  // 1, 2 or 4 pieces
    Task tk;
    tk.slot0 = (int)(d0 & 0xffffu) * p.B;
    tk.rows = (int)((d0 >> 16) & 15u) * p.B;
    tk.single = d0 >> 31;
    tk.n0 = task_channel_tile(d1) * kOut + ((int)(d0 >> 20) & 3) * (kOut >> shift);
    tk.n1 = tk.n0 + (kOut >> shift);
    tk.e = task_expert(d1);
    if (tk.e >= 0) ++it;
    return tk;
  };
  auto in_use = [&](int id) { return (uint32_t)id < (uint32_t)p.P; };
  // weight row of row r of a task's 256; the last channel again behind the task's end
  auto weight_row = [&](const Task& tk, int r) {
    if constexpr (MODE == kGateUpSilu)
      return min(tk.n0 + (r & 127), min(tk.n1, width) - 1) + (r >= 128 ? inter : 0);
    else
      return min(tk.n0 + r, min(tk.n1, width) - 1);
  };
  auto fetch_ids = [&](const Task& tk, TileAux& ax, int half) {
    const int row = half * 64 + lane;
    load_to_lds_4(p.sorted_ids + tk.slot0 + (row < tk.rows ? row : 0), lds_address(ax.ids) + half * 256);
  };
  // Inputs of a task's epilogue (its ids have landed), one load per wavefront.
  auto fetch_scales = [&](const Task& tk, TileAux& ax) {
    const int half = wave & 1;
    if (MODE == kAccI32 || wave >= 4) {
      const float* ws = MODE == kAccI32 ? reinterpret_cast<const float*>(p.w) : p.w_scale + (int64_t)tk.e * p.N + weight_row(tk, cg * 64 + lane);
      load_to_lds_4(ws, lds_address(ax.w_scale) + cg * 256);
    } else {
      const int row = half * 64 + lane;
      int id = ax.ids[row < tk.rows ? row : 0];
      if (!in_use(id)) id = 0;
      if (wave < 2)
        load_to_lds_4(p.a_scale + p.row_of(id), lds_address(ax.a_scale) + half * 256);
      else  // without routed weights the slot is filled with something readable and never used
        load_to_lds_4(MODE == kDown && p.row_weight ? p.row_weight + id : p.a_scale, lds_address(ax.row_w) + half * 256);
    }
  };
  // Lane fills LDS slot (lane & 7) of row base + 8 * i + (lane >> 3) of a wavefront's load i: it fetches chunk (lane & 7) ^
  // swizzle(row) of that row.
  auto setup_weights = [&](const Task& tk, TaskLoads& ld) {
    ld.wbase = p.w + (int64_t)tk.e * p.N * K;
    ld.stream = tk.single;
    ld.first = start_step(tk.e, p.rotate) * kStepBytes;
#pragma unroll
    for (int i = 0; i < 4; ++i)
      ld.woff[i] = (uint32_t)weight_row(tk, 32 * wave + 8 * i + (lane >> 3)) * (uint32_t)K + ((lane & 7) ^ (lane >> 3) ^ (i & 1)) * 16;
  };
  auto setup_tokens = [&](const Task& tk, const TileAux& ax, TaskLoads& ld) {
    // lane l looks at rows 2l and 2l + 1
    const int2 two = *reinterpret_cast<const int2*>(ax.ids + 2 * lane);
    const uint64_t used = __ballot(2 * lane < tk.rows && (in_use(two.x) || in_use(two.y)));
    ld.units = uniform(used ? (63 - __builtin_clzll(used)) / (kUnit / 2) + 1 : 0);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      // rows behind the last one in use fetch the tile's first row again
      int row = 16 * wave + 8 * i + (lane >> 3);
      if (row >= ld.units * kUnit) row = 0;
      const int32_t id = ax.ids[row];
      ld.xoff[i] = (in_use(id) ? p.row_of(id) : 0u) * (uint32_t)K + ((lane & 7) ^ (lane >> 3) ^ (i & 1)) * 16;
    }
  };

  // ---- MFMA operand reads: lane feeds row `lrow` of 32, chunk 2 * kk + lgrp; gate_up: 32 gate rows and their up rows ----
  int rd_w[4], rd_x[4];
#pragma unroll
  for (int kk = 0; kk < 4; ++kk) {
    const int at = lrow * kStepBytes + ((2 * kk + lgrp) ^ swizzle_of_row(lrow)) * 16;
    rd_w[kk] = (MODE == kGateUpSilu ? 32 : 64) * cg * kStepBytes + at;
    rd_x[kk] = kX0 + th * kUnit * kStepBytes + at;
  }
  constexpr int kSecondW = (MODE == kGateUpSilu ? 128 : 32) * kStepBytes;
  constexpr int kSecondX = 2 * kUnit * kStepBytes;

  // One unit's results: acc[ci][4q + r] is weight row 8q + 4 * lgrp + r of the wavefront's ci-th 32, token row row0 + lrow.
  // They go through `staging`, 4 KB of the wavefront's own, so that a store covers whole lines of few rows: the 16-byte chunks
  // of a row are kept at chunk ^ a part of the row, for the banks.
  auto epilogue = [&](const Task& tk, const TileAux& ax, const typename F::Acc (&acc)[2], int row0, char* staging) {
    const int row = row0 + lrow;
    const int limit = min(tk.n1, width);
    auto four = [&](const typename F::Acc& a, int q, int (&v)[4]) {
#pragma unroll
      for (int r = 0; r < 4; ++r) v[r] = a[4 * q + r];
    };
    if constexpr (MODE == kGateUpSilu) {
      const float as = ax.a_scale[row];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int c = 32 * cg + 8 * q + 4 * lgrp;
        int g[4], u[4];
        four(acc[0], q, g);
        four(acc[1], q, u);
        *reinterpret_cast<uint2*>(staging + lrow * 64 + (q ^ ((lrow >> 1) & 3)) * 16 + lgrp * 8) =
            silu_mul_epilogue4(g, u, as, *reinterpret_cast<const float4*>(ax.w_scale + c), *reinterpret_cast<const float4*>(ax.w_scale + 128 + c));
      }
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int r = 16 * i + (lane >> 2);
        const uint4 v = *reinterpret_cast<const uint4*>(staging + r * 64 + ((lane & 3) ^ ((r >> 1) & 3)) * 16);
        const int tok = ax.ids[row0 + r], n = tk.n0 + 32 * cg + 8 * (lane & 3);
        const bool ok = in_use(tok);
        store16_through(static_cast<uint16_t*>(p.out) + (int64_t)(ok ? tok : 0) * inter + n, v, __ballot(ok && n < limit));
      }
    } else if constexpr (MODE == kDown) {
      const float as = ax.a_scale[row];
      const float rw = p.row_weight ? ax.row_w[row] : 1.0f;
#pragma unroll
      for (int ci = 0; ci < 2; ++ci)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int c = 64 * cg + 32 * ci + 8 * q + 4 * lgrp;
          int v[4];
          four(acc[ci], q, v);
          *reinterpret_cast<uint2*>(staging + lrow * 128 + ((4 * ci + q) ^ (lrow & 7)) * 16 + lgrp * 8) =
              down_epilogue4(v, as, *reinterpret_cast<const float4*>(ax.w_scale + c), rw);
        }
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int r = 8 * i + (lane >> 3);
        const uint4 v = *reinterpret_cast<const uint4*>(staging + r * 128 + ((lane & 7) ^ (r & 7)) * 16);
        const int tok = ax.ids[row0 + r], n = tk.n0 + 64 * cg + 8 * (lane & 7);
        const bool ok = in_use(tok);
        store16_through(static_cast<uint16_t*>(p.out) + (int64_t)(ok ? tok : 0) * p.N + n, v, __ballot(ok && n < limit));
      }
    } else {
      const int32_t tok = ax.ids[row];
#pragma unroll
      for (int ci = 0; ci < 2; ++ci)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int n = tk.n0 + 64 * cg + 32 * ci + 8 * q + 4 * lgrp;
          int v[4];
          four(acc[ci], q, v);
          if (in_use(tok) && n < limit)
            *reinterpret_cast<v4i*>(static_cast<int32_t*>(p.out) + (int64_t)tok * p.N + n) = v4i{v[0], v[1], v[2], v[3]};
        }
    }
  };

  // ---- start-up: the first step's weights are requested while the token ids are on their way ----
  fill_table(0);
  __syncthreads();
  Task tk = next_task();
  if (tk.e < 0) return;
  Task nx = next_task();
  Task n2 = next_task();
  if (wave < 2)
    fetch_ids(tk, aux[0], wave);
  else if (wave < 4)
    fetch_ids(nx.e >= 0 ? nx : tk, aux[1], wave - 2);
  TaskLoads ld;  // of the task that the loads are in
  setup_weights(tk, ld);
  int next_at = ld.first;  // byte offset of the next step to fetch
  const uint32_t stage0 = lds_address(stages);
  const uint32_t wdst = (uint32_t)uniform((int)(stage0 + wave * 4096)), xdst = (uint32_t)uniform((int)(stage0 + kX0 + wave * 2048));
#pragma unroll
  for (int i = 0; i < 4; ++i) load_to_lds_16(ld.wbase + next_at, ld.woff[i], wdst + i * 1024);
  wait_vmcnt<4>();
  __syncthreads();
  setup_tokens(tk, aux[0], ld);
  fetch_scales(tk, aux[0]);
#pragma unroll
  for (int i = 0; i < 2; ++i) load_to_lds_16(p.a_q + next_at, ld.xoff[i], xdst + i * 1024);
  next_at = next_at + kStepBytes < K ? next_at + kStepBytes : 0;
#pragma unroll
  for (int i = 0; i < 4; ++i) load_to_lds_16(ld.wbase + next_at, ld.woff[i], wdst + kStage + i * 1024);
#pragma unroll
  for (int i = 0; i < 2; ++i) load_to_lds_16(p.a_q + next_at, ld.xoff[i], xdst + kStage + i * 1024);
  next_at = next_at + kStepBytes < K ? next_at + kStepBytes : 0;
  wait_vmcnt<kLoads>();

  int par = 0;                    // aux of the current task; the next ones follow
  int read_at = 0;                // ring offset of the step being multiplied
  int fill_at = kAhead * kStage;  // ... of the step being fetched
  int stores = 0;                 // of the last epilogue, behind the loads of the first two steps
  int units = ld.units, next_units = 0;
  while (true) {
    typename F::Acc acc[2][2];  // [unit][32 weight rows]
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int ci = 0; ci < 2; ++ci)
#pragma unroll
        for (int r = 0; r < F::kRegs; ++r) acc[u][ci][r] = 0;
    TileAux& ax_next = aux[par + 1 < 3 ? par + 1 : par - 2];
    TileAux& ax_n2 = aux[par + 2 < 3 ? par + 2 : par - 1];

    // Steps [s0, s1), during which the loads are those of one task: everything that does not change inside is decided outside.
    // MINE: units that this wavefront multiplies.
    int advance = kStepBytes;
    auto steps = [&](auto mine_tag, auto stream_tag, int s0, int s1) {
      constexpr int MINE = decltype(mine_tag)::value;
      constexpr bool STREAM = decltype(stream_tag)::value;
      for (int s = s0; s < s1; ++s) {
        // everybody's loads of step s have landed, and everybody is done reading the stage that is filled next
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        const char* st = stages + read_at;
        v4i a[4][2], b[4][2];
#pragma unroll
        for (int kk = 0; kk < 4; ++kk) {
          if constexpr (MINE > 0) {
            b[kk][0] = *reinterpret_cast<const v4i*>(st + rd_x[kk]);
            a[kk][0] = *reinterpret_cast<const v4i*>(st + rd_w[kk]);
            a[kk][1] = *reinterpret_cast<const v4i*>(st + rd_w[kk] + kSecondW);
          }
          if constexpr (MINE > 1) b[kk][1] = *reinterpret_cast<const v4i*>(st + rd_x[kk] + kSecondX);
        }
        auto mul = [&](int kk) {
#pragma unroll
          for (int u = 0; u < MINE; ++u)
#pragma unroll
            for (int ci = 0; ci < 2; ++ci) acc[u][ci] = F::mul(a[kk][ci], b[kk][u], acc[u][ci]);
        };
        const int8_t* wsrc = ld.wbase + next_at;
        const int8_t* xsrc = p.a_q + next_at;
        auto weight = [&](int i) {
          if constexpr (STREAM)
            load_to_lds_16_stream(wsrc, ld.woff[i], wdst + fill_at + i * 1024);
          else
            load_to_lds_16(wsrc, ld.woff[i], wdst + fill_at + i * 1024);
        };
        mul(0);
        weight(0);
        weight(1);
        mul(1);
        weight(2);
        weight(3);
        mul(2);
        load_to_lds_16(xsrc, ld.xoff[0], xdst + fill_at);
        load_to_lds_16(xsrc, ld.xoff[1], xdst + fill_at + 1024);
        mul(3);
        next_at = next_at + advance < K ? next_at + advance : 0;
        read_at = read_at + kStage < kStages * kStage ? read_at + kStage : 0;
        fill_at = fill_at + kStage < kStages * kStage ? fill_at + kStage : 0;
        // This wavefront's loads of the next step have landed; behind them are those of the step after, and in a task's first
        // two steps what is counted beside them: the stores of the last epilogue, and the loads issued here.
        if (s >= 2) {
          wait_vmcnt<kLoads>();
        } else if (s == 0) {
          if (stores == 0)
            wait_vmcnt<kLoads>();
          else if (stores == kUnitStores)
            wait_vmcnt<kLoads + kUnitStores>();
          else
            wait_vmcnt<kLoads + 2 * kUnitStores>();
        } else if (nx.e >= 0) {
          // inputs of the next task's epilogue and the ids of the one after it
          fetch_scales(nx, ax_next);
          if (wave < 2) fetch_ids(n2.e >= 0 ? n2 : nx, ax_n2, wave);
          if (it % kTable == 0) fill_table(it);  // (everybody has read the old one; read again behind the next step's barrier)
          if (wave < 2)
            wait_vmcnt<kLoads + 2>();
          else
            wait_vmcnt<kLoads + 1>();
        } else {
          wait_vmcnt<kLoads>();
        }
      }
    };
    for (int part = 0; part < 2; ++part) {
      const int s0 = part == 0 ? 0 : nk - kAhead, s1 = part == 0 ? nk - kAhead : nk;
      if (part == 1 && nx.e >= 0) {
        // the loads enter the next task (its ids were fetched a task ago)
        setup_weights(nx, ld);
        setup_tokens(nx, ax_next, ld);
        next_at = ld.first;
        next_units = ld.units;
      } else if (part == 1) {
        // nothing left: the last step again and again, which keeps the counts uniform
        next_at = (next_at > 0 ? next_at : K) - kStepBytes;
        advance = 0;
      }
      using I0 = std::integral_constant<int, 0>;
      using I1 = std::integral_constant<int, 1>;
      using I2 = std::integral_constant<int, 2>;
      if (ld.stream) {
        if (th + 2 < units)
          steps(I2{}, std::true_type{}, s0, s1);
        else if (th < units)
          steps(I1{}, std::true_type{}, s0, s1);
        else
          steps(I0{}, std::true_type{}, s0, s1);
      } else {
        if (th + 2 < units)
          steps(I2{}, std::false_type{}, s0, s1);
        else if (th < units)
          steps(I1{}, std::false_type{}, s0, s1);
        else
          steps(I0{}, std::false_type{}, s0, s1);
      }
    }
    // everybody is done with the stage of the last step; the next loads into it are behind the barrier of the next step
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    char* staging = stages + (read_at > 0 ? read_at : kStages * kStage) - kStage + wave * 4096;
    stores = 0;
    if (th < units) {
      epilogue(tk, aux[par], acc[0], th * kUnit, staging);
      stores = kUnitStores;
    }
    if (th + 2 < units) {
      epilogue(tk, aux[par], acc[1], (th + 2) * kUnit, staging);
      stores = 2 * kUnitStores;
    }
    if (nx.e < 0) break;
    units = next_units;
    tk = nx;
    nx = n2;
    n2 = next_task();
    par = par + 1 < 3 ? par + 1 : 0;
  }
  wait_vmcnt<0>();
}

template <int MODE>
hipError_t launch_mode(const GemmArgs& a, hipStream_t stream) {
  DeepParams p;
  p.a_q = a.a_q;
  p.a_scale = a.a_scale;
  p.w = a.w;
  p.w_scale = a.w_scale;
  p.row_weight = a.row_weight;
  p.sorted_ids = a.sorted_token_ids;
  p.npp = a.num_tokens_post_padded;
  p.P = (int)a.num_pairs;
  p.row_of = divider(a.row_div);
  p.N = a.n;
  p.K = a.k;
  p.B = a.block_size;
  p.tiles.expert_ids = a.expert_ids;
  p.tiles.E = a.num_experts;
  p.tiles.per_tile = kTok / a.block_size;
  p.tiles.by_per_tile = divider(p.tiles.per_tile);
  p.tiles.even = 0;
  p.tiles.ntiles = MODE == kGateUpSilu ? (a.n / 2 + 127) / 128 : (a.n + kCh - 1) / kCh;
  p.tiles.by_ntiles = divider(p.tiles.ntiles);
  p.tiles.blocks = (int)(a.sorted_cap / a.block_size);
  p.tiles.identity = a.identity ? 1 : 0;
  p.ascend = a.expert_ids_ascend && a.num_experts <= 2 * kThreads ? 1 : 0;
  p.rotate = rotation(a.k, (int64_t)a.num_experts * a.n * a.k, a.num_experts);
  p.out = a.out;
  const dim3 grid((unsigned)(device_cu_count() / kXcds * kXcds));
  hipLaunchKernelGGL((gemm_deep_kernel<MODE>), grid, dim3(kThreads), 0, stream, p);
  return hipGetLastError();
}

}  // namespace

bool gemm_deep_supports(const GemmArgs& a) {
  // per-lane source offsets are 32-bit: one expert's weights and the activation matrix must each
  // span less than 4 GiB
  const int64_t act_rows = (a.num_pairs + a.row_div - 1) / a.row_div;
  if (!((a.block_size == 64 || a.block_size == 128) && a.k % kStepBytes == 0 && a.k >= kMinSteps * kStepBytes && a.n % 16 == 0 &&
        (int64_t)a.n * a.k < (1ll << 32) && act_rows * a.k < (1ll << 32)))
    return false;
  // The tile list lives in LDS.  A run of equal expert ids of L blocks makes ceil(L / blocks per
  // tile) tiles; moe_align's ids ascend, so there is one run per expert.  Ids of unknown order could
  // make every block a tile of its own.  While the list is built the block ids sit in the stages.
  const int64_t blocks = (a.sorted_cap + a.block_size - 1) / a.block_size;
  const int per_tile = kTok / a.block_size;
  const int64_t tiles = a.expert_ids_ascend ? (blocks + per_tile - 1) / per_tile + a.num_experts : blocks;
  return tiles <= kMaxTiles && blocks <= (int64_t)(kStages * kStage / sizeof(int)) && blocks <= 65535;
}

hipError_t launch_gemm_deep(const GemmArgs& a, hipStream_t stream) {
  switch (a.mode) {
    case kGateUpSilu: return launch_mode<kGateUpSilu>(a, stream);
    case kDown: return launch_mode<kDown>(a, stream);
    case kAccI32: return launch_mode<kAccI32>(a, stream);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace moe_i8
