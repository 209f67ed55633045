// Grouped int8 GEMM for gfx950, wide tiles (prefill: from about a hundred routed rows per expert up).
//
// One persistent workgroup of eight wavefronts per compute unit walks tiles of up to 256 token rows (consecutive
// moe_align blocks of one expert) x 256 weight rows; the reduction runs in steps of 128 bytes through two 64 KB LDS
// stages filled by global -> LDS loads.  The MFMA is used "transposed" (A operand = weight rows), so a lane ends up
// with 4 consecutive channels of a token.  What bounds it at this size is the power the chip may draw: with random
// operands the clock falls from 2.4 to 1.8-2.0 GHz, so both cycles and energy per step count.
//
//  * v_mfma_i32_16x16x64_i8 sustains 4.2e15 operations per second on random operands from registers, 32x32x32 3.5e15.
//    A wavefront multiplies 64 weight rows x 128 token rows and holds a step's weight operands in registers while the
//    token operands of the two halves pass, which keeps the LDS reads at 24 KB per wavefront and step.
//  * The wavefronts form two groups, one wavefront of each per SIMD, half a turn apart: while one group issues nothing
//    but MFMAs (32 of them), the other reads its next operands and sends the next loads.  A step is four turns; every
//    turn ends with a barrier.  2048 cycles of MFMAs per step take 2630; in lock step they took 3100 and more.
//    (The barrier must not come before the last MFMA of a turn: with four left behind it, +700 cycles a step, because
//    the other turn starts late.)
//  * Weight rows and token rows 0..127 of a stage are free once both groups have read them, in the middle of a step,
//    and are filled again at once: 1 to 1.5 steps, 64 to 112 KB, of loads in flight.  One stage in flight gave 1.6 us a
//    step from loads alone where weights come from memory, two give 1.2.
//  * A tile's work follows its rows in units of 32: unit i belongs to half i / 4 and group i % 2, so that both
//    groups, and every SIMD, get an equal share of a partly filled tile.
//  * Everything a task needs is at hand when it starts: the tasks are looked up 64 at a time, token ids travel two tasks
//    ahead and scales one, all global -> LDS; results are transposed through 2 KB per wavefront that no load uses.  With
//    dependent reads and divisions at every task a step costs nothing more, but a task 4 us.
//
// Layer us, before -> after (one stage ahead, 32x32x32, all wavefronts in step): 128 experts of 2048 x 768 at 8192 tokens
// 526 -> 478, 256 experts of 7168 x 2048 at 16384 tokens 6874 -> 6274, gated MLP of 4096 x 1408 at 4096 rows 97.7 -> 87.9.
#include <type_traits>

#include "lds_loads.hpp"
#include "tile_list.hpp"

namespace moe_i8 {
namespace {

constexpr int kThreads = kTileThreads;
constexpr int kWaves = kThreads / kWave;
constexpr int kTok = 256;   // token rows per tile
constexpr int kCh = 256;    // weight rows per tile
constexpr int kMaxTiles = 6144;  // of a launch
constexpr int kX0 = kCh * kStepBytes;              // token rows 0..127 of a stage, behind the weight rows
constexpr int kX1 = kX0 + kTok / 2 * kStepBytes;   // token rows 128..255
constexpr int kStage = kX1 + kTok / 2 * kStepBytes;
constexpr int kTable = 64;       // tasks of a workgroup looked up at a time
constexpr int kStaging = 2048;  // bytes per wavefront for the transposition of results

struct WideParams {
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
  void* out;
};

struct Task {
  int e;      // expert; -1 = no more work
  int nt;     // channel tile
  int slot0;  // first slot of the tile in sorted_ids
  int rows;   // slots of the tile
};

struct TaskLoads {
  const int8_t* wbase;  // weights of the task's expert (wave-uniform)
  uint32_t woff[4];     // per lane: byte offset of its chunk of weight row i from wbase
  uint32_t xoff[2][2];  // per lane: byte offset of its chunk of token row 128 * half + i from a_q
  int units;            // 32-row units up to the last row in use
};

__device__ __forceinline__ void wait_lds() { __builtin_amdgcn_s_waitcnt(0xc07f); }  // lgkmcnt(0)

// 16 bytes per lane from base + offset into LDS at lds_addr + kAt + 16 * lane; base and lds_addr are wave-uniform
template <int kAt, bool NT>
__device__ __forceinline__ void stage_load(uint64_t base, uint32_t offset, uint32_t lds_addr) {
  lds_addr = (uint32_t)__builtin_amdgcn_readfirstlane((int)lds_addr);
  base = uniform_address(reinterpret_cast<const void*>(base));
  if constexpr (NT)
    asm volatile("s_add_u32 m0, %0, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2 nt"
                 :: "s"(lds_addr), "v"(offset), "s"(base), "n"(kAt) : "memory", "m0", "scc");
  else
    asm volatile("s_add_u32 m0, %0, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
                 :: "s"(lds_addr), "v"(offset), "s"(base), "n"(kAt) : "memory", "m0", "scc");
}

// f(0), f(1), ..., f(N - 1) with compile-time arguments
template <int N, int I = 0, class F>
__device__ __forceinline__ void unroll(F&& f) {
  if constexpr (I < N) {
    f(std::integral_constant<int, I>{});
    unroll<N, I + 1>(f);
  }
}

__device__ __forceinline__ void barrier() {
  __builtin_amdgcn_sched_barrier(0);
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_sched_barrier(0);
}

// KEEP: results are stored without the non-temporal hint where weight rows are shared.  (A template argument: of two
// stores behind a run-time flag the compiler makes one, without the hint.)
template <int MODE, bool KEEP>
__global__ __launch_bounds__(kThreads, 1) void gemm_wide_kernel(WideParams p) {
  __shared__ __align__(16) char stages[2 * kStage];
  __shared__ __align__(16) char staging[kWaves * kStaging];
  __shared__ __align__(16) int32_t ids[3][kTok];                          // slots of the current, the next and the task after it
  __shared__ __align__(16) float a_scales[2][kTok], row_weights[2][kTok], w_scales[2][kCh];
  __shared__ TileList<kMaxTiles> list;
  __shared__ uint2 table[kTable];                           // tasks it .. of this workgroup: block | blocks << 16, task_word

  const int t = threadIdx.x;
  const int lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int group = wave >> 2, cpart = wave & 3;
  const int col = lane & 15, quad = lane >> 4;
  const int nk = p.K / kStepBytes;
  const int inter = p.N / 2;

  const int xcd = blockIdx.x % kXcds;
  TileRange range = p.ascend ? build_ascending(p.tiles, xcd, reinterpret_cast<int*>(stages), list)
                             : build_any_order(p.tiles, __builtin_amdgcn_readfirstlane(*p.npp) / p.B, xcd, reinterpret_cast<int*>(stages), list);
  // (said to be wave-uniform: everything that follows from them then stays in scalar registers)
  range.lo = __builtin_amdgcn_readfirstlane(range.lo);
  range.hi = __builtin_amdgcn_readfirstlane(range.hi);
  range.tiles = __builtin_amdgcn_readfirstlane(range.tiles);
  const int total = range.tiles * p.tiles.ntiles;
  const int per_xcd = __builtin_amdgcn_readfirstlane((total + kXcds - 1) / kXcds);
  const int my_tasks = total - xcd * per_xcd < per_xcd ? max(total - xcd * per_xcd, 0) : per_xcd;  // of the XCD
  const int stride = gridDim.x / kXcds;
  int it = 0;  // tasks handed out

  // Looks up tasks n0 .. n0 + kTable - 1 of this workgroup.
  auto fill_table = [&](int n0) {
    if (t >= kTable) return;
    const TaskPiece tp = piece_at(blockIdx.x / kXcds + (n0 + t) * stride, my_tasks, stride);
    uint2 d = make_uint2(0u, kNoTask);
    if (tp.task >= 0) {
      const uint2 whole = look_up_task(p.tiles, list, range, xcd * per_xcd + tp.task);
      // a piece is a part of the tile's blocks
      const int blocks = (int)(whole.x >> 16) & 15, from = tp.piece * blocks / tp.pieces, to = (tp.piece + 1) * blocks / tp.pieces;
      if (tp.pieces == 1 || to > from) d = make_uint2(((whole.x & 0xffffu) + from) | (uint32_t)(to - from) << 16, whole.y);
    }
    table[t] = d;
  };
  auto next_task = [&]() {
    const uint2 d = table[it % kTable];
    const uint32_t d0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)d.x);
    const uint32_t d1 = (uint32_t)__builtin_amdgcn_readfirstlane((int)d.y);
    Task tk;
    tk.slot0 = (int)(d0 & 0xffffu) * p.B;
    tk.rows = (int)(d0 >> 16) * p.B;
    tk.nt = task_channel_tile(d1);
    tk.e = task_expert(d1);
    if (tk.e >= 0) ++it;
    return tk;
  };
  auto fetch_ids = [&](const Task& tk, int buf) {
    if (tk.e >= 0 && wave < 4) {
      const int row = wave * 64 + lane;
      load_to_lds_4(p.sorted_ids + tk.slot0 + (row < tk.rows ? row : 0), lds_address(&ids[buf][wave * 64]));
    }
  };
  // Where the task's rows are.  Lane fills LDS slot (lane & 7) of row base + 8 * i + (lane >> 3) of a wavefront's load i: it
  // fetches chunk (lane & 7) ^ swizzle.
  auto chunk_of = [&](int i) { return ((lane & 7) ^ (lane >> 3) ^ (i & 1)) * 16; };
  auto setup_weights = [&](const Task& tk, TaskLoads& ld) {
    ld.wbase = p.w + (int64_t)tk.e * p.N * p.K;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int row = 32 * wave + 8 * i + (lane >> 3);
      int n;
      if constexpr (MODE == kGateUpSilu) {
        const int ch = tk.nt * 128 + (row & 127);
        n = (ch < inter ? ch : inter - 1) + (row >= 128 ? inter : 0);
      } else {
        const int ch = tk.nt * kCh + row;
        n = ch < p.N ? ch : p.N - 1;
      }
      ld.woff[i] = (uint32_t)n * (uint32_t)p.K + chunk_of(i);
    }
  };
  // ... (its ids have landed)
  auto setup_tokens = [&](const Task& tk, int buf, TaskLoads& ld) {
    // lane l looks at rows 4l .. 4l + 3
    const int4 four = *reinterpret_cast<const int4*>(&ids[buf][4 * lane]);
    auto in_use = [&](int id) { return (uint32_t)id < (uint32_t)p.P; };
    const uint64_t used = __ballot(4 * lane < tk.rows && (in_use(four.x) || in_use(four.y) || in_use(four.z) || in_use(four.w)));
    ld.units = __builtin_amdgcn_readfirstlane(used ? (63 - __builtin_clzll(used)) / 8 + 1 : 0);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      // rows behind the last one in use fetch the tile's first row again
      int trow = (i >> 1) * 128 + 16 * wave + 8 * (i & 1) + (lane >> 3);
      if (trow >= ld.units * 32) trow = 0;
      const int32_t id = ids[buf][trow];
      ld.xoff[i >> 1][i & 1] = (in_use(id) ? p.row_of(id) : 0u) * (uint32_t)p.K + chunk_of(i);
    }
  };
  // inputs of the task's epilogue
  auto fetch_aux = [&](const Task& tk, int buf, int aux) {
    if constexpr (MODE != kAccI32) {
      const int row = (wave & 3) * 64 + lane;
      int32_t id = ids[buf][row < tk.rows ? row : 0];
      if (id < 0 || id >= p.P) id = 0;
      if (wave < 4) {
        load_to_lds_4(p.a_scale + p.row_of(id), lds_address(&a_scales[aux][wave * 64]));
      } else {
        if (MODE == kDown && p.row_weight) load_to_lds_4(p.row_weight + id, lds_address(&row_weights[aux][(wave & 3) * 64]));
        int n;
        if constexpr (MODE == kGateUpSilu) {
          const int ch = tk.nt * 128 + (row & 127);
          n = (ch < inter ? ch : inter - 1) + (row >= 128 ? inter : 0);
        } else {
          const int ch = tk.nt * kCh + row;
          n = ch < p.N ? ch : p.N - 1;
        }
        load_to_lds_4(p.w_scale + (int64_t)tk.e * p.N + n, lds_address(&w_scales[aux][(wave & 3) * 64]));
      }
    }
  };

  // (A last round in pieces makes up to four workgroups read one expert's rows as well, and the hint stays on there: the rounds
  // before it need it.  gate_up + down us of experts with 256 rows each, hint as it is / off for a range with such a round / last
  // round whole: 48 of 4096 x 1408 173 + 93 / 194 + 92 / 182 + 92, 136 of 2048 x 512 99 + 75 / 107 + 77 / 104 + 77, 24 of 4096 x
  // 1408 105 + 53.8 / 112 + 53.8 / 117 + 56; without a full round before it, 8 of 4096 x 1408 43.7 + 24.8 / 44.9 + 24.9 / 50.5 + 26.8,
  // 4 of them 39.9 + 22.0 / 39.4 + 20.2 / 49.6 + 25.0.)
  bool shared_local = false;
  for (int g = t; g < range.hi - range.lo; g += kThreads) shared_local |= (list.desc[g] >> 20) != (1u << 4);  // rank 0, group size 1
  const bool weights_shared = __builtin_amdgcn_readfirstlane(__syncthreads_or(shared_local ? 1 : 0)) != 0;

  const uint32_t stage0 = lds_address(stages);
  const int swz = swizzle_of_row(col);
  // operand reads: lane feeds row `col` of a 16-row tile, chunk 4 * kk + quad
  const int rd0 = col * kStepBytes + ((quad ^ swz) * 16), rd1 = col * kStepBytes + (((4 + quad) ^ swz) * 16);
  // first LDS weight row of the wavefront's 16-row tiles ci
  auto w_row = [&](int ci) { return MODE == kGateUpSilu ? (ci >> 1) * 128 + cpart * 32 + (ci & 1) * 16 : cpart * 64 + ci * 16; };
  char* my_staging = staging + wave * kStaging;

  auto run = [&](auto nt_tag) {
    constexpr bool NT = decltype(nt_tag)::value;
    // load i of the weight rows and token rows 0..127 of a step (six per wavefront), of token rows 128..255 (two)
    auto load_w = [&](auto i_tag, uint64_t wp, uint64_t xp, const uint32_t (&woff)[4], const uint32_t (&xoff)[2], uint32_t at_w, uint32_t at_x) {
      constexpr int i = decltype(i_tag)::value;
      if constexpr (i < 4)
        stage_load<i * 1024, NT>(wp, woff[i], at_w);
      else
        stage_load<kX0 + (i - 4) * 1024, false>(xp, xoff[i - 4], at_x);
    };
    auto load_x1 = [&](auto i_tag, uint64_t xp, const uint32_t (&xoff)[2], uint32_t at_x) {
      constexpr int i = decltype(i_tag)::value;
      stage_load<kX1 + i * 1024, false>(xp, xoff[i], at_x);
    };
    auto issue_w = [&](uint64_t wp, uint64_t xp, const uint32_t (&woff)[4], const uint32_t (&xoff)[2], uint32_t at_w, uint32_t at_x) {
      unroll<6>([&](auto i) { load_w(i, wp, xp, woff, xoff, at_w, at_x); });
    };
    auto issue_x1 = [&](uint64_t xp, const uint32_t (&xoff)[2], uint32_t at_x) {
      unroll<2>([&](auto i) { load_x1(i, xp, xoff, at_x); });
    };

    fill_table(0);
    __syncthreads();
    Task tk = next_task();
    if (tk.e < 0) return;
    Task nx = next_task();
    fetch_ids(tk, 0);
    fetch_ids(nx, 1);
    TaskLoads nld;  // of the next task; without one, of this one
    setup_weights(tk, nld);
    // Load cursors: where the next weight-and-first-half and the next second-half loads come from.  They run ahead of
    // the multiplication, into the next task where there is one, else over this task's first steps again.
    const uint64_t aq = uniform_address(p.a_q);
    uint64_t wp = uniform_address(nld.wbase), xp = aq, x1p = aq;
    uint32_t woff[4], x0off[2] = {0, 0}, x1off[2] = {0, 0};
#pragma unroll
    for (int i = 0; i < 4; ++i) woff[i] = nld.woff[i];
    const uint32_t at_w0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)(stage0 + wave * 4096));
    const uint32_t at_x0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)(stage0 + wave * 2048));
    // The first step's weights are requested while the token ids are on their way.
    unroll<4>([&](auto i) { load_w(i, wp, xp, woff, x0off, at_w0, at_x0); });
    wait_vmcnt<4>();
    __syncthreads();
    setup_tokens(tk, 0, nld);
    int units = nld.units;
#pragma unroll
    for (int i = 0; i < 2; ++i) x0off[i] = nld.xoff[0][i], x1off[i] = nld.xoff[1][i];
    fetch_aux(tk, 0, 0);
    load_w(std::integral_constant<int, 4>{}, wp, xp, woff, x0off, at_w0, at_x0);
    load_w(std::integral_constant<int, 5>{}, wp, xp, woff, x0off, at_w0, at_x0);
    issue_x1(x1p, x1off, at_x0);
    issue_w(wp + kStepBytes, xp + kStepBytes, woff, x0off, at_w0 + kStage, at_x0 + kStage);
    wp += 2 * kStepBytes, xp += 2 * kStepBytes, x1p += kStepBytes;
    wait_vmcnt<8>();  // all but the second half of step 0 and step 1
    barrier();
    bool fresh = true;  // the first step's waits are as in any other step; a later task's first step has landed as a whole
    int buf = 0, aux = 0, slot = 0;

    while (true) {
      const bool has_next = nx.e >= 0;
      // 32-row units of this wavefront in the two halves
      auto pairs = [&](int half) {
        const int n = (units - half * 4 - group + 1) >> 1;
        return n < 0 ? 0 : n > 2 ? 2 : n;
      };
      const int n0 = pairs(0), n1 = pairs(1);
      Task after;
      after.e = -1;
      v4i acc[4][8];
#pragma unroll
      for (int ci = 0; ci < 4; ++ci)
#pragma unroll
        for (int ti = 0; ti < 8; ++ti) acc[ci][ti] = v4i{0, 0, 0, 0};
      v4i wf[4][2], xf[4][2];
      auto read_x = [&](const char* half) {
#pragma unroll
        for (int ti = 0; ti < 4; ++ti) {
          const char* r = half + ((ti >> 1) * 64 + group * 32 + (ti & 1) * 16) * kStepBytes;
          xf[ti][0] = *reinterpret_cast<const v4i*>(r + rd0);
          xf[ti][1] = *reinterpret_cast<const v4i*>(r + rd1);
        }
      };
      // the 16 MFMAs of unit j of a half (16-row token tiles 2j, 2j + 1)
      auto multiply_unit = [&](auto half_tag, auto unit_tag) {
        constexpr int H = decltype(half_tag)::value, kUnit = decltype(unit_tag)::value;
        unroll<16>([&](auto i) {
          constexpr int m = decltype(i)::value, kk = m >> 3, ci = (m >> 1) & 3, ti = 2 * kUnit + (m & 1);
          acc[ci][4 * H + ti] = __builtin_amdgcn_mfma_i32_16x16x64_i8(wf[ci][kk], xf[ti][kk], acc[ci][4 * H + ti], 0, 0, 0);
          __builtin_amdgcn_sched_barrier(0);
        });
      };
      auto multiply = [&](auto half_tag, int n, int waits, bool meet) {
        __builtin_amdgcn_s_setprio(1);
        if (n > 0) multiply_unit(half_tag, std::integral_constant<int, 0>{});
        if (n > 1) multiply_unit(half_tag, std::integral_constant<int, 1>{});
        if (waits == 0) wait_vmcnt<8>();
        if (meet) barrier();
        __builtin_amdgcn_s_setprio(0);
      };

      if (group == 1) barrier();
      for (int s = 0; s < nk; ++s) {
        const char* st = stages + slot * kStage;
        const int waits = s > 0 || fresh ? group : 2;  // which group has loads to wait for
        // ---- read 0 ----
#pragma unroll
        for (int ci = 0; ci < 4; ++ci) {
          wf[ci][0] = *reinterpret_cast<const v4i*>(st + w_row(ci) * kStepBytes + rd0);
          wf[ci][1] = *reinterpret_cast<const v4i*>(st + w_row(ci) * kStepBytes + rd1);
        }
        read_x(st + kX0);
        if (s == nk - 1) {
#pragma unroll
          for (int i = 0; i < 2; ++i) x1off[i] = nld.xoff[1][i];
          x1p = aq;
        }
        issue_x1(x1p, x1off, at_x0 + (slot ^ 1) * kStage);
        x1p += kStepBytes;
        if (waits == 1) wait_vmcnt<8>();
        wait_lds();
        barrier();
        multiply(std::integral_constant<int, 0>{}, n0, waits, true);
        // ---- read 1 ----
        if (n1 > 0) read_x(st + kX1);
        if (s == 0 && has_next) {
          setup_weights(nx, nld);
          setup_tokens(nx, buf == 2 ? 0 : buf + 1, nld);
          fetch_aux(nx, buf == 2 ? 0 : buf + 1, aux ^ 1);
          after = next_task();
          fetch_ids(after, buf == 0 ? 2 : buf - 1);
        }
        if (s == nk - 2) {
#pragma unroll
          for (int i = 0; i < 4; ++i) woff[i] = nld.woff[i];
#pragma unroll
          for (int i = 0; i < 2; ++i) x0off[i] = nld.xoff[0][i];
          wp = uniform_address(nld.wbase);
          xp = aq;
        }
        issue_w(wp, xp, woff, x0off, at_w0 + slot * kStage, at_x0 + slot * kStage);
        wp += kStepBytes;
        xp += kStepBytes;
        if (waits == 1) wait_vmcnt<8>();
        wait_lds();
        barrier();
        multiply(std::integral_constant<int, 1>{}, n1, waits, group == 0 || s + 1 < nk);
        slot ^= 1;
      }

      // ---- epilogue ----
      const int32_t* my_ids = ids[buf];
      const float* as = a_scales[aux];
      const float* rw = row_weights[aux];
      const float* ws = w_scales[aux];
      // lane's 16 bytes of result row `id` behind `to`, where the row is a slot in use
      auto store = [&](uint64_t to, uint32_t row_bytes, int32_t id, uint32_t ids_below, const uint4& v) {
        const uint64_t lanes = __ballot((uint32_t)id < ids_below);
        store16_lanes<!(KEEP && !NT)>(reinterpret_cast<void*>(to + (uint64_t)(uint32_t)id * row_bytes), v, lanes);
      };
      fresh = false;
      if constexpr (MODE == kAccI32) {
#pragma unroll
        for (int ti = 0; ti < 8; ++ti) {
          const int row = (ti >> 2) * 128 + ((ti >> 1) & 1) * 64 + group * 32 + (ti & 1) * 16 + col;
          const int32_t id = my_ids[row];
          if (row >= units * 32 || id < 0 || id >= p.P) continue;
          int32_t* out = static_cast<int32_t*>(p.out) + (int64_t)id * p.N;
#pragma unroll
          for (int ci = 0; ci < 4; ++ci) {
            const int n = tk.nt * kCh + cpart * 64 + ci * 16 + 4 * quad;
            if (n < p.N) *reinterpret_cast<v4i*>(out + n) = acc[ci][ti];
          }
        }
      } else {
        // All that the results need besides the sums is requested at once, the stores are issued without branches, and a piece is
        // read back from its staging while the next one is computed.  The arithmetic (4.5 instructions of 4 cycles a value, 23 with
        // SiLU, for 128 or 64 values a lane and two wavefronts a SIMD) is what remains; as a chain of such reads and branches
        // an epilogue took a third longer: layers of 128 experts of 2048 x 768 at 4000 / 8192 / 12000 tokens 287 / 465 / 633 us,
        // now 281 / 461 / 615, of 4096 x 1408 at 4096 940 / 920.
        constexpr bool kSilu = MODE == kGateUpSilu;
        float4 wsc[4];
        if constexpr (kSilu) {
#pragma unroll
          for (int c = 0; c < 4; ++c) wsc[c] = *reinterpret_cast<const float4*>(ws + (c >> 1) * 128 + cpart * 32 + (c & 1) * 16 + 4 * quad);
        } else {
#pragma unroll
          for (int c = 0; c < 4; ++c) wsc[c] = *reinterpret_cast<const float4*>(ws + cpart * 64 + c * 16 + 4 * quad);
        }
        const int width = kSilu ? inter : p.N;
        const int n = kSilu ? tk.nt * 128 + cpart * 32 + (lane & 3) * 8 : tk.nt * kCh + cpart * 64 + (lane & 7) * 8;
        const uint32_t ids_below = n < width ? (uint32_t)p.P : 0u;
        const uint64_t to = reinterpret_cast<uint64_t>(static_cast<uint16_t*>(p.out) + n);
        float sc[8], rwt[8];
        int32_t id[4][kSilu ? 2 : 4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const int row0 = (u >> 1) * 128 + (u & 1) * 64 + group * 32;
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            sc[2 * u + h] = as[row0 + h * 16 + col];
            if constexpr (!kSilu) rwt[2 * u + h] = rw[row0 + h * 16 + col];
          }
#pragma unroll
          for (int r = 0; r < (kSilu ? 2 : 4); ++r) id[u][r] = my_ids[row0 + r * (kSilu ? 16 : 8) + (lane >> (kSilu ? 2 : 3))];
        }
        if constexpr (!kSilu)
          if (!p.row_weight)
#pragma unroll
            for (int i = 0; i < 8; ++i) rwt[i] = 1.0f;
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          if ((u >> 1) * 128 + (u & 1) * 64 + group * 32 >= units * 32) continue;
          if constexpr (kSilu) {
#pragma unroll
            for (int h = 0; h < 2; ++h) {
              const int ti = u * 2 + h, row = h * 16 + col;
#pragma unroll
              for (int c = 0; c < 2; ++c) {
                const int g[4] = {acc[c][ti][0], acc[c][ti][1], acc[c][ti][2], acc[c][ti][3]};
                const int up[4] = {acc[c + 2][ti][0], acc[c + 2][ti][1], acc[c + 2][ti][2], acc[c + 2][ti][3]};
                *reinterpret_cast<uint2*>(my_staging + row * 64 + (((c * 2 + (quad >> 1)) ^ ((row >> 2) & 3)) * 16) + (quad & 1) * 8) =
                    silu_mul_epilogue4(g, up, sc[ti], wsc[c], wsc[c + 2]);
              }
            }
            uint4 v[2];
#pragma unroll
            for (int r = 0; r < 2; ++r) {
              const int row = r * 16 + (lane >> 2), chunk = lane & 3;
              v[r] = *reinterpret_cast<const uint4*>(my_staging + row * 64 + ((chunk ^ ((row >> 2) & 3)) * 16));
            }
#pragma unroll
            for (int r = 0; r < 2; ++r) store(to, (uint32_t)width * 2, id[u][r], ids_below, v[r]);
          } else {
            uint4 v[4];
#pragma unroll
            for (int h = 0; h < 2; ++h) {
              const int ti = u * 2 + h;
#pragma unroll
              for (int ci = 0; ci < 4; ++ci) {
                const int q[4] = {acc[ci][ti][0], acc[ci][ti][1], acc[ci][ti][2], acc[ci][ti][3]};
                *reinterpret_cast<uint2*>(my_staging + col * 128 + (((ci * 2 + (quad >> 1)) ^ (col & 7)) * 16) + (quad & 1) * 8) =
                    down_epilogue4(q, sc[ti], wsc[ci], rwt[ti]);
              }
#pragma unroll
              for (int r = 0; r < 2; ++r) {
                const int row = r * 8 + (lane >> 3), chunk = lane & 7;
                v[2 * h + r] = *reinterpret_cast<const uint4*>(my_staging + row * 128 + ((chunk ^ (row & 7)) * 16));
              }
            }
#pragma unroll
            for (int r = 0; r < 4; ++r) store(to, (uint32_t)width * 2, id[u][r], ids_below, v[r]);
          }
        }
      }
      // The next task's first loads have landed; behind them are this task's stores, two or four for each of its units of this
      // wavefront.  (Waited for here, not in front of the results: layers of 128 experts of 2048 x 768 at 12000 tokens 661 / 640
      // us, of 4096 x 1408 at 8192 1593 / 1568, of 27 layers 1.0 % on average.)
      constexpr int kUnitStores = MODE == kGateUpSilu ? 2 : MODE == kDown ? 4 : 0;
      wait_groups<kUnitStores, kUnitStores ? 4 : 0>(n0 + n1);
      barrier();
      if (!has_next) break;
      if (it % kTable == 0) fill_table(it);  // (read again several barriers from here)
      tk = nx;
      nx = after;
      units = nld.units;
      buf = buf == 2 ? 0 : buf + 1;
      aux ^= 1;
    }
    wait_vmcnt<0>();
  };
  if (weights_shared)
    run(std::false_type{});
  else
    run(std::true_type{});
}

template <int MODE>
hipError_t launch_mode(const GemmArgs& a, hipStream_t stream) {
  WideParams p;
  p.a_q = a.a_q;
  p.a_scale = a.a_scale;
  p.w = a.w;
  p.w_scale = a.w_scale;
  p.row_weight = a.row_weight;
  p.sorted_ids = a.sorted_token_ids;
  p.npp = a.num_tokens_post_padded;
  p.P = (int)a.num_pairs;
  p.row_of = divider(a.row_div);
  p.tiles.expert_ids = a.expert_ids;
  p.tiles.E = a.num_experts;
  p.N = a.n;
  p.K = a.k;
  p.B = a.block_size;
  p.tiles.per_tile = kTok / a.block_size;
  // Nine blocks as 3 + 3 + 3 instead of 4 + 4 + 1: a step of one block costs far more than a quarter of a full one (its weight
  // rows are the same, and it runs ahead of the others, so that they come from memory twice: 757 MB instead of 419 for experts of
  // 264 rows).  Layer us, full tiles and a rest / even ones.  Reductions of 2048 and more: 256 experts of 7168 x 2048 at 8192 / 8800 /
  // 12000 tokens 3768 / 3601, 4458 / 4099, 5018 / 4794 (its down GEMM alone), at 16384 the same; 128 of 2048 x 768 at 4300 / 5000 / 8192
  // / 9000 320 / 315, 356 / 345, 481 / 475, 523 / 520; 64 of 2048 x 1408 at 3000 293 / 281; 256 of 2048 x 512 at 9000 506 / 480.  Below,
  // where a task is mostly its epilogue, nothing or a loss: down GEMMs of 768 and 1408 +-1 %, 32 experts of 1024 x 512, Zipf
  // routing, at 1500 / 5000 56.6 / 58.2, 97.2 / 99.3.
  p.tiles.even = a.k >= 2048;
  p.tiles.ntiles = MODE == kGateUpSilu ? (a.n / 2 + 127) / 128 : (a.n + kCh - 1) / kCh;
  p.tiles.by_ntiles = divider(p.tiles.ntiles);
  p.tiles.by_per_tile = divider(p.tiles.per_tile);
  p.tiles.blocks = (int)(a.sorted_cap / a.block_size);
  p.tiles.identity = a.identity ? 1 : 0;
  p.ascend = a.expert_ids_ascend && a.num_experts <= 2 * kThreads ? 1 : 0;
  // The next launch of a layer reads the results back from the last-level cache where they about fit it and the weights do
  // not sweep it.  Layer us with / without the hint: 128 experts of 2048 x 768 at 8192 tokens 488 / 480, of 4096 x 1536 at
  // 4000 881 / 865; the other side of the line: 256 experts of 7168 x 2048 at 8192 tokens 3780 / 3813, a gated MLP of 4096 x
  // 1408 at 4096 rows, whose weights stay cached, 88.3 / 89.7.
  const bool keep = MODE != kAccI32 && a.num_experts > 1 && (int64_t)a.num_experts * a.n * a.k < (2048ll << 20) &&
                    a.num_pairs * (MODE == kGateUpSilu ? a.n / 2 : a.n) * 2 < (600ll << 20);
  p.out = a.out;
  const dim3 grid((unsigned)(device_cu_count() / kXcds * kXcds));
  if (keep)
    hipLaunchKernelGGL((gemm_wide_kernel<MODE, true>), grid, dim3(kThreads), 0, stream, p);
  else
    hipLaunchKernelGGL((gemm_wide_kernel<MODE, false>), grid, dim3(kThreads), 0, stream, p);
  return hipGetLastError();
}

}  // namespace

bool gemm_wide_supports(const GemmArgs& a) {
  // per-lane source offsets are 32-bit: one expert's weights and the activation matrix must each span less than 4 GiB
  const int64_t act_rows = (a.num_pairs + a.row_div - 1) / a.row_div;
  if (!((a.block_size == 64 || a.block_size == 128) && a.k % kStepBytes == 0 && a.k >= 2 * kStepBytes && a.n % 16 == 0 &&
        (int64_t)a.n * a.k < (1ll << 32) && act_rows * a.k < (1ll << 32)))
    return false;
  // The tile list lives in LDS.  A run of equal expert ids of L blocks makes ceil(L / blocks per tile) tiles;
  // moe_align's ids ascend, so there is one run per expert.  Ids of unknown order could make every block a tile
  // of its own.  While the list is built the block ids sit in the stages.
  const int64_t blocks = (a.sorted_cap + a.block_size - 1) / a.block_size;
  const int per_tile = kTok / a.block_size;
  const int64_t tiles = a.expert_ids_ascend ? (blocks + per_tile - 1) / per_tile + a.num_experts : blocks;
  return tiles <= kMaxTiles && blocks <= (int64_t)(2 * kStage / sizeof(int)) && blocks <= 65535;
}

hipError_t launch_gemm_wide(const GemmArgs& a, hipStream_t stream) {
  switch (a.mode) {
    case kGateUpSilu: return launch_mode<kGateUpSilu>(a, stream);
    case kDown: return launch_mode<kDown>(a, stream);
    case kAccI32: return launch_mode<kAccI32>(a, stream);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace moe_i8
