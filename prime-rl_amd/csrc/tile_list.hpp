// The list of a launch's tiles, derived inside the kernels with LDS-staged tiles from expert_ids (block -> expert).
//
// A tile is a run of moe_align blocks of one expert.  Every workgroup builds the part of the list that the workgroups of
// its XCD look at: tasks (tile, channel tile) are split into 8 contiguous ranges, one per XCD (workgroup id % 8), so that
// workgroups that run side by side share token rows and expert weights in that XCD's L2.
#pragma once

#include "common.hpp"

namespace moe_i8 {

constexpr int kTileThreads = 512;  // of a workgroup
constexpr int kXcds = 8;
constexpr int kGroupTiles = 8;  // token tiles of one expert whose tasks are interleaved per channel tile

// id / div for 0 <= id < 2^31 as a multiplication: (id * magic) >> (32 + shift), div > 1 (a reciprocal of 31 + l
// fraction bits, rounded up, 2^(l-1) < row_div <= 2^l)
struct Divider {
  int div;
  uint32_t magic;
  int shift;
  __device__ __forceinline__ uint32_t operator()(int32_t id) const {
    return div == 1 ? (uint32_t)id : __umulhi((uint32_t)id, magic) >> shift;
  }
};
inline Divider divider(int div) {
  int l = 0;
  while ((1ll << l) < div) ++l;
  return Divider{div, div > 1 ? (uint32_t)(((uint64_t)1 << (31 + l)) / (uint64_t)div + 1) : 0, l - 1};
}

struct TileListArgs {
  const int32_t* expert_ids;
  int E;
  int per_tile;  // most blocks of a tile
  Divider by_per_tile;
  int even;      // an expert's blocks are dealt evenly to its tiles, instead of full tiles and a rest
  int ntiles;    // channel tiles
  Divider by_ntiles;
  int blocks;    // entries of expert_ids, used or not
  int identity;  // one expert owns all of them
};

// MAX: most tiles of a launch
template <int MAX>
struct TileList {
  static constexpr int kMaxTiles = MAX;
  static constexpr int kMaxLocal = MAX / kXcds + 2 + 2 * kGroupTiles;  // ... that one XCD's workgroups look at
  uint32_t desc[kMaxLocal];    // first block | blocks << 16 | rank in group << 20 | group size << 24
  uint16_t expert[kMaxLocal];  // 0xffff: ids outside [0, E)
  int wave_part[kTileThreads / kWave];
};

struct TileRange {
  int lo, hi;  // tiles [lo, hi) of the launch are in the list, tile t at t - lo
  int tiles;   // of the launch
};

__device__ __forceinline__ int wave_scan_max(int v) {
#pragma unroll
  for (int d = 1; d < kWave; d <<= 1) {
    const int n = __shfl_up(v, d);
    if (lane_id() >= d) v = n > v ? n : v;
  }
  return v;
}

// The tiles that the workgroups of one XCD look at: those of its range of tasks, and the rest of their groups.
template <int MAX>
__device__ __forceinline__ TileRange tile_range_of(const TileListArgs& p, int tiles, int xcd) {
  const int total = tiles * p.ntiles;
  const int per_xcd = (total + kXcds - 1) / kXcds;
  const int first = (int)p.by_ntiles(xcd * per_xcd), last = (int)p.by_ntiles(max((xcd + 1) * per_xcd - 1, 0));
  TileRange r;
  r.lo = first - (kGroupTiles - 1) > 0 ? first - (kGroupTiles - 1) : 0;
  r.hi = last + kGroupTiles < tiles ? last + kGroupTiles : tiles;
  if (r.hi > r.lo + TileList<MAX>::kMaxLocal) r.hi = r.lo + TileList<MAX>::kMaxLocal;
  r.tiles = tiles;
  return r;
}

// Tiles start at multiples of `per_tile` blocks inside each run of equal expert ids and never cross a run; up
// to kGroupTiles consecutive tiles of a run form a group.  scratch holds nblocks ints.
template <int MAX>
__device__ TileRange build_any_order(const TileListArgs& p, int nblocks, int xcd, int* scratch, TileList<MAX>& list) {
  const int per_tile = p.per_tile;
  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  for (int j = tid; j < nblocks; j += kTileThreads) scratch[j] = p.expert_ids[j];
  __syncthreads();
  const int chunk = (nblocks + kTileThreads - 1) / kTileThreads;
  const int j0 = tid * chunk < nblocks ? tid * chunk : nblocks;
  const int j1 = j0 + chunk < nblocks ? j0 + chunk : nblocks;
  // start of the run that contains block j = prefix max of (j if a run starts at j else -1)
  int start = -1;
  for (int j = j0; j < j1; ++j)
    if (j == 0 || scratch[j] != scratch[j - 1]) start = j;
  const int scan = wave_scan_max(start);
  int before = __shfl_up(scan, 1);
  if (lane == 0) before = -1;
  if (lane == kWave - 1) list.wave_part[wave] = scan;
  __syncthreads();
  for (int i = 0; i < wave; ++i) before = list.wave_part[i] > before ? list.wave_part[i] : before;
  __syncthreads();
  int leaders = 0;
  int cur = before;
  for (int j = j0; j < j1; ++j) {
    if (j == 0 || scratch[j] != scratch[j - 1]) cur = j;
    if ((j - cur) % per_tile == 0) ++leaders;
  }
  const int incl = wave_inclusive_scan_add(leaders);
  if (lane == kWave - 1) list.wave_part[wave] = incl;
  __syncthreads();
  int t = incl - leaders, tiles = 0;
  for (int i = 0; i < kTileThreads / kWave; ++i) {
    if (i < wave) t += list.wave_part[i];
    tiles += list.wave_part[i];
  }
  const TileRange r = tile_range_of<MAX>(p, tiles < MAX ? tiles : MAX, xcd);
  cur = before;
  for (int j = j0; j < j1; ++j) {
    if (j == 0 || scratch[j] != scratch[j - 1]) cur = j;
    if ((j - cur) % per_tile != 0) continue;
    if (t >= r.lo && t < r.hi) {
      int nb = 1;
      while (nb < per_tile && j + nb < nblocks && scratch[j + nb] == scratch[j]) ++nb;
      const int e = scratch[j];
      list.desc[t - r.lo] = (uint32_t)j | ((uint32_t)nb << 16) | ((uint32_t)(((j - cur) / per_tile) % kGroupTiles) << 20);
      list.expert[t - r.lo] = e >= 0 && e < p.E ? (uint16_t)e : (uint16_t)0xffff;
    }
    ++t;
  }
  __syncthreads();
  // the leader of a group counts its members and writes the size into all of them
  const int count = r.hi - r.lo;
  for (int g = tid; g < count; g += kTileThreads) {
    if (((list.desc[g] >> 20) & 7u) != 0) continue;
    int size = 1;
    while (size < kGroupTiles && g + size < count && ((list.desc[g + size] >> 20) & 7u) == (uint32_t)size) ++size;
    for (int i = 0; i < size; ++i) list.desc[g + i] |= (uint32_t)size << 24;
  }
  __syncthreads();
  return r;
}

// Entry t: tile r of the n tiles of expert e, whose run of `blocks` blocks starts at `first_block`.
template <int MAX>
__device__ __forceinline__ void put_tile(const TileListArgs& p, TileList<MAX>& list, const TileRange& range, int t, int e,
                                         int first_block, int blocks, int n, int r) {
  if (t < range.lo || t >= range.hi) return;
  const int in_group = n - (r & ~(kGroupTiles - 1));
  int from = r * p.per_tile, to = from + p.per_tile < blocks ? from + p.per_tile : blocks;
  if (p.even) from = r * blocks / n, to = (r + 1) * blocks / n;
  list.desc[t - range.lo] = (uint32_t)(first_block + from) | ((uint32_t)(to - from) << 16) | ((uint32_t)(r & (kGroupTiles - 1)) << 20) |
                            ((uint32_t)(in_group < kGroupTiles ? in_group : kGroupTiles) << 24);
  list.expert[t - range.lo] = (uint16_t)e;
}

// The same list when the expert ids are known to ascend over the used blocks, with -1 behind them (what moe_align
// writes): every expert then owns at most one run of blocks, found by comparing a block with its neighbours, and the
// number of tiles in front of an expert is one scan over the experts instead of two over the blocks.  Runs of ids outside
// [0, E) get no tiles.  scratch holds 2 * E ints, E <= 2 * kTileThreads.  All entries are read, used or not, so that nothing
// waits for their number, and four per thread at a time: this is in front of everything a workgroup does (with 1150
// entries the first step began 11.2 us into the launch, 5.2 of them here; now 8.9 and 4.0; in a dense layer, where nothing has
// to be looked up, 5.6 and 1.9, now 3.8 and 0.6).
template <int MAX>
__device__ TileRange build_ascending(const TileListArgs& p, int xcd, int* scratch, TileList<MAX>& list) {
  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  if (p.identity) {  // a dense layer: all tiles are one expert's, nothing to look up
    const int n = (int)p.by_per_tile(p.blocks + p.per_tile - 1);
    const TileRange range = tile_range_of<MAX>(p, n < MAX ? n : MAX, xcd);
    for (int r = range.lo + tid; r < range.hi; r += kTileThreads) put_tile(p, list, range, r, 0, 0, p.blocks, n, r);
    __syncthreads();
    return range;
  }
  int* first = scratch;        // first block of the expert's run
  int* end = scratch + p.E;    // one past its last block
  for (int e = tid; e < 2 * p.E; e += kTileThreads) scratch[e] = 0;
  for (int j0 = 0; j0 < p.blocks; j0 += 4 * kTileThreads) {
    int e[4], prev[4], next[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int j = j0 + i * kTileThreads + tid, last = p.blocks - 1;
      e[i] = p.expert_ids[j < last ? j : last];
      prev[i] = p.expert_ids[j < last ? (j > 0 ? j - 1 : 0) : last > 0 ? last - 1 : 0];
      next[i] = p.expert_ids[j + 1 < last ? j + 1 : last];
    }
    if (j0 == 0) __syncthreads();
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int j = j0 + i * kTileThreads + tid;
      if (j < p.blocks && e[i] >= 0 && e[i] < p.E) {
        if (j == 0 || e[i] != prev[i]) first[e[i]] = j;
        if (j + 1 == p.blocks || e[i] != next[i]) end[e[i]] = j + 1;
      }
    }
  }
  __syncthreads();
  // thread t owns experts 2t and 2t + 1
  int f[2], nb[2], tiles[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int e = 2 * tid + i;
    f[i] = e < p.E ? first[e] : 0;
    nb[i] = e < p.E ? end[e] - f[i] : 0;
    tiles[i] = (int)p.by_per_tile(nb[i] + p.per_tile - 1);
  }
  const int mine = tiles[0] + tiles[1];
  const int incl = wave_inclusive_scan_add(mine);
  if (lane == kWave - 1) list.wave_part[wave] = incl;
  __syncthreads();
  int t = incl - mine, total = 0;
#pragma unroll
  for (int i = 0; i < kTileThreads / kWave; ++i) {
    const int w = list.wave_part[i];
    if (i < wave) t += w;
    total += w;
  }
  const TileRange range = tile_range_of<MAX>(p, total < MAX ? total : MAX, xcd);
  if (p.E == 1) {  // all tiles are one expert's
    for (int r = tid; r < total; r += kTileThreads) put_tile(p, list, range, r, 0, first[0], end[0] - first[0], total, r);
  } else {
#pragma unroll
    for (int i = 0; i < 2; ++i)
      for (int r = 0; r < tiles[i]; ++r, ++t) put_tile(p, list, range, t, 2 * tid + i, f[i], nb[i], tiles[i], r);
  }
  __syncthreads();
  return range;
}

// A task's second word: expert | channel tile << 16.  Both halves are full ranges (a matrix of less than 2^32 bytes in rows of at
// least 256 has up to 65536 channel tiles), so no bit is left for "no more tasks": that is the word with all bits set, whose
// expert no layer has.
constexpr uint32_t kNoTask = 0xffffffffu;
__host__ __device__ constexpr uint32_t task_word(uint32_t expert, uint32_t channel_tile) { return expert | channel_tile << 16; }
__host__ __device__ constexpr int task_expert(uint32_t word) { return word == kNoTask ? -1 : (int)(word & 0xffffu); }
__host__ __device__ constexpr int task_channel_tile(uint32_t word) { return (int)(word >> 16); }
static_assert(kMaxExperts <= 0xffff, "an expert's half of a task word is never all ones");

// Task `task` of a launch: its tile's entry (0 blocks where the expert id is out of range) and its task_word.
// The tasks of a group of T token tiles of one expert run channel tile by channel tile: T consecutive tasks (on
// neighbouring compute units) stream the same weight tile.
template <int MAX>
__device__ __forceinline__ uint2 look_up_task(const TileListArgs& p, const TileList<MAX>& list, const TileRange& range, int task) {
  const int tile0 = (int)p.by_ntiles(task);
  const uint32_t d0 = list.desc[tile0 - range.lo];
  const int first = tile0 - (int)((d0 >> 20) & 7u);
  const int T = (int)((d0 >> 24) & 15u);
  const int pos = task - first * p.ntiles;
  // pos / T: (pos + 0.5) / T is at least 1 / (2 * kGroupTiles) = 2^-4 away from any integer; with a quotient below 2^16 (channel
  // tiles), the reciprocal's 1 ulp and the product's rounding are an error below 2^-6
  const int nt = (int)(((float)pos + 0.5f) * __builtin_amdgcn_rcpf((float)T));
  const int tile = first + (pos - nt * T) - range.lo;
  const int e = list.expert[tile];
  return make_uint2(e == 0xffff ? list.desc[tile] & 0xff00ffffu : list.desc[tile], task_word(e == 0xffff ? 0u : (uint32_t)e, (uint32_t)nt));
}

// The last round of an XCD's tasks is rarely full: where its tasks leave at least half of the workgroups idle, each is cut
// into two or four pieces that run side by side.  A piece does not cost its share (its steps are shorter, not fewer), so
// nothing is cut where more than half are busy.  Whole / in pieces, us: narrow tiles, gate_up, experts of 4096 x 1408 with 20
// rows each: 24 (2.06 rounds) 54.3 / 51.9, 40 (3.44) 78.4 / 76.3, 64 (5.5) 121.3 / 118.3; 34 (2.92: nothing to cut) 65.5 / 65.4;
// deep tiles, 4096 x 1408 with skewed routing at 517 tokens, the layer 315.8 / 314.4; wide tiles, 128 of 2048 x 768 at 8192
// tokens (7.2 and 9.7 rounds), the layer 469.4 / 468.7.
// Task and piece of place `at` (= workgroup of the XCD + round * stride), of `tasks` of the XCD.
struct TaskPiece {
  int task;    // -1: none
  int piece;
  int pieces;
};
__device__ __forceinline__ TaskPiece piece_at(int at, int tasks, int stride) {
  const int full = tasks / stride * stride, rest = tasks - full;
  if (at < full) return TaskPiece{at, 0, 1};
  const int shift = 4 * rest <= stride ? 2 : 2 * rest <= stride ? 1 : 0;
  const int i = at - full;
  if (i >= rest << shift) return TaskPiece{-1, 0, 1};
  return TaskPiece{full + (i >> shift), i & ((1 << shift) - 1), 1 << shift};
}

// Rows whose stride is a multiple of 4096 bytes have one reduction step of all of them on a few memory channels, and
// workgroups that start together stay together for a while.  There a task starts its reduction (int32 sums, exact in any order)
// at start_step and wraps around; all channel tiles of an expert at the same one, so that they still share its token rows
// (with the channel tile in it too, the wide tiles lost up to 8 %).  Long launches spread by themselves, and it then depends on
// how far apart the XCDs' ranges lie, and even on where the weights lie, whether it helps.  gate_up of 92 layer shapes, several
// allocations each, both sides on the same buffers: by how many per cent it is faster with it, by the weights of all experts, mean
// (worst .. best).  Evenly routed, up to 0.65 GiB 12 (-2 .. 24) with narrow tiles of 16 rows, 13 (-8 .. 32) with deep ones of 64,
// 0.65-0.8 GiB 6 (-1 .. 19) and 10 (2 .. 27); beyond, narrow, K = 4096 0 to 1 (-8 .. 14), 8192 0.85-1.2 GiB -6 (-13 .. 5), 1.2-1.7 2,
// 1.7-2.2 -1 (-10 .. 5), 12288 -3 to 1; deep, K = 4096 1 to 3 (-5 .. 19), 8192 -2 (-15 .. 15), 2, -1 (-16 .. 8), 12288 -8 to 3.  64
// experts of 8192 x 1024 (1 GiB), narrow, 161 us without and 179 with it, of 8192 x 2048, deep, 335 and 385.  Zipf routing: 4 and 6 up
// to 0.8 GiB, beyond -1 to 1, but layers of 17 to 80 tokens, whose launches read a part of the experts, 1 to 4 (128 experts of 4096 x
// 1408, 1536 and 2560), -3 (64 of 8192 x 1024) and -4 (32 of 8192 x 2048).  Hence up to 0.8 GiB, K = 4096 at any size.  Given away:
// 64 experts of 4096 x 2048 (1 GiB), narrow, 5 to 7 %, 96 of 4096 x 1408, deep, 4.  Of K = 1024, 2048, 2560, 3072, 3584, 5120, 6144
// and 7168 none moves by more than 1 %.  The wide tiles do not use it: with many rows per expert it changes nothing.
// The starts of few experts are spread over all 4096 bytes: next to each other, one step apart, they share channels again.  One
// step apart / spread, us, narrow tiles: 8 experts of 8192 x 1536 40 / 36 (all at the first step: 38.5), of 8192 x 2048 53 / 45, 16
// of 4096 x 1536 39 / 35, of 8192 x 1024 48 / 44; deep: 16 of 4096 x 2048 57 / 49, of 8192 x 2048 107 / 92; of 17 layer shapes none slower.
constexpr int64_t kRotateBytes = 819ll << 20;  // 0.8 GiB
constexpr int kStartSteps = 32;                // of 128 bytes
// Steps between the starts of two experts that follow each other; 0: all tasks start at the first one.
__host__ __device__ constexpr int rotation(int k, int64_t weight_bytes, int experts) {
  if (k % 4096 != 0 || (k > 4096 && weight_bytes > kRotateBytes)) return 0;
  return experts < kStartSteps ? kStartSteps / experts : 1;
}
__host__ __device__ constexpr int start_step(int expert, int rotation) { return expert * rotation % kStartSteps; }

}  // namespace moe_i8
