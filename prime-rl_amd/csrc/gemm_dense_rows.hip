// Dense int8 GEMM that quantises its own rows, for gfx950: linear layers and gated MLPs of 5 rows and more, mostly tens to
// hundreds (thousands where the channels are few: 6000 rows x 128 channels x 768).
//
// At this size a dense layer is two dependent launches, quantisation and product, and little else: 100 rows x 1000 channels x 1024
// took 7.7 us for 0.1 us of bytes and 0.3 of operations.  Here a workgroup quantises the token rows of its tile itself, into
// LDS, where they stay for the whole reduction; the weights run through a ring of stages as in the dense kernel, whose split of
// the reduction, swizzle and epilogue it shares.  What bounds it: one latency for the rows, the vector units' work on them (about
// 5 operations per element, 1 us for 32 rows of 1024), which hides the latency of the first weights, then the steps of the ring.
// Repeating the quantisation per channel tile is what limits it: 64 rows per workgroup cost as much as the launch that they save
// (64 x 64 tiles 6.9-7.7 us, never faster), and reductions beyond 4096 do not fit.
// us per call, quantisation launch and dense kernel / here: 17 rows x 2672 channels x 896 6.75 / 3.9, 103 x 992 x 1024 7.7 / 4.2,
// 309 x 512 x 896 7.2 / 4.9, 54 x 1248 x 1152 7.1 / 4.4, 122 x 8448 x 704 7.5 / 6.2, 45 x 624 x 2880 7.3 / 5.7; over 343 problems of
// 17..1000 rows x 512..14336 channels x 192..4200, taken where the estimates say so, 22 % faster on average.
#include <iterator>

#include "dense_body.hpp"
#include "quant_body.hpp"

namespace moe_i8 {
namespace {

constexpr int kWaves = 8;

struct DenseRowsParams {
  const uint16_t* x;     // [M, K] bf16
  const int8_t* w;       // [N, K]
  const float* w_scale;  // [N]
  uint16_t* out;         // [M, N] (down) or [M, N / 2] (gate_up)
  int M;
  int N;
  int K;
  int mtiles;
  int ntiles;
};

// TM x TN: tile; KS: groups of wavefronts that split the reduction; WM x WN: wavefronts of a group; S: stages; V: 1 KB vectors of a
// bf16 row (K <= 512 * V).
template <int MODE, int TM, int TN, int KS, int WM, int WN, int S, int V>
__global__ __launch_bounds__(64 * kWaves, 2) void gemm_dense_rows_kernel(DenseRowsParams p) {
  using T = DenseTiling<TM, TN, KS, WM, WN, S, TN>;
  constexpr int G = T::G, L = T::L, kThreads = T::kThreads, MT = T::MT, NT = T::NT, MF = T::MF, MI = T::MI, NI = T::NI;
  using F = typename T::F;
  static_assert(KS * G == kWaves && TM % kWaves == 0);
  constexpr int R = TM / kWaves;               // rows that a wavefront quantises
  constexpr int kPiece = TM * kStepBytes;      // 128 reduction bytes of all rows
  constexpr int kRowsAt = S * T::kStage;          // quantised rows, behind the stages: [piece][row][128]
  constexpr int kUsed = kRowsAt + V * 4 * kPiece;
  constexpr int kLds = kUsed > KS * T::kPart ? kUsed : KS * T::kPart;
  static_assert(kLds + 4 * (TM + TN) <= 160 * 1024, "LDS");
  __shared__ __align__(16) char lds[kLds];
  __shared__ __align__(16) float scales[(TN + 63) / 64 * 64 + TM];
  constexpr int kRowScales = (TN + 63) / 64 * 64;

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int g = wave / G, wg = wave % G;
  const int wm = wg / WN, wn = wg % WN;

  int tile;  // token tiles fastest
  if (!dense_tile(p.mtiles * p.ntiles, tile)) return;
  const int m0 = tile % p.mtiles * TM;
  const int nt = tile / p.mtiles;
  const int K = p.K;

  // ---- the tile's rows, the first things in flight (rows behind the last one: that one again) ----
  const int vectors = (K + 511) / 512;
  uint4 v[R][V];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int row = m0 + wave * R + r;
    const uint4* x = reinterpret_cast<const uint4*>(p.x + (int64_t)(row < p.M ? row : p.M - 1) * K);
#pragma unroll
    for (int i = 0; i < V; ++i)
      if (i < vectors) v[r][i] = i * kWave + lane < K / kQuantVec ? x[i * kWave + lane] : make_uint4(0u, 0u, 0u, 0u);
  }

  auto weight_row = [&](int r) { return dense_weight_row<MODE, TN>(nt, r, p.N); };
  const uint32_t lds0 = lds_address(lds);
  uint32_t off[L];
  bool hi[L];  // chunk in the upper 64 bytes of the step
#pragma unroll
  for (int i = 0; i < L; ++i) {
    const int r = (wg * L + i) * 8 + (lane >> 3);
    const int chunk = (lane & 7) ^ swizzle_of_row(r);
    off[i] = (uint32_t)weight_row(r) * (uint32_t)K + chunk * 16;
    hi[i] = chunk >= 4;
  }
  const int nk = (K + kStepBytes - 1) / kStepBytes;  // 128-byte pieces of the reduction; piece s * KS + g is this group's step s
  const int steps = (nk + KS - 1) / KS;
  const int mine = (nk - g + KS - 1) / KS;
  const bool ragged = K % kStepBytes != 0;
  auto issue = [&](int s, int slot, int from, int to) {
    const int piece = s * KS + g;
    const uint32_t base = lds0 + slot * T::kStage + g * T::kGroupBytes + wg * L * 1024;
    // Last 64 bytes of a ragged reduction: the rows are zero there, so the weights may be anything readable: the lower half
    // again (the next row would lie past the end of the matrix for the last one).
    const uint32_t back = ragged && piece == nk - 1 ? 64u : 0u;
#pragma unroll
    for (int i = 0; i < L; ++i)
      if (i >= from && i < to) load_to_lds_16(p.w + piece * kStepBytes, off[i] - (hi[i] ? back : 0u), base + i * 1024);
  };

  float top[R];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    top[r] = 0.0f;
#pragma unroll
    for (int i = 0; i < V; ++i)
      if (i < vectors) top[r] = fmaxf(top[r], absmax8(v[r][i]));
    asm volatile("" ::"v"(top[r]));  // the rows are waited for here, in front of the loads that follow
  }
  for (int j0 = wave * 64; j0 < TN; j0 += kThreads)
    load_to_lds_4(p.w_scale + weight_row(j0 + lane < TN ? j0 + lane : TN - 1), lds_address(scales + j0));
#pragma unroll
  for (int s = 0; s < S - 1; ++s)
    if (s < mine) issue(s, s, 0, L);

  // ---- quantisation, while the first weights are on their way ----
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int row = wave * R + r;
    const float absmax = fmaxf(wave_max(top[r]), 1e-10f);
    const float inv = 127.0f / absmax;
    if (lane == 0) scales[kRowScales + row] = absmax / 127.0f;
    char* to = lds + kRowsAt + row * kStepBytes + (((lane >> 1) & 7) ^ swizzle_of_row(row)) * 16 + (lane & 1) * 8;
#pragma unroll
    for (int i = 0; i < V; ++i)
      if (i < vectors) *reinterpret_cast<uint2*>(to + (4 * i + (lane >> 4)) * kPiece) = quant8<true>(v[r][i], inv);
  }

  int w_ld[NI], x_ld[MI], chunk[F::kSub];
  const int lrow = lane % MF;
#pragma unroll
  for (int i = 0; i < NI; ++i) w_ld[i] = (wn * NT + i * MF + lrow) * kStepBytes;
#pragma unroll
  for (int i = 0; i < MI; ++i) x_ld[i] = kRowsAt + (wm * MT + i * MF + lrow) * kStepBytes;
#pragma unroll
  for (int kk = 0; kk < F::kSub; ++kk) chunk[kk] = ((kk * (64 / MF) + lane / MF) ^ swizzle_of_row(lrow)) * 16;

  typename T::Acc acc;
#pragma unroll
  for (int i = 0; i < NI; ++i)
#pragma unroll
    for (int j = 0; j < MI; ++j)
#pragma unroll
      for (int r = 0; r < F::kRegs; ++r) acc[i][j][r] = 0;
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");  // (not __syncthreads: the loads stay in flight)

  int slot = 0;
  for (int s = 0; s < steps; ++s) {
    // this wavefront's loads of step s are in (those of the next S - 2 steps, as far as there are any, stay in flight)
    const int later = mine - 1 - s;
    wait_groups<L, S - 2>(later < 0 ? 0 : later);
    if constexpr (G > 1)
      asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    else
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    const int fill = slot == 0 ? S - 1 : slot - 1;  // the slot of step s - 1: everybody is done reading it
    const bool more = s + S - 1 < mine;
    if (s < mine) {
      const char* st = lds + slot * T::kStage + g * T::kGroupBytes;
      const char* rows = lds + (s * KS + g) * kPiece;
      v4i a[2][NI], b[2][MI];
      auto read = [&](int kk) {
#pragma unroll
        for (int i = 0; i < NI; ++i) a[kk & 1][i] = *reinterpret_cast<const v4i*>(st + w_ld[i] + chunk[kk]);
#pragma unroll
        for (int j = 0; j < MI; ++j) b[kk & 1][j] = *reinterpret_cast<const v4i*>(rows + x_ld[j] + chunk[kk]);
      };
      read(0);
#pragma unroll
      for (int kk = 0; kk < F::kSub; ++kk) {
        if (kk + 1 < F::kSub) read(kk + 1);
        // the loads of the step S - 1 ahead go out a few at a time between the multiplications
        // (with two stages they have only this step to arrive in: all of them first)
        if (more && (S > 2 || kk == 0)) issue(s + S - 1, fill, S > 2 ? kk * L / F::kSub : 0, S > 2 ? (kk + 1) * L / F::kSub : L);
#pragma unroll
        for (int i = 0; i < NI; ++i)
#pragma unroll
          for (int j = 0; j < MI; ++j) acc[i][j] = F::mul(a[kk & 1][i], b[kk & 1][j], acc[i][j]);
      }
    }
    slot = slot + 1 == S ? 0 : slot + 1;
  }
  wait_vmcnt<0>();
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  dense_results<T, MODE, true, TM, TN, KS>(acc, lds, g, wm * MT, wn * NT, scales, scales + kRowScales, m0, nt, p.M, p.N, p.out);
}

template <int MODE, int TM, int TN, int KS, int WM, int WN, int S, int V>
hipError_t launch_config(const DenseRowsParams& p0, hipStream_t stream) {
  DenseRowsParams p = p0;
  constexpr int kOut = MODE == kGateUpSilu ? TN / 2 : TN;
  const int width = MODE == kGateUpSilu ? p.N / 2 : p.N;
  p.mtiles = (p.M + TM - 1) / TM;
  p.ntiles = (width + kOut - 1) / kOut;
  const int per_xcd = (p.mtiles * p.ntiles + kXcds - 1) / kXcds;
  hipLaunchKernelGGL((gemm_dense_rows_kernel<MODE, TM, TN, KS, WM, WN, S, V>), dim3((unsigned)(per_xcd * kXcds)), dim3(64 * kWaves), 0,
                     stream, p);
  return hipGetLastError();
}

// One way to cut the problem up and what it costs: a launch takes about
//   start + rounds * (per_round + per_k * K / 1024) + waves * (per_wave + per_wave_k * K / 1024)
// where a round is as many workgroups as the device holds at a time and a wave as many as it has compute units (the same, where a
// unit holds one: then the second term is 0).  Least-squares fits to 2600 problems of 5..8192 rows x 64..20000 channels x 64..4096, the mean of the
// times with weights from memory and from the last-level cache (rms error of a fit 4-9 %).  Over 1300 problems of 5 rows and more the choice
// between these and the launches that they replace takes on average 0.2 % longer than the fastest way with weights from memory and 0.1 % with cached
// ones, 0.2 % in a captured graph (3000 problems).  Wrong by most where a nearly full round of 32 x 256 has a long reduction: 2009 rows x 832 x 832 9.3 us, quantised
// by a launch of its own 8.8.
// The 256 and 512 channel tiles are one round where the 128 channel ones are two, and a workgroup's rows serve twice as many channels; no
// split of the reduction is left, and none is missed: 16 x 256 is faster than 32 x 128, which was here, also where both are one round
// (170 rows x 4112 channels x 256 4.7 / 4.2 us).  Without / with the three of them, 60 drawn linear layers that they are picked for:
// 13 % faster on average (two 5 % slower); 67 x 12848 x 192 6.9 / 4.2, 396 x 2544 x 704 8.5 / 6.0, 135 x 6640 x 1024 8.8 / 6.3, 1073 x 960
// x 384 7.3 / 5.4, 146 x 17392 x 512 9.0 / 7.3.  Beside them 32 x 64, 48 x 64, 48 x 128, 48 x 256, 64 x 128 and 64 x 256 up to 1024,
// 32 x 64, 32 x 128, 16 x 256 and 32 x 256 up to 2048 and 16 x 64 and 16 x 128 up to 4096 gain 0.2 % or nothing.
struct Config {
  int tm, tn;   // tile
  int longest;  // reduction
  int per_cu;   // workgroups a compute unit holds at a time
  float start, per_round, per_k, per_wave, per_wave_k;  // us
  hipError_t (*gate_up)(const DenseRowsParams&, hipStream_t);
  hipError_t (*down)(const DenseRowsParams&, hipStream_t);
};
#define MOE_I8_ROWS(TM, TN, KS, WM, WN, S, V, PER_CU, START, ROUND, PER_K, WAVE, WAVE_K)                                          \
  {TM, TN, 512 * V, PER_CU, START, ROUND, PER_K, WAVE, WAVE_K, launch_config<kGateUpSilu, TM, TN, KS, WM, WN, S, V>, \
   launch_config<kDown, TM, TN, KS, WM, WN, S, V>}
const Config kConfigs[] = {
    MOE_I8_ROWS(16, 32, 4, 1, 2, 3, 2, 2, 1.63f, 0.80f, 0.23f, 0.73f, 0.63f),
    MOE_I8_ROWS(16, 64, 2, 1, 4, 3, 2, 2, 1.48f, 0.98f, 0.51f, 0.66f, 0.85f),
    MOE_I8_ROWS(16, 128, 2, 1, 4, 3, 2, 1, 0.76f, 2.41f, 1.93f, 0.0f, 0.0f),
    MOE_I8_ROWS(16, 256, 1, 1, 8, 3, 2, 1, 0.57f, 2.65f, 3.26f, 0.0f, 0.0f),
    MOE_I8_ROWS(32, 256, 1, 1, 8, 3, 2, 1, 0.15f, 4.07f, 3.42f, 0.0f, 0.0f),
    MOE_I8_ROWS(32, 512, 1, 1, 8, 2, 1, 1, -0.52f, 4.94f, 5.82f, 0.0f, 0.0f),
    MOE_I8_ROWS(16, 32, 8, 1, 1, 3, 4, 1, 0.55f, 2.86f, 0.88f, 0.0f, 0.0f),
    MOE_I8_ROWS(16, 64, 4, 1, 2, 3, 4, 1, 0.23f, 3.31f, 1.20f, 0.0f, 0.0f),
    MOE_I8_ROWS(16, 128, 2, 1, 4, 3, 4, 1, -0.29f, 3.81f, 1.81f, 0.0f, 0.0f),
    MOE_I8_ROWS(16, 32, 8, 1, 1, 2, 8, 1, -0.51f, 3.93f, 1.05f, 0.0f, 0.0f),
};

}  // namespace

// A row more costs the kernel of a few rows a pass over its registers' weights, this one nothing up to 16.  Up to 4 rows that kernel is the
// faster one or even on all but the widest matrices (4 x 8848 x 1536 6.3 / 5.1).  From 5 on both are estimated.  Over 1200 problems of 5 to 16 rows the choice
// takes 0.1 % longer than the faster of the two, 0.2 % in a captured graph (3500 problems); by fits to calls that a host sends one every 3.7 us, which hide
// how long a kernel of 3 us takes, 5 and 7 %.  us there / here in a graph: 6 x 6272 x 192 5.2 / 3.6, 7 x 4496 x 256 4.8 / 3.3, 16 x 640 x 1280 6.7 / 4.3, 5 x
// 1792 x 832 3.5 / 4.2, 5 x 3760 x 2368 4.6 / 5.7, 6 x 4080 x 3072 6.3 / 8.2, 5 x 3680 x 576 3.8 / 4.4; wrong by most 6 x 4464 x 4032 9.4 / 10.3 and 8 x 1216 x
// 1088 4.6 / 4.9.  A quantisation launch adds about 2.6 us and 0.66 per 10^6 elements to the dense kernels' estimate.
int dense_rows_pick(int64_t m, int n, int k, bool few, float us) {
  if (m < kDenseRowsFrom || (int64_t)n * k >= (1ll << 32) || n % 16 != 0 || k % 64 != 0) return -1;
  float least = few ? dense_few_estimate(m, n, k) : us + 2.6f + 0.66e-6f * (float)m * (float)k;
  int best = -1;
  const float kb = (float)k / 1024.0f, cus = (float)device_cu_count();
  for (int i = 0; i < (int)std::size(kConfigs); ++i) {
    const Config& c = kConfigs[i];
    if (k > c.longest || (c.longest > 1024 && k <= c.longest / 2)) continue;  // (fitted to reductions between the two)
    const float tiles = (float)(((m + c.tm - 1) / c.tm) * ((n + c.tn - 1) / c.tn));
    const float t = c.start + ceilf(tiles / (cus * c.per_cu)) * (c.per_round + c.per_k * kb) + ceilf(tiles / cus) * (c.per_wave + c.per_wave_k * kb);
    if (t < least) best = i, least = t;
  }
  return best;
}

DenseTile dense_rows_tile(int entry) { return {kConfigs[entry].tm, kConfigs[entry].tn}; }

hipError_t launch_dense_rows(const DenseFewArgs& a, int entry, hipStream_t stream) {
  if (entry < 0 || entry >= (int)std::size(kConfigs) || a.k > kConfigs[entry].longest) return hipErrorInvalidValue;
  DenseRowsParams p{};
  p.x = a.x;
  p.w = a.w;
  p.w_scale = a.w_scale;
  p.out = a.out;
  p.M = a.m;
  p.N = a.n;
  p.K = a.k;
  return a.mode == kGateUpSilu ? kConfigs[entry].gate_up(p, stream) : kConfigs[entry].down(p, stream);
}

}  // namespace moe_i8
