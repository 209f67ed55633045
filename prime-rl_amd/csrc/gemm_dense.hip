// Dense int8 GEMM for gfx950: one weight matrix that every row visits (linear layers, shared experts).
//
// The grouped families cut such a problem into tiles of 128 or 256 channels, sized for a layer whose
// experts fill the chip.  One matrix does not: 5 rows x 2816 channels were 22-44 workgroups on 256
// compute units, each alone with the latency of its reduction.  Here the tile is chosen so that about
// one workgroup per compute unit results, down to 16 rows x 16 channels, and inside a workgroup the
// REDUCTION is split: its wavefronts form KS groups, group g multiplies the 128-byte pieces g, g + KS, ...
// of every row through LDS stages of its own, and the int32 partial sums (exact in any order) meet in
// LDS at the end.  With one wavefront per group no barrier is needed before that.  What bounds a
// workgroup is the rate at which its operands arrive (about 50 bytes per clock and compute unit), so up
// to 150 KB of loads stay in flight (S stages) and 128 bytes of every row are fetched at a time.
//
// Kernel durations in a trace, the fastest grouped family (narrow tiles) / this kernel, rows x channels x reduction, us:
// 64x4096x4096 18.0 / 6.2, 333x4096x2048 14.0 / 8.5, 1115x1792x1536 11.6 / 7.7 (about 3 of each are what the trace shows for
// a kernel that does nothing); from a few thousand rows and channels on the 256 x 256 tiles win: see kConfigs.
//
// Loads go global -> LDS (16 bytes per lane, 8 rows x 128 bytes each) with the 16-byte chunk index
// XOR-swizzled with the row, as in the grouped families.  They are issued a few at a time between the
// multiplications of a step: all of them at its start hold up the wavefront until the address unit has
// taken them (333x4096x2048 9.0 -> 8.5 us, 333x4096x4096 14.2 -> 13.0, 1000x2384x3200 16.7 -> 15.7).  Activation rows are padded with zeros to a multiple of 128
// bytes (the quantiser writes them), which lets a reduction of any multiple of 64 run on the same path.
#include <iterator>

#include "dense_body.hpp"

namespace moe_i8 {
namespace {

struct DenseParams {
  const int8_t* a_q;     // [M, lda], zero between K and lda
  const float* a_scale;  // [M]
  const int8_t* w;       // [N, K]
  const float* w_scale;  // [N]
  uint16_t* out;         // [M, N] (down) or [M, N / 2] (gate_up)
  int M;
  int N;
  int K;
  int lda;
  int mtiles;
  int ntiles;
};

// Results of a launch up to which they are written through to memory: left in the L2s all of them are written back when the launch
// ends, in one go.  Beyond, the L2s have written most of them back by then, and stores to memory cost more.  Linear layers with
// their quantisation, 270 problems of 20..8192 rows, 512..14336 channels and a reduction of 512 / 1024 / 2048 / 4096 / 7168, by how
// many per cent faster on average through to memory, by the size of the results: up to 1 MB 0, 1-2 MB 0 / 1 / 1 / 1 / 1, 2-4 MB 4 /
// 4 / 3 / 2 / 1, 4-8 MB 7 / 6 / 4 / 2 / 1, 8-16 MB 13 / 11 / 5 / 2 / 0, 16-32 MB 9 / 6 for the first two (from here on the others run on
// the wide tiles), 32-64 MB 3; of 512 and 640, 68 MB 2, 94 MB 0, 109 MB -1, 128 MB and more -3 (8192 x 512 x 8192 66.6 us left in
// the L2s, 70.0 through to memory).
constexpr int64_t kThroughBytes = 96 << 20;

// THROUGH: results are written through to memory.  (A template argument: decided at run time it cost the smallest launches 0.2 of 7 us.)
template <int MODE, bool THROUGH, int TM, int TN, int KS, int WM, int WN, int S, int WPE>
__global__ __launch_bounds__(64 * KS * WM * WN, WPE) void gemm_dense_kernel(DenseParams p) {
  using T = DenseTiling<TM, TN, KS, WM, WN, S, TM + TN>;
  using F = typename T::F;
  constexpr int G = T::G, L = T::L, kThreads = T::kThreads, MT = T::MT, NT = T::NT, MF = T::MF, MI = T::MI, NI = T::NI;
  // Sums that are not partial, of tiles whose int32 sums would not fit or that are pairs of half as many results: finished in registers,
  // they meet in LDS as bf16 (gate_up of 128 x 128: 1-1.4 % of an MLP; plain results of it, 1-3 % slower, stay below).
  // For gate_up 16 weight rows of 32 are then gate rows and 16 the matching up rows: a lane has both in its registers.
  constexpr bool kFinished = KS == 1 && (TM * TN > 128 * 128 || MODE == kGateUpSilu);
  constexpr int kOut = MODE == kGateUpSilu ? TN / 2 : TN;  // output channels of the tile
  constexpr int kOutRow = kOut * 2 + 16;
  constexpr int kResults = kFinished ? TM * kOutRow : KS * T::kPart;
  constexpr int kLds = S * T::kStage > kResults ? S * T::kStage : kResults;
  static_assert(kLds + 4 * (TM + TN) <= 160 * 1024, "LDS");
  __shared__ __align__(16) char lds[kLds];
  __shared__ __align__(16) float scales[(TM + TN + 63) / 64 * 64];

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int g = wave / G, wg = wave % G;
  const int wm = wg / WN, wn = wg % WN;

  int tile;
  if (!dense_tile(p.mtiles * p.ntiles, tile)) return;
  constexpr int kBand = 8;  // token tiles that run together over all channel tiles
  const int band = tile / (kBand * p.ntiles);
  const int in_band = tile - band * kBand * p.ntiles;
  const int band_m = p.mtiles - band * kBand < kBand ? p.mtiles - band * kBand : kBand;
  const int m0 = (band * kBand + in_band % band_m) * TM;
  const int nt = in_band / band_m;
  auto weight_row = [&](int r) { return dense_weight_row<MODE, TN, kFinished>(nt, r, p.N); };

  const uint32_t lds0 = lds_address(lds);
  // scales of the tile's channels and rows, the first things in flight
  for (int j0 = wave * 64; j0 < TM + TN; j0 += kThreads) {
    const int j = j0 + lane < TM + TN ? j0 + lane : TM + TN - 1;
    const int m = m0 + j - TN;
    load_to_lds_4(j < TN ? p.w_scale + weight_row(j) : p.a_scale + (m < p.M ? m : p.M - 1), lds_address(scales + j0));
  }

  // ---- loads: 1 KB load i of this wavefront fills rows 8 * (wg * L + i) .. + 8 of its group's stage ----
  uint32_t off[L];
  bool hi[L];  // weight chunk in the upper 64 bytes of the step
#pragma unroll
  for (int i = 0; i < L; ++i) {
    const int rb = wg * L + i;
    const int r = rb * 8 + (lane >> 3);
    const int chunk = (lane & 7) ^ swizzle_of_row(r);
    if (rb * 8 < TN) {
      off[i] = (uint32_t)weight_row(r) * (uint32_t)p.K + chunk * 16;
      hi[i] = chunk >= 4;
    } else {
      const int m = m0 + r - TN;
      off[i] = (uint32_t)(m < p.M ? m : p.M - 1) * (uint32_t)p.lda + chunk * 16;
      hi[i] = false;
    }
  }
  const int nk = (p.K + kStepBytes - 1) / kStepBytes;  // 128-byte pieces of the reduction; piece s * KS + g is this group's step s
  const int steps = (nk + KS - 1) / KS;
  const int mine = (nk - g + KS - 1) / KS;
  const bool ragged = p.K % kStepBytes != 0;
  auto issue = [&](int s, int slot, int from, int to) {
    const int piece = s * KS + g;
    const int koff = piece * kStepBytes;
    const uint32_t base = lds0 + slot * T::kStage + g * T::kGroupBytes;
    // Last 64 bytes of a ragged reduction: the activation rows are zero there, so the weights may be anything
    // readable: the lower half again (the next row would lie past the end of the matrix for the last one).
    const uint32_t back = ragged && piece == nk - 1 ? 64u : 0u;
#pragma unroll
    for (int i = 0; i < L; ++i) {
      if (i < from || i >= to) continue;
      const int rb = wg * L + i;
      const bool is_w = rb * 8 < TN;
      load_to_lds_16((is_w ? p.w : p.a_q) + koff, off[i] - (hi[i] ? back : 0u), base + rb * 1024);
    }
  };

  int w_ld[NI], x_ld[MI], chunk[F::kSub];
  const int lrow = lane % MF;
#pragma unroll
  for (int i = 0; i < NI; ++i) w_ld[i] = (wn * NT + i * MF + lrow) * kStepBytes;
#pragma unroll
  for (int i = 0; i < MI; ++i) x_ld[i] = (TN + wm * MT + i * MF + lrow) * kStepBytes;
#pragma unroll
  for (int kk = 0; kk < F::kSub; ++kk) chunk[kk] = ((kk * (64 / MF) + lane / MF) ^ swizzle_of_row(lrow)) * 16;

  typename T::Acc acc;
#pragma unroll
  for (int i = 0; i < NI; ++i)
#pragma unroll
    for (int j = 0; j < MI; ++j)
#pragma unroll
      for (int r = 0; r < F::kRegs; ++r) acc[i][j][r] = 0;

#pragma unroll
  for (int s = 0; s < S - 1; ++s)
    if (s < mine) issue(s, s, 0, L);

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
      v4i a[2][NI], b[2][MI];
      auto read = [&](int kk) {
#pragma unroll
        for (int i = 0; i < NI; ++i) a[kk & 1][i] = *reinterpret_cast<const v4i*>(st + w_ld[i] + chunk[kk]);
#pragma unroll
        for (int j = 0; j < MI; ++j) b[kk & 1][j] = *reinterpret_cast<const v4i*>(st + x_ld[j] + chunk[kk]);
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

  if constexpr (kFinished) {
    constexpr int kPieces = kOut / 8;  // 16-byte pieces of an output row
    const int width = MODE == kGateUpSilu ? p.N / 2 : p.N;
    static_assert(MODE != kGateUpSilu || NT % 32 == 0, "gate and up rows in turns of 16");
    constexpr int kSets = MODE == kGateUpSilu ? NI * F::kRegs / 8 : NI * F::kRegs / 4;  // of 4 channels of a lane and token
#pragma unroll
    for (int j = 0; j < MI; ++j) {
      const int tok = wm * MT + j * MF + lrow;
      const float as = scales[TN + tok];
#pragma unroll
      for (int t = 0; t < kSets; ++t) {
        // set t: registers 4 * q .. of block i; of gate_up the up rows are the ones 16 weight rows on
        const int i = MF == 32 ? t / (MODE == kGateUpSilu ? 2 : 4) : MODE == kGateUpSilu ? 2 * t : t;
        const int q = MF == 32 ? t % (MODE == kGateUpSilu ? 2 : 4) : 0;
        const int at = wn * NT + i * MF + 8 * q + 4 * (lane / MF);  // row of the tile
        const float4 ws = *reinterpret_cast<const float4*>(scales + at);
        int v[4], up[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          v[r] = acc[i][j][4 * q + r];
          if constexpr (MODE == kGateUpSilu) up[r] = MF == 32 ? acc[i][j][(4 * q + 8 + r) % F::kRegs] : acc[(i + 1) % NI][j][r];
        }
        uint2 o;
        if constexpr (MODE == kGateUpSilu)
          o = silu_mul_epilogue4(v, up, as, ws, *reinterpret_cast<const float4*>(scales + at + 16));
        else
          o = down_epilogue4(v, as, ws, 1.0f);
        const int c = MODE == kGateUpSilu ? at / 32 * 16 + at % 16 : at;
        *reinterpret_cast<uint2*>(lds + tok * kOutRow + c * 2) = o;
      }
    }
    __syncthreads();
    for (int u = threadIdx.x; u < TM * kPieces; u += kThreads) {
      const int tok = u / kPieces, c = u % kPieces * 8;
      const int m = m0 + tok, n = nt * kOut + c;
      if (m < p.M && n < width) store16(p.out + (int64_t)m * width + n, *reinterpret_cast<const v4i*>(lds + tok * kOutRow + c * 2), THROUGH);
    }
  } else {
    dense_results<T, MODE, THROUGH, TM, TN, KS>(acc, lds, g, wm * MT, wn * NT, scales, scales + TN, m0, nt, p.M, p.N, p.out);
  }
}

template <int MODE, bool THROUGH, int TM, int TN, int KS, int WM, int WN, int S, int WPE>
hipError_t launch_config(const DenseParams& p0, hipStream_t stream) {
  DenseParams p = p0;
  constexpr int kOut = MODE == kGateUpSilu ? TN / 2 : TN;
  const int width = MODE == kGateUpSilu ? p.N / 2 : p.N;
  p.mtiles = (p.M + TM - 1) / TM;
  p.ntiles = (width + kOut - 1) / kOut;
  const int per_xcd = (p.mtiles * p.ntiles + kXcds - 1) / kXcds;
  hipLaunchKernelGGL((gemm_dense_kernel<MODE, THROUGH, TM, TN, KS, WM, WN, S, WPE>), dim3((unsigned)(per_xcd * kXcds)),
                     dim3(64 * KS * WM * WN), 0, stream, p);
  return hipGetLastError();
}

// One way to cut the problem up and what it costs.  A launch takes about
//   start + rounds * per_round + (full rounds * per_k + the last one's share) * K / 1024 + per_mb * MB of results,
// where a round is as many workgroups as the device holds at a time, and a last round of a few tiles takes per_k_few and one of many up to per_k
// (the chip's power is the limit: its clock falls as more matrix cores work).  Small tiles are bound by a round's
// latency and by how fast a compute unit takes in its two operands, large ones by the matrix pipes at the
// clock the power limit allows.
struct Config {
  int tm, tn;       // tile
  int per_cu;       // workgroups a compute unit holds at a time
  float start;      // us
  float per_round;  // us
  float per_k;      // us per 1024 reduction bytes of a full round
  float per_k_few;  // ... of a nearly empty one
  float per_mb, per_mb_gate_up;  // us per MB of results, plain ones and gate_up's with its SiLU
  hipError_t (*gate_up)(const DenseParams&, hipStream_t);
  hipError_t (*down)(const DenseParams&, hipStream_t);
};
#define MOE_I8_DENSE_STORES(THROUGH, TM, TN, KS, WM, WN, S, WPE, PER_CU, START, ROUND, PER_K, PER_K_FEW, MB, MB_GU) \
  {TM, TN, PER_CU, START, ROUND, PER_K, PER_K_FEW, MB, MB_GU, launch_config<kGateUpSilu, THROUGH, TM, TN, KS, WM, WN, S, WPE>, \
   launch_config<kDown, THROUGH, TM, TN, KS, WM, WN, S, WPE>}
#define MOE_I8_DENSE(...) MOE_I8_DENSE_STORES(true, __VA_ARGS__)
// The constants are least-squares fits: those of the tiles up to 96 x 96 to 2000 linear layers and 1500 gate_up GEMMs of 5..2500 rows, 64..14000 weight rows
// and 64..8192 (rms error of a fit 6-10 %), the others' and the 256-row ones' to 1700 and 1200 of 500..16384, 768..16384 and 256..6144 (5-6 %).  The choice takes on
// average 0.2 % longer than the fastest tile over the former; over 400 linear layers and 400 gate_up GEMMs that nothing was fitted to, of the latter's range, 0.38 and
// 0.33 %.  Without a charge for the results of the dense tiles, and with one of the wide ones' that did not go by the mode or the reduction, it was 0.4 and 1.3 %.
// The four largest are for problems that fill the chip badly in 128 x 128 tiles (more rounds of less) and in 256 x 256 ones (half a
// round): linear layers, us without / with them, 1818 rows x 4384 channels x 3008 54.0 / 39.1, 4868 x 3456 x 7680 164 / 138, 6508 x
// 3984 x 6592 231 / 193, 5755 x 1488 x 1536 33.6 / 28.1.  192 x 192, 192 x 256, 256 x 256, 320 x 192, 128 x 256, 256 x 128, 64 x 192,
// 64 x 256 and 128 x 64 beside them add nothing.
// 96 x 96 is for what takes two rounds of 64 x 128 and half a round of 128 x 128 (which it meets at 256 tiles, 2.4 million results):
// 40 drawn linear layers that it is picked for are 4-16 % faster, 9.6 % on average, us without / with it: 151 rows x 11472 channels x
// 2880 18.3 / 15.4, 550 x 4000 x 3136 20.2 / 17.7, 2167 x 944 x 1728 17.1 / 15.5, 567 x 3968 x 704 9.12 / 8.63.  With four wavefronts of
// 96 x 32 or six of 96 x 32 (three stages as well) it is up to 12 % slower over several rounds; 96 x 64, 64 x 96, 48 x 64, 80 x 64,
// 48 x 96 and 96 x 128 (two stages only) beside it gain 0.1 % or nothing.
const Config kConfigs[] = {
    MOE_I8_DENSE(16, 16, 8, 1, 1, 2, 4, 1, 2.72f, 0.49f, 0.35f, 0.54f, 0.51f, 4.37f),
    MOE_I8_DENSE(16, 32, 8, 1, 1, 3, 2, 1, 1.94f, 1.36f, 0.62f, 0.60f, 0.0f, 2.52f),
    MOE_I8_DENSE(32, 32, 8, 1, 1, 2, 2, 1, 1.81f, 1.55f, 0.84f, 0.73f, 0.0f, 0.73f),
    MOE_I8_DENSE(32, 64, 4, 1, 2, 3, 2, 1, 1.64f, 1.75f, 1.37f, 1.15f, 0.03f, 0.23f),
    MOE_I8_DENSE(64, 64, 2, 2, 2, 4, 2, 1, 1.68f, 1.73f, 1.98f, 1.61f, 0.10f, 0.19f),
    MOE_I8_DENSE(64, 128, 2, 2, 2, 3, 2, 1, 1.64f, 1.98f, 2.82f, 2.46f, 0.07f, 0.29f),
    MOE_I8_DENSE(96, 96, 2, 2, 2, 3, 2, 1, 1.68f, 2.12f, 3.17f, 3.11f, 0.14f, 0.47f),
    MOE_I8_DENSE(128, 128, 1, 2, 4, 4, 2, 1, 1.57f, 2.24f, 4.52f, 3.76f, 0.05f, 0.19f),
    MOE_I8_DENSE(128, 128, 1, 2, 2, 2, 2, 2, 2.15f, 1.43f, 7.62f, 5.74f, 0.12f, 0.27f),
    MOE_I8_DENSE(128, 192, 1, 4, 2, 3, 2, 1, 1.56f, 2.83f, 6.10f, 4.81f, 0.05f, 0.21f),
    MOE_I8_DENSE(256, 192, 1, 4, 2, 2, 2, 1, 1.45f, 4.51f, 10.25f, 8.34f, 0.07f, 0.22f),
    MOE_I8_DENSE(192, 320, 1, 4, 2, 2, 2, 1, 1.60f, 5.54f, 11.72f, 10.92f, 0.08f, 0.18f),
    MOE_I8_DENSE(192, 384, 1, 2, 4, 2, 2, 1, 0.80f, 6.54f, 14.22f, 11.98f, 0.07f, 0.21f),
};
// The 256-row tiles of the grouped family (one persistent workgroup per compute unit).  Their stores are not hidden behind another round's product: 0.18
// us per MB, where rows of the result begin inside 64 bytes 0.20 more, up to 0.09 of which a longer reduction hides (5780 rows x 2672 channels x 512:
// 24.8 us, in 192 x 384 tiles 19.4); gate_up 0.41 per MB of its own results, half as many as it has weight rows, with the SiLU that is not hidden either.
// us, the dense tiles taken with the former charges / the wide ones: 14508 x 3328 x 256 43.9 / 35.2, 9405 x 11520 x 256 77.8 / 63.0, 8747 x 8448 x 640 82.4 /
// 69.5, 4025 x 15536 x 768 89.1 / 76.2; gate_up 2048 x 7936 x 1024 30.4 / 26.6, 6510 x 11264 x 640 81.4 / 72.0, 4096 x 2816 x 4096 58.5 / 58.6; left to the dense
// tiles: gate_up of 5047 x 1920 x 2304 37.7 / 40.2; wrong by most: 1605 x 13504 x 512 28.1 / 25.3 and, between two
// dense tiles, 8018 x 7088 x 512 72.4 in 128 x 128 / 63.8 in 192 x 320.
const Config kWide = {256, 256, 1, 5.99f, 0.13f, 10.29f, 7.13f, 0.18f, 0.41f, nullptr, nullptr};

// Those tiles of kConfigs that the estimates choose for results of more than kThroughBytes (of 200 000 random ones up to 4 GB: a large
// result fills the chip with the larger tiles, and 128 x 128 with one workgroup per compute unit and 128 x 192 are for those that do not).
const Config kLarge[] = {
    MOE_I8_DENSE_STORES(false, 128, 128, 1, 2, 2, 2, 2, 2, 2.15f, 1.43f, 7.62f, 5.74f, 0.12f, 0.27f),
    MOE_I8_DENSE_STORES(false, 256, 192, 1, 4, 2, 2, 2, 1, 1.45f, 4.51f, 10.25f, 8.34f, 0.07f, 0.22f),
    MOE_I8_DENSE_STORES(false, 192, 320, 1, 4, 2, 2, 2, 1, 1.60f, 5.54f, 11.72f, 10.92f, 0.08f, 0.18f),
    MOE_I8_DENSE_STORES(false, 192, 384, 1, 2, 4, 2, 2, 1, 0.80f, 6.54f, 14.22f, 11.98f, 0.07f, 0.21f),
};

float estimate(const Config& c, int mode, int64_t m, int64_t n, int64_t k) {
  const int64_t tiles = ((m + c.tm - 1) / c.tm) * ((n + c.tn - 1) / c.tn);
  const int64_t room = (int64_t)device_cu_count() * c.per_cu;
  const float full = (float)(tiles / room), last = (float)(tiles % room) / (float)room;
  const float rounds = last > 0.0f ? full + 1.0f : full;
  const float turns = full * c.per_k + (last > 0.0f ? c.per_k_few + last * (c.per_k - c.per_k_few) : 0.0f);
  float per_mb = mode == kGateUpSilu ? c.per_mb_gate_up : c.per_mb;  // (rows that begin inside 64 bytes cost more)
  if (mode != kGateUpSilu && n % 32) per_mb += &c == &kWide ? 0.195f - 0.121f * (k < 768 ? (float)k / 1024.0f : 0.75f) : 0.022f;
  const float mb = (float)(mode == kGateUpSilu ? m * (n / 2) : m * n) * 2e-6f;
  return c.start + rounds * c.per_round + turns * (float)k / 1024.0f + per_mb * mb;
}

}  // namespace

int dense_row_stride(int k) { return (k + kStepBytes - 1) / kStepBytes * kStepBytes; }

DensePick gemm_dense_pick(int mode, int64_t m, int n, int k, bool wide_allowed) {
  DensePick best{-1, wide_allowed ? estimate(kWide, mode, m, n, k) : 0.0f};
  for (int i = 0; i < (int)std::size(kConfigs); ++i) {
    const float us = estimate(kConfigs[i], mode, m, n, k);
    if (us < best.us || (i == 0 && !wide_allowed)) best = {i, us};
  }
  // per-lane source offsets are 32-bit: the weights and the activation matrix must each span less than 4 GiB
  if (m < 1 || (int64_t)n * k >= (1ll << 32) || m * dense_row_stride(k) >= (1ll << 32)) best.entry = -1;
  return best;
}

DenseTile gemm_dense_tile(int entry) { return {kConfigs[entry].tm, kConfigs[entry].tn}; }

bool gemm_dense_through(int mode, int64_t m, int n) { return m * (mode == kGateUpSilu ? n / 2 : n) * 2 <= kThroughBytes; }

hipError_t launch_gemm_dense(const DenseArgs& a, int entry, hipStream_t stream) {
  if (entry < 0 || entry >= (int)std::size(kConfigs)) return hipErrorInvalidValue;
  DenseParams p{};
  p.a_q = a.a_q;
  p.a_scale = a.a_scale;
  p.w = a.w;
  p.w_scale = a.w_scale;
  p.out = static_cast<uint16_t*>(a.out);
  p.M = (int)a.m;
  p.N = a.n;
  p.K = a.k;
  p.lda = dense_row_stride(a.k);
  const Config* c = kConfigs + entry;
  if (!gemm_dense_through(a.mode, a.m, a.n))
    for (const Config& l : kLarge)
      if (l.tm == c->tm && l.tn == c->tn && l.per_cu == c->per_cu) c = &l;
  return a.mode == kGateUpSilu ? c->gate_up(p, stream) : c->down(p, stream);
}

}  // namespace moe_i8
