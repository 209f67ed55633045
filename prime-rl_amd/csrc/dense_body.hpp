// What the two dense kernels share, the one that reads quantised rows and the one that quantises them: the tile of a workgroup,
// its weight rows and the partial sums' way out.  The loop over the reduction's steps stands in each kernel: as a function the compiler
// arranges it anew, and the dense kernel's 192 x 320 tile keeps ten of its registers in scratch.
#pragma once

#include "lds_loads.hpp"

namespace moe_i8 {

constexpr int kXcds = 8;

// TM x TN: tile; KS: groups of wavefronts that split the reduction; WM x WN: wavefronts of a group; S: stages; ROWS: rows of a
// group's stage.
template <int TM, int TN, int KS, int WM, int WN, int S, int ROWS>
struct DenseTiling {
  static constexpr int G = WM * WN;              // wavefronts of a group: they share the group's stages
  static constexpr int kThreads = 64 * KS * G;
  static constexpr int L = ROWS / 8 / G;         // 1 KB loads per wavefront and step
  static_assert(ROWS % (8 * G) == 0, "a group's loads divide evenly");
  static_assert((S - 2) * L <= 63 && S >= 2, "counted waits");
  static constexpr int kGroupBytes = ROWS * kStepBytes;
  static constexpr int kStage = KS * kGroupBytes;
  static constexpr int MT = TM / WM, NT = TN / WN;
  static constexpr int MF = MT % 32 == 0 && NT % 32 == 0 ? 32 : 16;
  static constexpr int MI = MT / MF, NI = NT / MF;
  using F = Mfma<MF>;
  using Acc = typename F::Acc[NI][MI];
  static constexpr int kPartRow = TN * 4 + 16;   // bytes of a token's row of partial sums
  static constexpr int kPart = TM * kPartRow;
};

// Whether this workgroup has a tile, and which.  The workgroups of one XCD (id % 8) take neighbouring tiles.
__device__ __forceinline__ bool dense_tile(int total, int& tile) {
  const int per_xcd = (total + kXcds - 1) / kXcds;
  tile = (blockIdx.x % kXcds) * per_xcd + blockIdx.x / kXcds;
  return !(tile >= total || (int)(blockIdx.x / kXcds) >= per_xcd);
}

// LDS weight row r of channel tile nt -> row of w (behind the last one: that one again).  gate_up: the gate rows of a tile in front of
// the up rows, or (TURNS) 16 of one and 16 of the other in turns.
template <int MODE, int TN, bool TURNS = false>
__device__ __forceinline__ int dense_weight_row(int nt, int r, int N) {
  if constexpr (MODE == kGateUpSilu) {
    const int inter = N / 2, half = TN / 2;
    const int ch = nt * half + (TURNS ? r / 32 * 16 + r % 16 : r < half ? r : r - half);
    return (ch < inter ? ch : inter - 1) + ((TURNS ? r % 32 < 16 : r < half) ? 0 : inter);
  } else {
    const int n = nt * TN + r;
    return n < N ? n : N - 1;
  }
}

// The int32 partial sums of the KS groups meet in LDS, [group][token][channel], and leave as results.  tok0, ch0: the wavefront's
// first row and channel of the tile; w_scales, row_scales: of the tile, in LDS.
template <class T, int MODE, bool THROUGH, int TM, int TN, int KS>
__device__ __forceinline__ void dense_results(const typename T::Acc& acc, char* lds, int g, int tok0, int ch0, const float* w_scales,
                                              const float* row_scales, int m0, int nt, int M, int N, uint16_t* to) {
  constexpr int MF = T::MF;
  const int lane = threadIdx.x & 63;
  char* part = lds + g * T::kPart;
#pragma unroll
  for (int i = 0; i < T::NI; ++i)
#pragma unroll
    for (int j = 0; j < T::MI; ++j)
#pragma unroll
      for (int q = 0; q < T::F::kRegs / 4; ++q) {
        const int tok = tok0 + j * MF + lane % MF;
        const int ch = ch0 + i * MF + (MF == 32 ? 8 * q : 0) + 4 * (lane / MF);
        *reinterpret_cast<v4i*>(part + tok * T::kPartRow + ch * 4) =
            v4i{acc[i][j][4 * q], acc[i][j][4 * q + 1], acc[i][j][4 * q + 2], acc[i][j][4 * q + 3]};
      }
  __syncthreads();

  constexpr int kOut = MODE == kGateUpSilu ? TN / 2 : TN;  // output channels of the tile
  constexpr int kPieces = kOut / 8;                        // 16-byte pieces of an output row
  const int width = MODE == kGateUpSilu ? N / 2 : N;
  auto total4 = [&](int tok, int ch, int (&v)[4]) {
    v4i s = *reinterpret_cast<const v4i*>(lds + tok * T::kPartRow + ch * 4);
#pragma unroll
    for (int k = 1; k < KS; ++k) s += *reinterpret_cast<const v4i*>(lds + k * T::kPart + tok * T::kPartRow + ch * 4);
    v[0] = s[0], v[1] = s[1], v[2] = s[2], v[3] = s[3];
  };
  for (int u = threadIdx.x; u < TM * kPieces; u += T::kThreads) {
    const int tok = u / kPieces, c = u % kPieces * 8;
    const int m = m0 + tok, n = nt * kOut + c;
    if (m >= M || n >= width) continue;
    const float as = row_scales[tok];
    uint2 o[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int ch = c + 4 * h;
      int v[4];
      total4(tok, ch, v);
      const float4 ws = *reinterpret_cast<const float4*>(w_scales + ch);
      if constexpr (MODE == kGateUpSilu) {
        int up[4];
        total4(tok, ch + kOut, up);
        o[h] = silu_mul_epilogue4(v, up, as, ws, *reinterpret_cast<const float4*>(w_scales + ch + kOut));
      } else {
        o[h] = down_epilogue4(v, as, ws, 1.0f);
      }
    }
    store16(to + (int64_t)m * width + n, v4i{(int)o[0].x, (int)o[0].y, (int)o[1].x, (int)o[1].y}, THROUGH);
  }
}

}  // namespace moe_i8
