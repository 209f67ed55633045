// Dense W8A8 layer of a few rows in one launch, for gfx950: quantisation of the rows, product and epilogue.
//
// For a handful of rows the quantisation launch in front of a dense GEMM costs as much as the GEMM (3.0 and 5.2 us
// for 5 rows x 2816 channels x 4096).  Here every workgroup quantises all rows itself, one wavefront per row, into
// LDS, while its own weights are on their way from memory; a wavefront holds R weight rows in registers (16
// consecutive reduction bytes per lane) and multiplies them with row after row by v_dot4_i32_i8; the lanes' int32 sums
// (exact in any order) meet by lane permutes.  What bounds it: one memory latency and the weights' bytes, as long
// as repeating the quantisation per workgroup stays hidden behind them.
#include "quant_body.hpp"

namespace moe_i8 {
namespace {

constexpr int kWaves = 8;

// lane l: the value of lane l ^ (R / 2)
template <int R>
__device__ __forceinline__ int partner_half(int v) {
  if constexpr (R == 2) return __builtin_amdgcn_update_dpp(0, v, 0xb1, 0xf, 0xf, false);
  if constexpr (R == 4) return __builtin_amdgcn_update_dpp(0, v, 0x4e, 0xf, 0xf, false);
  const int up = __builtin_amdgcn_update_dpp(0, v, 0x104, 0xf, 0x5, false);
  return __builtin_amdgcn_update_dpp(up, v, 0x114, 0xf, 0xa, false);
}

// C: 1 KB pieces of a row (k <= 1024 * C); R: weight rows of a wavefront (gate_up: half gate, half up)
template <int MODE, int C, int R>
__global__ __launch_bounds__(64 * kWaves) void dense_few_kernel(DenseFewArgs p) {
  extern __shared__ __align__(16) int8_t xq[];  // [m][C * 1024], zero behind k
  __shared__ float a_scale[kDenseFewRows];
  constexpr int kOut = MODE == kGateUpSilu ? R / 2 : R;  // channels of a wavefront
  constexpr int kRowsAtOnce = kWave / kOut < kDenseFewRows ? kWave / kOut : kDenseFewRows;  // rows that share an epilogue
  const int lane = lane_id();
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int K = p.k, width = MODE == kGateUpSilu ? p.n / 2 : p.n;

  // the row first: its loads are waited for first
  uint4 v[2 * C];
  auto fetch = [&](int row) __attribute__((always_inline)) {
    const uint4* x = reinterpret_cast<const uint4*>(p.x + (int64_t)row * K);
#pragma unroll
    for (int i = 0; i < 2 * C; ++i) v[i] = row < p.m && i * kWave + lane < K / kQuantVec ? x[i * kWave + lane] : make_uint4(0u, 0u, 0u, 0u);
  };
  fetch(wave);
  v4i w[R][C], next[R][C];
  float ws, wu = 0.0f, next_ws, next_wu = 0.0f;
  auto fetch_weights = [&](int ch0) {
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int c0 = ch0 + r % kOut < width ? ch0 + r % kOut : width - 1;
      const v4i* row = reinterpret_cast<const v4i*>(p.w + (int64_t)(r < kOut ? c0 : width + c0) * K);
#pragma unroll
      for (int c = 0; c < C; ++c) next[r][c] = __builtin_nontemporal_load(row + (c * kWave + lane < K / 16 ? c * kWave + lane : 0));
    }
    // lane l: scales of channel ch0 + l % kOut
    const int mine = ch0 + lane % kOut < width ? ch0 + lane % kOut : width - 1;
    next_ws = p.w_scale[mine];
    if constexpr (MODE == kGateUpSilu) next_wu = p.w_scale[width + mine];
  };
  int ch0 = (blockIdx.x * kWaves + wave) * kOut;
  const int stride = gridDim.x * kWaves * kOut;
  fetch_weights(ch0);

  auto quantise = [&](int row) __attribute__((always_inline)) {
    float m = 0.0f;
#pragma unroll
    for (int i = 0; i < 2 * C; ++i) m = fmaxf(m, absmax8(v[i]));
    const float absmax = fmaxf(wave_max(m), 1e-10f);
    const float inv = 127.0f / absmax;
    if (lane == 0) a_scale[row] = absmax / 127.0f;
#pragma unroll
    for (int i = 0; i < 2 * C; ++i)
      *reinterpret_cast<uint2*>(xq + row * (C * 1024) + (i * kWave + lane) * kQuantVec) = quant8<true>(v[i], inv);
  };
  // The first row apart from the loop, in front of whose loads it would wait for the weights as well: 4 rows of 8192 on
  // 2048 channels 8.2 us in the loop, 7.4 apart, of 5120 on 4096 6.9 / 6.8.
  if (wave < p.m) quantise(wave);
  for (int row = wave + kWaves; row < p.m; row += kWaves) {
    fetch(row);
    quantise(row);
  }
  __syncthreads();

  while (true) {
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
      for (int c = 0; c < C; ++c) w[r][c] = next[r][c];
    ws = next_ws, wu = next_wu;
    const bool more = ch0 + stride < width;
    if (more) fetch_weights(ch0 + stride);
    int g = 0, u = 0;  // lane row * kOut + l: the sums of row `row`, channel ch0 + l
    for (int row = 0; row < p.m; ++row) {
      v4i q[C];
#pragma unroll
      for (int c = 0; c < C; ++c) q[c] = *reinterpret_cast<const v4i*>(xq + row * (C * 1024) + (c * kWave + lane) * 16);
      int acc[R];
#pragma unroll
      for (int r = 0; r < R; ++r) {
        acc[r] = 0;
#pragma unroll
        for (int c = 0; c < C; ++c) acc[r] = dot16(w[r][c], q[c], acc[r]);
      }
      const int totals = wave_totals<R>(acc);
      const bool mine = lane / kOut == row % kRowsAtOnce;
      if constexpr (MODE == kGateUpSilu) {
        // R totals repeat through the lanes: gate in the lower half of R lanes, up in the upper
        const int other = partner_half<R>(totals);
        const bool upper = lane & kOut;
        g = mine ? (upper ? other : totals) : g;
        u = mine ? (upper ? totals : other) : u;
      } else {
        g = mine ? totals : g;
      }
      if (row % kRowsAtOnce == kRowsAtOnce - 1 || row == p.m - 1) {
        const int first = row - row % kRowsAtOnce, at = first + lane / kOut, ch = ch0 + lane % kOut;
        if (at <= row && lane < kRowsAtOnce * kOut && ch < width)
          p.out[(int64_t)at * width + ch] = (uint16_t)(MODE == kGateUpSilu ? silu_mul_epilogue1(g, u, a_scale[at], ws, wu)
                                                                           : down_epilogue1(g, a_scale[at], ws, 1.0f));
      }
    }
    if (!more) break;
    ch0 += stride;
  }
}

template <int MODE, int C, int R>
hipError_t launch_rows(const DenseFewArgs& a, hipStream_t stream) {
  constexpr int kOut = kWaves * (MODE == kGateUpSilu ? R / 2 : R);
  const int width = MODE == kGateUpSilu ? a.n / 2 : a.n;
  const size_t lds = (size_t)a.m * C * 1024;
  const int groups = (width + kOut - 1) / kOut, most = device_cu_count();  // a workgroup per compute unit: one quantisation each
  static DynamicLds limit;
  const hipError_t err = limit.allow((const void*)dense_few_kernel<MODE, C, R>, kDenseFewRows * C * 1024);
  if (err != hipSuccess) return err;
  hipLaunchKernelGGL((dense_few_kernel<MODE, C, R>), dim3((unsigned)(groups < most ? groups : most)), dim3(64 * kWaves), lds, stream, a);
  return hipGetLastError();
}

// As many weight rows per wavefront, up to 16 KB, as leave work for every compute unit.
int rows_per_wave(int n, int pieces) {
  const int most = n / (kWaves * 200);
  return pieces <= 2 && most >= 8 ? 8 : pieces <= 4 && most >= 4 ? 4 : 2;
}

template <int MODE, int C>
hipError_t launch_pieces(const DenseFewArgs& a, hipStream_t stream) {
  const int rows = rows_per_wave(a.n, C);
  if constexpr (C <= 2)
    if (rows == 8) return launch_rows<MODE, C, 8>(a, stream);
  if constexpr (C <= 4)
    if (rows == 4) return launch_rows<MODE, C, 4>(a, stream);
  return launch_rows<MODE, C, 2>(a, stream);
}

template <int MODE>
hipError_t launch_mode(const DenseFewArgs& a, hipStream_t stream) {
  switch ((a.k + 1023) / 1024) {
    case 1: return launch_pieces<MODE, 1>(a, stream);
    case 2: return launch_pieces<MODE, 2>(a, stream);
    case 3: return launch_pieces<MODE, 3>(a, stream);
    case 4: return launch_pieces<MODE, 4>(a, stream);
    case 5: return launch_pieces<MODE, 5>(a, stream);
    case 6: return launch_pieces<MODE, 6>(a, stream);
    case 7: return launch_pieces<MODE, 7>(a, stream);
    default: return launch_pieces<MODE, 8>(a, stream);
  }
}

}  // namespace

// Every row adds its quantisation and its products, on the vector units, to each workgroup; a quantisation launch and
// the matrix units cost the same for 1 or 16 rows.  us per call here / there at 1, 4, 8 and 16 rows: 512 x 512 channels x
// reduction 4.6 4.6 4.6 6.4 / 7.6, 4096 x 2048 4.9 4.8 5.1 7.8 / 7.5, 1440 x 5696 5.1 6.0 8.0 12.8 / 8.5, 8192 x 4096 6.9 8.7
// 10.8 16.7 / 10.3, 8192 x 8192 12.9 14.6 19.3 28.8 / 15.8; gated MLP of 4096 x 1408 7.5 9.5 12.2 19.3 / 14.8.
bool dense_few_takes(int64_t m, int n, int k) {
  const int64_t weights = (int64_t)n * k;
  const int64_t most = weights <= 1 << 20 ? kDenseFewRows : weights <= 12 << 20 ? 8 : weights <= 40 << 20 ? 6 : 4;
  return m <= most && n % 16 == 0 && k % 16 == 0 && k <= 8 * 1024;
}

// Least-squares fit to 1200 problems of 5 to 16 rows, the mean of the times with weights from memory and from the last-level cache (rms error
// 3 % with a seventh term, 0.08 us per MB of weights, which the kernel that it is weighed against takes as well: both leave it out).
float dense_few_estimate(int64_t m, int n, int k) {
  const int pieces = (k + 1023) / 1024, rows = rows_per_wave(n, pieces), per_round = kWaves * rows * device_cu_count();
  const float rounds = (float)((n + per_round - 1) / per_round), held = rounds * (float)(rows * pieces);
  return 1.91f + 0.236f * (float)pieces + 0.271f * (float)((m + kWaves - 1) / kWaves - 1) + 0.022f * held +
         (float)m * (0.131f * rounds + 0.0292f * held);
}

hipError_t launch_dense_few(const DenseFewArgs& a, hipStream_t stream) {
  return a.mode == kGateUpSilu ? launch_mode<kGateUpSilu>(a, stream) : launch_mode<kDown>(a, stream);
}

}  // namespace moe_i8
