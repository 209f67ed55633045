// Symmetric int8 quantisation for gfx950, one scale per row: activations (per token, optionally
// fused with a row gather) and weights (per output channel).
//
// Activations: one 64-lane wavefront owns one output row.  The row is read once with 16-byte loads
// (8 bf16 per lane per load, all loads issued before the first use), the absolute maximum is
// reduced across the wavefront with lane permutes, and 8 int8 per lane are written with 8-byte
// stores.  HBM traffic is the minimum 2 + 1 bytes per element plus 4 bytes per row.
// Arithmetic (fp32): absmax = max(max|x|, 1e-10); scale = absmax / 127;
// q = round(x * (127 / absmax)), ties away from zero (MoE path) or to even (dense path).
//
// Weights: scale = max(absmax / 127, 1e-12); q = rint(x / scale); a wavefront walks several
// consecutive rows with the next rows' loads in flight (see quant_weights_kernel).
#include "quant_body.hpp"

namespace moe_i8 {
namespace {

constexpr int kThreads = 256;
constexpr int kRowsPerBlock = kThreads / kWave;

template <int VPL, int kMode>
__global__ __launch_bounds__(kThreads) void quant_rows_kernel(QuantArgs a) {
  const int64_t row = (int64_t)blockIdx.x * kRowsPerBlock + threadIdx.x / kWave;
  if (row < a.rows) quant_one_row<VPL, kMode>(a, row);
  if (a.route_sorted != nullptr) {
    // identity routing of a.rows rows, written by all threads of the launch in strides
    const int rows = (int)a.rows;
    const int padded = (rows + a.route_block - 1) / a.route_block * a.route_block;
    const int64_t blocks_cap = (a.route_cap + a.route_block - 1) / a.route_block;
    const int64_t step = (int64_t)gridDim.x * kThreads;
    for (int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x; i < a.route_cap; i += step) {
      a.route_sorted[i] = i < rows ? (int32_t)i : rows;
      if (i < blocks_cap) a.route_expert_ids[i] = i < padded / a.route_block ? 0 : -1;
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) *a.route_npp = padded;
  }
}

template <int kMode>
void launch_quant_rows_mode(const QuantArgs& a, dim3 grid, dim3 block, hipStream_t stream) {
  switch (quant_vectors_per_lane(a.q_stride > a.cols ? a.q_stride : a.cols)) {
    case 1: hipLaunchKernelGGL((quant_rows_kernel<1, kMode>), grid, block, 0, stream, a); break;
    case 2: hipLaunchKernelGGL((quant_rows_kernel<2, kMode>), grid, block, 0, stream, a); break;
    case 4: hipLaunchKernelGGL((quant_rows_kernel<4, kMode>), grid, block, 0, stream, a); break;
    case 8: hipLaunchKernelGGL((quant_rows_kernel<8, kMode>), grid, block, 0, stream, a); break;
    case 16: hipLaunchKernelGGL((quant_rows_kernel<16, kMode>), grid, block, 0, stream, a); break;
    default: hipLaunchKernelGGL((quant_rows_kernel<0, kMode>), grid, block, 0, stream, a); break;
  }
}

// Weights: HBM-bound, every byte touched once (nontemporal loads and stores).  A wavefront walks several
// rows through a ring of kDepth row buffers in registers: the loads of the next kDepth - 1 rows stay in
// flight while the current row is reduced, quantised and stored (a wavefront that lives for a single row
// spends much of its life with nothing outstanding, and short rows need several in flight to cover the
// HBM latency).  kDepth * VPL = 8 vectors of 16 bytes per lane, 8 KB per wavefront.  Neighbouring
// wavefronts take neighbouring rows and step over the matrix together: the whole chip reads one moving
// front (128 x 768 x 2048 x 3: 5.12-5.18 TB/s, against 4.84 with 16 consecutive rows per wavefront).
constexpr int kWeightVectorsInFlight = 8;  // 16-byte loads per lane kept in flight
constexpr int weight_ring_depth(int vpl) { return kWeightVectorsInFlight / vpl > 1 ? kWeightVectorsInFlight / vpl : 1; }

// No branch around the loads (the compiler would wait for everything outstanding at the join):
// lanes past the end of the row, and rows past the end of the wavefront's share, read the first
// vector of the share instead, one cached line for the whole wavefront.
template <int VPL>
__device__ __forceinline__ void load_weight_row(const v4i* first, const v4i* in, bool row_valid, int nvec,
                                                int lane, v4i (&v)[VPL]) {
#pragma unroll
  for (int i = 0; i < VPL; ++i) {
    const int c = lane + i * kWave;
    v[i] = __builtin_nontemporal_load(row_valid && c < nvec ? in + c : first);
  }
}

__device__ __forceinline__ uint4 as_uint4(const v4i& v) {
  return make_uint4((uint32_t)v[0], (uint32_t)v[1], (uint32_t)v[2], (uint32_t)v[3]);
}

// Rows wave, wave + waves, wave + 2 * waves, ... of the matrix `a`.
template <int VPL>
__device__ __forceinline__ void quant_weight_rows(const QuantArgs& a, int64_t wave, int64_t waves) {
  constexpr int kDepth = weight_ring_depth(VPL);
  const int lane = lane_id();
  if (wave >= a.rows) return;
  const int n = (int)((a.rows - wave + waves - 1) / waves);
  const int nvec = a.cols / kQuantVec;
  const int64_t vec_stride = a.row_stride / kQuantVec * waves;
  const v4i* first = reinterpret_cast<const v4i*>(a.x + wave * a.row_stride);
  v4i ring[kDepth][VPL];
#pragma unroll
  for (int s = 0; s < kDepth; ++s) load_weight_row<VPL>(first, first + s * vec_stride, s < n, nvec, lane, ring[s]);
  for (int r0 = 0; r0 < n; r0 += kDepth) {
#pragma unroll
    for (int s = 0; s < kDepth; ++s) {
      const int r = r0 + s;
      float m = 0.0f;
#pragma unroll
      for (int i = 0; i < VPL; ++i)
        m = fmaxf(m, lane + i * kWave < nvec ? absmax8_packed(as_uint4(ring[s][i])) : 0.0f);
      const WeightRcp ws = weight_rcp(fmaxf(wave_max(m) / 127.0f, 1e-12f));
      if (r < n) {
        const int64_t row = wave + r * waves;
        int64_t orow = row;
        if (a.rows_per_group > 0) {
          const int64_t g = a.rows >> 32 ? row / a.rows_per_group : (int64_t)((uint32_t)row / (uint32_t)a.rows_per_group);
          orow = g * a.out_rows_per_group + a.out_row_offset + (row - g * a.rows_per_group);
        }
        if (lane == 0) a.scale[orow] = ws.scale;
        uint2* out = reinterpret_cast<uint2*>(a.q + orow * (int64_t)a.cols);
#pragma unroll
        for (int i = 0; i < VPL; ++i) {
          const int c = lane + i * kWave;
          if (c < nvec) {
            const uint2 q = quant8_weights(as_uint4(ring[s][i]), ws);
            uint32_t* p = reinterpret_cast<uint32_t*>(out + c);
            __builtin_nontemporal_store(q.x, p);
            __builtin_nontemporal_store(q.y, p + 1);
          }
        }
      }
      load_weight_row<VPL>(first, first + (r + kDepth) * vec_stride, r + kDepth < n, nvec, lane, ring[s]);
    }
  }
}

// Up to three matrices in one launch (an expert layer's gate, up and down projections): workgroups in front
// of `first[1]` take matrix 0, in front of `first[2]` matrix 1, the others matrix 2.  The first two have
// rows of VA vectors per lane, the third of VB.
struct WeightQuantParams {
  QuantArgs matrix[3];
  unsigned first[3];
};
template <int VA, int VB>
__global__ __launch_bounds__(kThreads) void quant_weights_kernel(WeightQuantParams p) {
  const unsigned b = blockIdx.x;
  const int wave = threadIdx.x / kWave;
  if (b >= p.first[2]) {
    quant_weight_rows<VB>(p.matrix[2], (int64_t)(b - p.first[2]) * kRowsPerBlock + wave,
                          (int64_t)(gridDim.x - p.first[2]) * kRowsPerBlock);
  } else {
    const int i = b >= p.first[1] ? 1 : 0;
    quant_weight_rows<VA>(p.matrix[i], (int64_t)(b - p.first[i]) * kRowsPerBlock + wave,
                         (int64_t)(p.first[i + 1] - p.first[i]) * kRowsPerBlock);
  }
}

// Rows too long to hold in registers: one wavefront per row, read twice.
__global__ __launch_bounds__(kThreads) void quant_weights_long_rows_kernel(QuantArgs a) {
  const int64_t row = (int64_t)blockIdx.x * kRowsPerBlock + threadIdx.x / kWave;
  if (row < a.rows) quant_one_row<0, kQuantWeights>(a, row);
}

}  // namespace

hipError_t launch_quant_rows(const QuantArgs& a, hipStream_t stream) {
  if (a.rows == 0) return hipSuccess;
  const dim3 grid((unsigned)((a.rows + kRowsPerBlock - 1) / kRowsPerBlock));
  const dim3 block(kThreads);
  if (a.round_even)
    launch_quant_rows_mode<kQuantEven>(a, grid, block, stream);
  else
    launch_quant_rows_mode<kQuantAway>(a, grid, block, stream);
  return hipGetLastError();
}

namespace {
template <int VA, int VB>
hipError_t launch_weights(WeightQuantParams& p, int count, hipStream_t stream) {
  // Rows per wavefront: 8, unless that leaves the chip short of wavefronts (a small layer then takes as few as
  // the ring holds).  Measured over layers of 12 MB to 4.4 GB with 4 to 64 rows and 4096 to 16384 wavefronts:
  // 8 and 8192 are within 2 % of the best everywhere.
  constexpr int64_t kEnough = 8192;
  int64_t total = 0;
  int rows_per_wave[2];
  for (int most = 8;; most /= 2) {
    rows_per_wave[0] = most > weight_ring_depth(VA) ? most : weight_ring_depth(VA);
    rows_per_wave[1] = most > weight_ring_depth(VB) ? most : weight_ring_depth(VB);
    total = 0;
    for (int i = 0; i < count; ++i) {
      const int r = rows_per_wave[i == 2];
      total += (p.matrix[i].rows + r - 1) / r;
    }
    if (total >= kEnough || most == 1) break;
  }
  unsigned blocks = 0;
  for (int i = 0; i < 3; ++i) {
    p.first[i] = blocks;
    if (i >= count) continue;
    const int r = rows_per_wave[i == 2];
    const int64_t w = (p.matrix[i].rows + r - 1) / r;
    blocks += (unsigned)((w + kRowsPerBlock - 1) / kRowsPerBlock);
  }
  if (count < 3) p.first[2] = blocks;
  if (count < 2) p.first[1] = blocks;
  hipLaunchKernelGGL((quant_weights_kernel<VA, VB>), dim3(blocks), dim3(kThreads), 0, stream, p);
  return hipGetLastError();
}

template <int VA>
hipError_t launch_weights_for(WeightQuantParams& p, int vb, int count, hipStream_t stream) {
  switch (vb) {
    case 1: return launch_weights<VA, 1>(p, count, stream);
    case 2: return launch_weights<VA, 2>(p, count, stream);
    case 4: return launch_weights<VA, 4>(p, count, stream);
    case 8: return launch_weights<VA, 8>(p, count, stream);
    default: return launch_weights<VA, 16>(p, count, stream);
  }
}
}  // namespace

hipError_t launch_quant_weights(const QuantArgs* a, int count, hipStream_t stream) {
  WeightQuantParams p{};
  for (int i = 0; i < count; ++i) p.matrix[i] = a[i];
  const int va = quant_vectors_per_lane(a[0].cols), vb = count == 3 ? quant_vectors_per_lane(a[2].cols) : va;
  if (va == 0 || vb == 0) {
    for (int i = 0; i < count; ++i) {
      if (quant_vectors_per_lane(a[i].cols) != 0) {
        const hipError_t err = launch_quant_weights(a + i, 1, stream);
        if (err != hipSuccess) return err;
        continue;
      }
      hipLaunchKernelGGL(quant_weights_long_rows_kernel,
                         dim3((unsigned)((a[i].rows + kRowsPerBlock - 1) / kRowsPerBlock)), dim3(kThreads), 0, stream, a[i]);
      const hipError_t err = hipGetLastError();
      if (err != hipSuccess) return err;
    }
    return hipSuccess;
  }
  switch (va) {
    case 1: return launch_weights_for<1>(p, vb, count, stream);
    case 2: return launch_weights_for<2>(p, vb, count, stream);
    case 4: return launch_weights_for<4>(p, vb, count, stream);
    case 8: return launch_weights_for<8>(p, vb, count, stream);
    default: return launch_weights_for<16>(p, vb, count, stream);
  }
}

}  // namespace moe_i8
