// Grouped int8 GEMM for gfx950: the streaming family's kernel for a handful of tokens, where the weights of
// the few experts in use are too little work for one wavefront per 32 weight rows.
//
// At one token of 8 experts x 1536 x 2048 the streaming kernel has 384 wavefronts for 256 compute units and
// each walks its 64 KB in eight dependent windows: the launch is the latency of that chain, not the 25 MB it
// reads.  Here a workgroup takes 16 or 32 weight rows of a block and its wavefronts split the reduction
// (128-byte pieces g, g + KS, ...), each with a private ring of LDS stages and no barrier on the way, so that
// nearly everything is requested in the first microsecond; the int32 partial sums (exact in any order) meet in
// LDS.  The token rows, of which there are few, lie whole in LDS; the down GEMM can quantise them itself from
// bf16 with the stand-alone quantiser's arithmetic (one launch less).
//
// us per launch, streaming kernel -> this one (8 experts per token, gate_up / self-quantising down):
// 1 token 11.4 -> 7.2 / 8.0 -> 5.9, 2 tokens 12.7 -> 11.3 / 9.2 -> 7.9, 3 tokens 18.1 -> 14.7 / 10.9 -> 9.5; even
// at 4 to 5 tokens, slower from 6 on (15.3 -> 16.2).
//
// Where it runs: calls of a few tokens that the two-launch layer does not take (a reduction of the down GEMM
// beyond 4096, 5 to 16 tokens on a handful of experts), and the streaming family when it is demanded.  Layer us,
// streaming kernel -> this one: 8 experts (2 per token) of 2048 x 5632 at 1 / 4 / 10 tokens 54.7 -> 29.5, 63.1 -> 47.8,
// 73.6 -> 62.1; of 4096 x 1408 at 5 / 9 tokens 41.1 -> 34.9, 42.5 -> 37.0; 4 experts of 8192 x 1024 at 14 tokens 52.8 -> 37.7.
#include "lds_loads.hpp"
#include "quant_body.hpp"

namespace moe_i8 {
namespace {

constexpr int kRows = 16;       // token rows of a tile (MFMA columns)
constexpr int kRowPad = 16;     // bytes behind a token row in LDS: 16 rows' operand reads fall on different banks
constexpr int kMaxK = 8192;
constexpr int kMaxFusedK = 2048;  // ... where the workgroup quantises its rows itself
constexpr int kMaxLds = 160 * 1024;

struct SplitParams {
  const uint16_t* a_bf16;  // down: bf16 activations [P, K] quantised here, or null
  const int8_t* a_q;
  const float* a_scale;
  const int8_t* w;
  const float* w_scale;
  const float* row_weight;
  const int32_t* sorted_ids;
  const int32_t* expert_ids;
  const int32_t* npp;
  int64_t P;
  int row_div;
  int E;
  int N;
  int K;
  int B;
  int rows;    // most rows any block holds, at most kRows
  int ntiles;  // channel tiles
  int round_even;
  uint16_t* out;
};

template <int MODE, bool kFused, int TN, int KS, int S>
__global__ __launch_bounds__(64 * KS) void gemm_split_kernel(SplitParams p) {
  constexpr int kThreads = 64 * KS;
  constexpr int NI = TN / 16;
  constexpr int L = TN / 8;  // 1 KB loads per wavefront and step
  static_assert((S - 2) * L <= 63 && S >= 2, "counted waits");
  constexpr int kStage = TN * kStepBytes;
  constexpr int kPartRow = TN * 4 + 16;
  constexpr int kPart = kRows * kPartRow;
  constexpr int kRing = S * KS * kStage > KS * kPart ? S * KS * kStage : KS * kPart;
  using F = Mfma<16>;
  extern __shared__ __align__(16) char lds[];  // ring (later: partial sums) | token rows [rows][K + pad]
  __shared__ __align__(16) float scales[TN];
  __shared__ float row_scale[kRows], row_weight[kRows];
  __shared__ int32_t row_tok[kRows];
  char* tokens = lds + kRing;

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int g = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int blk = blockIdx.y;
  const int nt = blockIdx.x;
  const int K = p.K;
  const int inter = p.N / 2;

  // one round trip: blocks in use, the block's expert and its row list (inside the arrays whatever is in use)
  const int npp = *p.npp;
  const int e = p.expert_ids[blk];
  const int32_t id = p.sorted_ids[(int64_t)blk * p.B + (lane & (kRows - 1))];
  if (blk * p.B >= npp || e < 0 || e >= p.E) return;

  auto weight_row = [&](int r) {
    if constexpr (MODE == kGateUpSilu) {
      const int half = TN / 2;
      const int ch = nt * half + (r < half ? r : r - half);
      return (ch < inter ? ch : inter - 1) + (r < half ? 0 : inter);
    } else {
      const int n = nt * TN + r;
      return n < p.N ? n : p.N - 1;
    }
  };

  // ---- weights: piece s * KS + g of every row is this wavefront's step s ----
  const int8_t* wbase = p.w + (int64_t)e * p.N * K;
  uint32_t off[L];
  bool hi[L];
#pragma unroll
  for (int i = 0; i < L; ++i) {
    const int r = i * 8 + (lane >> 3);
    const int chunk = (lane & 7) ^ swizzle_of_row(r);
    off[i] = (uint32_t)weight_row(r) * (uint32_t)K + chunk * 16;
    hi[i] = chunk >= 4;
  }
  const int nk = (K + kStepBytes - 1) / kStepBytes;
  const int mine = (nk - g + KS - 1) / KS;
  const uint32_t ring = lds_address(lds) + g * S * kStage;
  const bool ragged = K % kStepBytes != 0;
  auto issue = [&](int s, int slot) {
    const int piece = s * KS + g;
    // last 64 bytes of a ragged reduction: their products are left out below, so any readable weights do
    const uint32_t back = ragged && piece == nk - 1 ? 64u : 0u;
#pragma unroll
    for (int i = 0; i < L; ++i)
      load_to_lds_16_stream(wbase + piece * kStepBytes, off[i] - (hi[i] ? back : 0u), ring + slot * kStage + i * 1024);
  };
#pragma unroll
  for (int s = 0; s < S - 1; ++s)
    if (s < mine) issue(s, s);

  // ---- token rows, scales and routed weights into LDS, behind the first weights ----
  const bool valid = id >= 0 && id < p.P;
  const uint64_t valid_rows = __ballot(valid) & 0xffffull;
  const int nrows = __popcll(valid_rows) < p.rows ? __popcll(valid_rows) : p.rows;  // valid rows are a prefix of the block
  const int row_bytes = K + kRowPad;
  for (int i = tid; i < TN; i += kThreads) scales[i] = p.w_scale[(int64_t)e * p.N + weight_row(i)];
  if (tid < kRows) {
    row_tok[tid] = tid < nrows ? id : -1;
    row_weight[tid] = tid < nrows && p.row_weight ? p.row_weight[id] : 1.0f;
    if constexpr (!kFused) row_scale[tid] = tid < nrows ? p.a_scale[id / p.row_div] : 0.0f;
  }
  if constexpr (kFused) {
    constexpr int kVec = kMaxFusedK / kQuantVec / kWave;
    for (int r = g; r < nrows; r += KS) {
      const int32_t t = __builtin_amdgcn_readlane(id, r);
      const uint4* in = reinterpret_cast<const uint4*>(p.a_bf16 + (int64_t)t * K);
      const int nvec = K / kQuantVec;
      uint4 v[kVec];
      float m = 0.0f;
#pragma unroll
      for (int c = 0; c < kVec; ++c) {
        const int idx = lane + c * kWave;
        v[c] = idx < nvec ? in[idx] : make_uint4(0u, 0u, 0u, 0u);
        m = fmaxf(m, absmax8(v[c]));
      }
      const float absmax = fmaxf(wave_max(m), 1e-10f);
      const float inv = 127.0f / absmax;
      if (lane == 0) row_scale[r] = absmax / 127.0f;
#pragma unroll
      for (int c = 0; c < kVec; ++c) {
        const int idx = lane + c * kWave;
        if (idx < nvec)
          *reinterpret_cast<uint2*>(tokens + r * row_bytes + idx * 8) =
              p.round_even ? quant8<true>(v[c], inv) : quant8<false>(v[c], inv);
      }
    }
  } else {
    constexpr int kVec = kMaxK / 16 / kWave;
    for (int r = g; r < nrows; r += KS) {
      const int32_t t = __builtin_amdgcn_readlane(id, r);
      const v4i* in = reinterpret_cast<const v4i*>(p.a_q + (int64_t)(t / p.row_div) * K);
      v4i v[kVec];
#pragma unroll
      for (int c = 0; c < kVec; ++c)
        if (lane + c * kWave < K / 16) v[c] = in[lane + c * kWave];
#pragma unroll
      for (int c = 0; c < kVec; ++c)
        if (lane + c * kWave < K / 16) *reinterpret_cast<v4i*>(tokens + r * row_bytes + (lane + c * kWave) * 16) = v[c];
    }
  }
  __syncthreads();

  // ---- multiply ----
  typename F::Acc acc[NI];
#pragma unroll
  for (int i = 0; i < NI; ++i) acc[i] = v4i{0, 0, 0, 0};
  const int col = lane & 15, grp = lane >> 4;
  const char* b_row = tokens + (col < nrows ? col : nrows - 1) * row_bytes + grp * 16;
  int slot = 0;
  for (int s = 0; s < mine; ++s) {
    wait_groups<L, S - 2>(mine - 1 - s);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // and it has read the slot that is filled next
    const int fill = slot == 0 ? S - 1 : slot - 1;
    if (s + S - 1 < mine) issue(s + S - 1, fill);
    const char* st = lds + (g * S + slot) * kStage;
    const int k0 = (s * KS + g) * kStepBytes;
#pragma unroll
    for (int kk = 0; kk < F::kSub; ++kk) {
      if (k0 + kk * 64 >= K) continue;  // the half that a ragged reduction does not have
      const v4i b = *reinterpret_cast<const v4i*>(b_row + k0 + kk * 64);
#pragma unroll
      for (int i = 0; i < NI; ++i) {
        const v4i a = *reinterpret_cast<const v4i*>(st + (i * 16 + col) * kStepBytes + (((kk * 4 + grp) ^ swizzle_of_row(col)) * 16));
        acc[i] = F::mul(a, b, acc[i]);
      }
    }
    slot = slot + 1 == S ? 0 : slot + 1;
  }
  wait_vmcnt<0>();
  __syncthreads();  // everybody is done with the ring

  // ---- partial sums meet in LDS: [group][token][channel] ----
#pragma unroll
  for (int i = 0; i < NI; ++i) *reinterpret_cast<v4i*>(lds + g * kPart + col * kPartRow + (i * 16 + 4 * grp) * 4) = acc[i];
  __syncthreads();
  constexpr int kOut = MODE == kGateUpSilu ? TN / 2 : TN;
  const int width = MODE == kGateUpSilu ? inter : p.N;
  auto total4 = [&](int tok, int ch, int (&v)[4]) {
    v4i s = *reinterpret_cast<const v4i*>(lds + tok * kPartRow + ch * 4);
#pragma unroll
    for (int k = 1; k < KS; ++k) s += *reinterpret_cast<const v4i*>(lds + k * kPart + tok * kPartRow + ch * 4);
    v[0] = s[0], v[1] = s[1], v[2] = s[2], v[3] = s[3];
  };
  for (int u = tid; u < nrows * (kOut / 4); u += kThreads) {
    const int tok = u / (kOut / 4), c = u % (kOut / 4) * 4;
    const int n = nt * kOut + c;
    if (n >= width) continue;
    int v[4];
    total4(tok, c, v);
    const float4 ws = *reinterpret_cast<const float4*>(scales + c);
    uint2 o;
    if constexpr (MODE == kGateUpSilu) {
      int up[4];
      total4(tok, c + kOut, up);
      o = silu_mul_epilogue4(v, up, row_scale[tok], ws, *reinterpret_cast<const float4*>(scales + c + kOut));
    } else {
      o = down_epilogue4(v, row_scale[tok], ws, row_weight[tok]);
    }
    *reinterpret_cast<uint2*>(p.out + (int64_t)row_tok[tok] * width + n) = o;
  }
}

// LDS in front of the token rows: the ring, later the partial sums.
constexpr int ring_bytes(int tn, int ks, int stages) {
  return stages * ks * tn * kStepBytes > ks * kRows * (tn * 4 + 16) ? stages * ks * tn * kStepBytes : ks * kRows * (tn * 4 + 16);
}

template <int MODE, bool kFused, int TN, int KS, int S>
hipError_t launch_config(const SplitParams& p0, int64_t blocks, hipStream_t stream) {
  SplitParams p = p0;
  constexpr int kOut = MODE == kGateUpSilu ? TN / 2 : TN;
  constexpr int kRing = ring_bytes(TN, KS, S);
  p.ntiles = ((MODE == kGateUpSilu ? p.N / 2 : p.N) + kOut - 1) / kOut;
  const size_t bytes = kRing + (size_t)p.rows * (p.K + kRowPad);
  static DynamicLds limit;
  const hipError_t err = limit.allow((const void*)gemm_split_kernel<MODE, kFused, TN, KS, S>, kMaxLds - 1024);
  if (err != hipSuccess) return err;
  hipLaunchKernelGGL((gemm_split_kernel<MODE, kFused, TN, KS, S>), dim3((unsigned)p.ntiles, (unsigned)blocks), dim3(64 * KS), bytes,
                     stream, p);
  return hipGetLastError();
}

int64_t blocks_of(const GemmArgs& a) { return (a.sorted_cap + a.block_size - 1) / a.block_size; }

// Eight wavefronts on 16 rows while that makes no more than four workgroups per compute unit, then two on 32
// (fewer, longer workgroups: 11.3 against 11.5-12.0 us at two tokens, 17.7 against 19.6 at four).
bool eight_wavefronts(int64_t blocks, int n) { return blocks * (n / 16) <= 4 * (int64_t)device_cu_count(); }

template <int MODE, bool kFused>
hipError_t launch_mode(const SplitParams& p, int64_t blocks, hipStream_t stream) {
  return eight_wavefronts(blocks, p.N) ? launch_config<MODE, kFused, 16, 8, 2>(p, blocks, stream)
                                       : launch_config<MODE, kFused, 32, 2, 2>(p, blocks, stream);
}

}  // namespace

// Measured crossover with the streaming kernel, in the wavefronts that one would have (one per 32 weight rows
// and block) on a device that holds 3072 of them: gate_up 18.1 -> 14.7 us at 1152, 19.0 -> 17.6 at 1536, even
// at 2048 and 2304; down 10.9 -> 9.5 at 1536, 12.1 -> 11.1 at 2048, even at 2560, slower at 3072.
//
// The token rows lie whole in LDS, so they decide how many workgroups of two wavefronts a compute unit holds, and a second
// round of workgroups costs more than the split saves.  us per gate_up, streaming kernel / this one: 8 experts of 4096 x
// 1408 (704 workgroups) 21.7 / 21.3 at 9 rows, three to a unit, and 21.8 / 30.2 at 10, two to a unit; 16 experts of 2048
// x 1024 (1024 workgroups) 12.4 / 17.3 at 12 rows, three to a unit.
bool gemm_split_takes(const GemmArgs& a) {
  const int64_t most_rows = a.max_rows_per_expert > 0 && a.max_rows_per_expert < a.num_pairs ? a.max_rows_per_expert : a.num_pairs;
  const int64_t cus = device_cu_count(), blocks = blocks_of(a);
  if (a.mode == kAccI32 || most_rows > kRows || a.k > kMaxK || (int64_t)a.n * a.k >= (1ll << 32) ||
      blocks * (a.n / 32) > (a.mode == kGateUpSilu ? 8 : 10) * cus)
    return false;
  const int64_t rows_lds = most_rows * (a.k + kRowPad);
  if (eight_wavefronts(blocks, a.n)) return ring_bytes(16, 8, 2) + rows_lds <= kMaxLds - 1024;
  const int64_t used = blocks < a.num_experts ? blocks : a.num_experts;  // (an expert's rows fit one block)
  return used * ((a.n + 31) / 32) <= cus * (kMaxLds / (ring_bytes(32, 2, 2) + rows_lds));
}
bool gemm_split_fuses_quant(int k) { return k <= kMaxFusedK; }

hipError_t launch_gemm_split(const GemmArgs& a, hipStream_t stream) {
  SplitParams p{};
  p.a_bf16 = a.a_bf16;
  p.a_q = a.a_q;
  p.a_scale = a.a_scale;
  p.w = a.w;
  p.w_scale = a.w_scale;
  p.row_weight = a.row_weight;
  p.sorted_ids = a.sorted_token_ids;
  p.expert_ids = a.expert_ids;
  p.npp = a.num_tokens_post_padded;
  p.P = a.num_pairs;
  p.row_div = a.row_div;
  p.E = a.num_experts;
  p.N = a.n;
  p.K = a.k;
  p.B = a.block_size;
  const int64_t most_rows = a.max_rows_per_expert > 0 && a.max_rows_per_expert < a.num_pairs ? a.max_rows_per_expert : a.num_pairs;
  p.rows = (int)most_rows;
  p.round_even = a.a_round_even ? 1 : 0;
  p.out = static_cast<uint16_t*>(a.out);
  const int64_t blocks = blocks_of(a);
  if (a.mode == kGateUpSilu) return launch_mode<kGateUpSilu, false>(p, blocks, stream);
  return a.a_bf16 ? launch_mode<kDown, true>(p, blocks, stream) : launch_mode<kDown, false>(p, blocks, stream);
}

}  // namespace moe_i8
