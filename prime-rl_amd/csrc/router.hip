// Token-choice top-k routing for gfx950: scores, optional grouped pre-selection, top-k, weight
// normalisation and the compact routed-experts record, one launch, one wavefront per token.  HBM traffic is the
// minimum: the logits once in, k weights and k indices out.
#include "router_body.hpp"

namespace moe_i8 {
namespace {

constexpr int kThreads = 256;
constexpr int kTokensPerBlock = kThreads / kWave;

template <int C>
__global__ __launch_bounds__(kThreads) void route_topk_kernel(RouteArgs a) {
  const int64_t tok = (int64_t)blockIdx.x * kTokensPerBlock + threadIdx.x / kWave;
  if (tok >= a.m) return;
  float logits[C], w;
  int id;
  route_logits<C>(a, tok, logits);
  route_select<C>(a, logits, a.top_k, id, w);
  route_write(a, tok, id, w);
}

}  // namespace

int route_experts_per_lane(int num_experts) {
  int c = 1;
  while (c * kWave < num_experts) c <<= 1;
  return c;
}

hipError_t launch_route_topk(const RouteArgs& a, hipStream_t stream) {
  if (a.m == 0) return hipSuccess;
  const dim3 grid((unsigned)((a.m + kTokensPerBlock - 1) / kTokensPerBlock));
  const dim3 block(kThreads);
  switch (route_experts_per_lane(a.num_experts)) {
    case 1: hipLaunchKernelGGL(route_topk_kernel<1>, grid, block, 0, stream, a); break;
    case 2: hipLaunchKernelGGL(route_topk_kernel<2>, grid, block, 0, stream, a); break;
    case 4: hipLaunchKernelGGL(route_topk_kernel<4>, grid, block, 0, stream, a); break;
    case 8: hipLaunchKernelGGL(route_topk_kernel<8>, grid, block, 0, stream, a); break;
    case 16: hipLaunchKernelGGL(route_topk_kernel<16>, grid, block, 0, stream, a); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

}  // namespace moe_i8
