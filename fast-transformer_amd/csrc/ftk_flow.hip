// FLOW kind dispatch.
#include "ftk_internal.h"

namespace ftk {

typedef void (*FlowKernel)(ProjArgs, int);
FlowKernel pick_flow_x1(int c, int epi, bool pro);
FlowKernel pick_flow_x2(int c, int epi, bool pro);
FlowKernel pick_flow_x4(int c, int epi, bool pro);
FlowKernel pick_flow_x6(int c, int epi, bool pro);
FlowKernel pick_flow_x8(int c, int epi, bool pro);

static FlowKernel pick_flow(int M, int K, int epi, bool pro) {
  if (M < 1 || M > kFlowMaxRows || K < 8 || K % 8) return nullptr;
  const int c = flow_segments(K);
  switch (flow_x_loads(M)) {
    case 1: return pick_flow_x1(c, epi, pro);
    case 2: return pick_flow_x2(c, epi, pro);
    case 4: return pick_flow_x4(c, epi, pro);
    case 6: return pick_flow_x6(c, epi, pro);
    default: return pick_flow_x8(c, epi, pro);
  }
}

bool flow_supported(int M, int K, int epi, bool pro) { return pick_flow(M, K, epi, pro) != nullptr; }

hipError_t launch_flow(const ProjArgs& a, int epi, const FlowShape& s, hipStream_t stream) {
  FlowKernel k = pick_flow(a.M, a.K, epi, a.gamma != nullptr);
  if (k == nullptr || s.grid < 1 || s.grid > s.tiles || s.tiles != flow_tiles(epi, a.N, kFlowTile) ||
      a.out_add != nullptr || a.residual != nullptr)
    return hipErrorInvalidValue;
  hipLaunchKernelGGL(k, dim3(s.grid), dim3(64 * kFlowWaves), 0, stream, a, s.tiles);
  return hipGetLastError();
}

}  // namespace ftk
