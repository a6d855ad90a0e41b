// FLOW kind kernels for up to 8 x rows.
#include "ftk_flow.h"

namespace ftk {

FlowKernel pick_flow_x2(int c, int epi, bool pro) {
  return pro ? pick_flow_segments<2, true>(c, epi) : pick_flow_segments<2, false>(c, epi);
}

}  // namespace ftk
