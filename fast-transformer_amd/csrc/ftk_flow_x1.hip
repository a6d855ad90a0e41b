// FLOW kind kernels for up to 4 x rows.
#include "ftk_flow.h"

namespace ftk {

FlowKernel pick_flow_x1(int c, int epi, bool pro) {
  return pro ? pick_flow_segments<1, true>(c, epi) : pick_flow_segments<1, false>(c, epi);
}

}  // namespace ftk
