// FLOW kind kernels for up to 16 x rows.
#include "ftk_flow.h"

namespace ftk {

FlowKernel pick_flow_x4(int c, int epi, bool pro) {
  return pro ? pick_flow_segments<4, true>(c, epi) : pick_flow_segments<4, false>(c, epi);
}

}  // namespace ftk
