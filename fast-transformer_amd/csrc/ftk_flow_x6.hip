// FLOW kind kernels for up to 24 x rows.
#include "ftk_flow.h"

namespace ftk {

FlowKernel pick_flow_x6(int c, int epi, bool pro) {
  return pro ? pick_flow_segments<6, true>(c, epi) : pick_flow_segments<6, false>(c, epi);
}

}  // namespace ftk
