// FLOW kind kernels for up to 32 x rows.
#include "ftk_flow.h"

namespace ftk {

FlowKernel pick_flow_x8(int c, int epi, bool pro) {
  return pro ? pick_flow_segments<8, true>(c, epi) : pick_flow_segments<8, false>(c, epi);
}

}  // namespace ftk
