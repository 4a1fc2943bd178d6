// Forward, hand-scheduled (D = 32): the instances for rows of two and four key slabs.
#include "fta_fwd1_kernel.h"

namespace fta {

hipError_t launch_fwd1_slabs(const FwdParams& p, const FwdPlan& pl, int dtype, bool tl, dim3 grid, dim3 block, hipStream_t st) {
  FTA_FWD1_CASE(9, 4, 2, 2) FTA_FWD1_CASE(10, 4, 2, 2) FTA_FWD1_CASE(11, 4, 2, 2) FTA_FWD1_CASE(12, 4, 2, 2)
  FTA_FWD1_CASE(13, 4, 2, 2) FTA_FWD1_CASE(14, 4, 2, 2) FTA_FWD1_CASE(15, 4, 2, 2) FTA_FWD1_CASE(16, 4, 2, 2)
  FTA_FWD1_CASE(10, 8, 2, 2) FTA_FWD1_CASE(12, 8, 2, 2) FTA_FWD1_CASE(14, 8, 2, 2) FTA_FWD1_CASE(16, 8, 2, 2)
  FTA_FWD1_CASE(9, 8, 2, 4) FTA_FWD1_CASE(11, 8, 2, 4) FTA_FWD1_CASE(13, 8, 2, 4)
  FTA_FWD1_CASE(10, 8, 2, 4) FTA_FWD1_CASE(12, 8, 2, 4) FTA_FWD1_CASE(14, 8, 2, 4)
  return hipErrorInvalidConfiguration;
}

}  // namespace fta
