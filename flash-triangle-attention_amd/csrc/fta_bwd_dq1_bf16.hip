// dQ and dBias, hand-scheduled: the bf16 instances.
#include "fta_bwd_dq1w_kernel.h"

namespace fta {

hipError_t launch_dq1_bf16(const BwdParams& p, int range, int D, bool hilo, dim3 grid, size_t smem, hipStream_t st) {
  if (D == 64) return launch_dq1_range<BF16, 64, false, false>(p, range, grid, smem, st);
  return hilo ? launch_dq1_range<BF16, 32, true, false>(p, range, grid, smem, st) : launch_dq1_range<BF16, 32, false, false>(p, range, grid, smem, st);
}

hipError_t launch_dq1w_bf16(const BwdParams& p, int range, dim3 grid, size_t smem, hipStream_t st) { return launch_dq1w_range<BF16>(p, range, grid, smem, st); }

}  // namespace fta
