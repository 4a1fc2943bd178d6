// dK and dV, hand-scheduled: the bf16 instances.
#include "fta_bwd_dkdv1_kernel.h"

namespace fta {

hipError_t launch_dkdv1_bf16(const BwdParams& p, int range, int D, bool hilo, dim3 grid, size_t smem, hipStream_t st) {
  if (D == 64) return launch_dkdv1_range<BF16, 64, false, false>(p, range, grid, smem, st);
  return hilo ? launch_dkdv1_range<BF16, 32, true, false>(p, range, grid, smem, st) : launch_dkdv1_range<BF16, 32, false, false>(p, range, grid, smem, st);
}

}  // namespace fta
