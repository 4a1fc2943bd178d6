// dK and dV, hand-scheduled: the launch plan, the dispatch and the fp16 instances (the kernel is in fta_bwd_dkdv1_kernel.h; the
// bf16 instances are compiled in fta_bwd_dkdv1_bf16.hip).
#include "fta_bwd_dkdv1_kernel.h"

namespace fta {

// Query ranges of one launch each (a wave's stationary bias^T tile and the stage size are compiled in), in units of 64
// queries and as even as the row divides: four to eight units.  D = 64 has no instance of seven (14 tiles divide into stages of seven,
// of which LDS holds no three): seven and six are cut as eight and five, two sevens as eight and six, and three or more ranges that are
// not equal, or equal to seven, as ranges of four and five.  That is the slower side: as ranges of four and five / of eight, six and five (ms a
// step, dQ/dBias the same) B1 H4 1088 keys 12.2 / 11.7, 1153 15.7 / 15.2, 1280 18.3 / 17.7, 1408 25.9 / 24.2, B1 H2 1664 in bf16 22.0 / 20.8,
// 1792 25.1 / 23.8.
static int dkdv1_ranges(int L2, int D, int* out) {
  const int units = L2 / 64;
  const int n = even_ranges(units, 8, 64, out);
  if (D == 32) return n;
  if (n <= 2 ? units == 15 : (units % n != 0 || out[0] == 448)) return even_ranges(units, 5, 64, out);
  if (n == 2 && out[0] == 448) { out[0] += 64; out[1] -= 64; }
  return n;
}
// queries per stage: half of the range where that is at most 256, a short one at once; D = 64: 128, of a range of 320 160
static int dkdv1_stage(int range, int D) {
  if (D == 64 && range % 128 == 0) return 128;
  return range > 256 ? range / 2 : range;
}

bool plan_dkdv1(int B, int H, int L1, int L2, int D, Dkdv1Plan& pl) {
  if (D != 32 && D != 64) return false;
  if (L2 % 64 != 0 || L2 < 256 || L2 > (D == 64 ? 256 : 512) * kMaxRanges) return false;
  if (D == 64 && L2 == 448) return false;  // (seven units: tiled as 512)
  pl.nlaunch = dkdv1_ranges(L2, D, pl.range);
  pl.JR = pl.range[0];
  pl.NJT = pl.JR / 32;
  pl.nkg = (L2 + 127) / 128;
  pl.threads = 256;
  pl.smem = 0;
  for (int n = 0; n < pl.nlaunch; ++n) {
    const int jt = dkdv1_stage(pl.range[n], D), row = 2 * D, copy = 4096 / row;
    const size_t rows = (size_t)(jt + copy - 1) / copy * copy, pairs = (size_t)(jt * 8 + 1023) / 1024 * 1024;
    const size_t smem = 3 * (2 * rows * row + pairs) + (size_t)(pl.range[n] == jt ? 2 : 1) * 2 * 128 * row;
    pl.smem_range[n] = smem;
    if (smem > pl.smem) pl.smem = smem;
  }
  const int nch = balanced_chunks((long)B * H * pl.nkg, L1, 256, least_rows(L2));  // one workgroup per CU
  pl.rows_per_chunk = (L1 + nch - 1) / nch;
  pl.nchunks = (L1 + pl.rows_per_chunk - 1) / pl.rows_per_chunk;
  return true;
}

hipError_t launch_dkdv1(BwdParams p, const Dkdv1Plan& pl, int D, int dtype, bool hilo, bool nat, hipStream_t st) {
  p.nkg = pl.nkg; p.nchunks2 = pl.nchunks; p.rows_per_chunk2 = pl.rows_per_chunk;
  const dim3 grid((unsigned)(p.B * p.H * pl.nkg * pl.nchunks));
  p.jr0 = 0;
  for (int n = 0; n < pl.nlaunch; ++n) {
    hipError_t e = hipErrorInvalidConfiguration;
    // (nat: the caller asks for it at D = 32 with fp16 tensors only)
    if (nat) e = (dtype == kF16 && D == 32) ? launch_dkdv1_range<F16, 32, true, true>(p, pl.range[n], grid, pl.smem_range[n], st) : e;
    else if (dtype == kBF16) e = launch_dkdv1_bf16(p, pl.range[n], D, hilo, grid, pl.smem_range[n], st);
    else if (D == 64) e = launch_dkdv1_range<F16, 64, false, false>(p, pl.range[n], grid, pl.smem_range[n], st);
    else e = launch_dkdv1_range<F16, 32, false, false>(p, pl.range[n], grid, pl.smem_range[n], st);
    if (e != hipSuccess) return e;
    p.jr0 += pl.range[n];
  }
  return hipSuccess;
}

}  // namespace fta
