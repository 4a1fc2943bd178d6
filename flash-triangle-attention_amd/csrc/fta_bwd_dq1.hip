// dQ and dBias, hand-scheduled: the launch plan, the dispatch and the fp16 instances (the kernel is in fta_bwd_dq1_kernel.h; the
// bf16 instances are compiled in fta_bwd_dq1_bf16.hip).
#include "fta_bwd_dq1w_kernel.h"

namespace fta {

// Key ranges of one launch each, as even as the row divides: later ones add into the dQ that the first stored.
// D = 32: two slabs of four to eight tiles (256 to 512 keys); rows of 256 keys, which one slab covers, take that
// (128 queries per workgroup instead of 64, and no exchange between slabs).  D = 64: one slab of five to eight tiles.
static int dq1_ranges(int L2, int D, int* out) {
  return D == 64 ? even_ranges(L2 / 32, 8, 32, out) : even_ranges(L2 / 64, 8, 64, out);
}
static int dq1_slabs(int L2, int D) { return (D == 64 || L2 <= 256) ? 1 : 2; }

// D = 64, rows of more than 384 keys: ranges of 256, 384 or 512 keys in one workgroup's two slabs, tiled to the next multiple of 128.  Q, dO and
// O are read, and dQ written, once a range, and a range of up to 256 keys, as below, is half as long: training steps (us), those ranges / these:
// B2 H8 400 keys 2823 / 2726, 448 in bf16 3170 / 3000, 460 3425 / 3215, 512 3895 / 3610 (dQ/dBias 2 x 856 / 1408); B1 H4 530 1808 / 1652, 640 2293 / 2160,
// 701 in bf16 3283 / 3109, 1024 8660 / 8000, 1536 29.4 / 27.2 ms.  257 to 384 keys stay as below: the two slabs of one would tile their two ranges of
// up to 192 no shorter.  Three or more ranges that are not equal stay as below, too, in five to seven launches, although that is the slower side: as
// below / in unequal ranges of these (ms a step) B1 H4 1153 keys 15.7 / 15.0, 1280 18.3 / 17.4, 1408 25.9 / 24.2, B1 H2 1664 in bf16 22.0 / 20.8,
// 1792 25.1 / 23.8.
static bool plan_dq1w(int B, int H, int L1, int L2, int row, Dq1Plan& pl) {
  const int units = (row + 127) / 128;
  const int n = row > 384 && row <= 512 * kMaxRanges ? even_ranges(units, 4, 128, pl.range) : 0;
  if (n == 0 || (n > 2 && units % n != 0)) return false;
  pl.Lt = units * 128;
  pl.nlaunch = n;
  pl.threads = 256;
  pl.ring = 4; pl.nb = 1; pl.SK = 2; pl.QB = 2;
  pl.nqg = (L2 + 63) / 64;
  pl.KR = pl.range[0];
  pl.smem = 160 * 1024;  // four stages of 32 KB, Q and dO rows of 16 KB, exchange records of 16 KB
  for (int r = 0; r < n; ++r) pl.smem_range[r] = pl.smem;
  const int nch = balanced_chunks((long)B * H * pl.nqg, L1, 256, least_rows(L2));
  pl.rows_per_chunk = (L1 + nch - 1) / nch;
  pl.nchunks = (L1 + pl.rows_per_chunk - 1) / pl.rows_per_chunk;
  return true;
}

bool plan_dq1(int B, int H, int L1, int L2, int row, int D, Dq1Plan& pl) {
  if (D != 32 && D != 64) return false;
  pl.wide = D == 64 && plan_dq1w(B, H, L1, L2, row, pl);
  if (pl.wide) return true;
  // D = 64: the tiles end at the row's next multiple of 32 keys, whatever length dK/dV takes (that ends with the same
  // group of 128 queries, so the aux it reads is all written).  257 to 288 keys stay at two ranges of
  // 160, as 128 keys are less than the shortest instance.  Training step, before -> now: 150 keys 109 -> 90 us (8 -> 5 tiles),
  // 200 keys 128 -> 123 (8 -> 7), 2x4 heads of 400 keys 1635 -> 1580 (2 x 8 -> 7 + 6).  D = 32 pairs its slabs: 64 keys.
  if (D == 64 && row > 128) L2 = (row > 256 && row <= 288) ? 320 : (row + 31) / 32 * 32;
  pl.Lt = L2;
  if (L2 % (D == 64 ? 32 : 64) != 0 || L2 < (D == 64 ? 160 : 256) || L2 > (D == 64 ? 256 : 512) * kMaxRanges) return false;
  pl.nlaunch = dq1_ranges(L2, D, pl.range);
  pl.threads = 256;
  pl.ring = (D == 64) ? 3 : 4;  // as compiled into the kernel
  pl.nb = pl.ring / 2;
  pl.smem = 0;
  pl.SK = dq1_slabs(L2, D);
  pl.QB = 4 / pl.SK;
  pl.nqg = (L2 + 32 * pl.QB - 1) / (32 * pl.QB);
  pl.KR = pl.range[0];
  for (int n = 0; n < pl.nlaunch; ++n) {
    const int nkt = pl.range[n] / (32 * pl.SK), ts = (nkt + 1) / 2;  // tiles of a slab's first stage
    const size_t slot = (size_t)2 * pl.SK * (ts * 32) * D * 2;
    const size_t qbuf = ((size_t)2 * pl.QB * 32 * D) * 2;
    const size_t xchg = (pl.SK == 2) ? (size_t)4 * (4 * (4 * (D / 32) / 2)) * 64 * 4 : 0;
    pl.smem_range[n] = pl.ring * slot + pl.nb * qbuf + xchg;
    if (pl.smem_range[n] > 160 * 1024) return false;
    if (pl.smem_range[n] > pl.smem) pl.smem = pl.smem_range[n];
  }
  // every launch cuts L1 into the same chunks (the dBias partial sums are indexed by chunk)
  // (one workgroup per CU; short rows in chunks of fewer rows where eight would leave CUs idle, as in dK/dV: B1 H4 of 150 keys
  // at D = 64 240 workgroups instead of 152, 200 keys 232 instead of 200: at D = 32 80.3 -> 79.4 us a training step)
  const int nch = balanced_chunks((long)B * H * pl.nqg, L1, 256, least_rows(L2));
  pl.rows_per_chunk = (L1 + nch - 1) / nch;
  pl.nchunks = (L1 + pl.rows_per_chunk - 1) / pl.rows_per_chunk;
  return true;
}

hipError_t launch_dq1(BwdParams p, const Dq1Plan& pl, int D, int dtype, bool hilo, bool nat, hipStream_t st) {
  p.nchunks = pl.nchunks; p.rows_per_chunk = pl.rows_per_chunk;
  p.ring = pl.ring; p.nb = pl.nb;
  p.SK = pl.SK; p.QB = pl.QB; p.nqg = pl.nqg; p.Lt = pl.Lt;
  const dim3 grid((unsigned)(p.B * p.H * pl.nqg * pl.nchunks));
  p.kr0 = 0;
  for (int n = 0; n < pl.nlaunch; ++n) {
    hipError_t e = hipErrorInvalidConfiguration;
    if (pl.wide) e = dtype == kBF16 ? launch_dq1w_bf16(p, pl.range[n], grid, pl.smem, st) : launch_dq1w_range<F16>(p, pl.range[n], grid, pl.smem, st);
    else
    // (nat: the caller asks for it at D = 32 with fp16 tensors only)
    if (nat) e = (dtype == kF16 && D == 32) ? launch_dq1_range<F16, 32, true, true>(p, pl.range[n], grid, pl.smem_range[n], st) : e;
    else if (dtype == kBF16) e = launch_dq1_bf16(p, pl.range[n], D, hilo, grid, pl.smem_range[n], st);
    else if (D == 64) e = launch_dq1_range<F16, 64, false, false>(p, pl.range[n], grid, pl.smem_range[n], st);
    else e = launch_dq1_range<F16, 32, false, false>(p, pl.range[n], grid, pl.smem_range[n], st);
    if (e != hipSuccess) return e;
    p.kr0 += pl.range[n];
  }
  return hipSuccess;
}

}  // namespace fta
