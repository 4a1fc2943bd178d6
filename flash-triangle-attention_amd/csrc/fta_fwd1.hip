// Forward, hand-scheduled (D = 32): the launch plan and the instances for rows of one key slab (fta_fwd1_kernel.h; those
// for several slabs are compiled in fta_fwd1_slabs.hip).
#include "fta_fwd1_kernel.h"

namespace fta {

// ---- host side ---------------------------------------------------------------------------------

bool plan_fwd1(int B, int H, int L1, int L2, int D, int row, bool scattered, FwdPlan& pl) {
  if (D != 32 || L2 % 32 != 0 || L2 < 64 || L2 == 96 || L2 > 1792) return false;
  pl = FwdPlan{};
  // rows beyond 512 keys in two slabs, beyond 1024 in four (three would leave two of the four SIMDs with one wave);
  // four slabs of 512 keys have no registers left for the ends of rows.  Any number of tiles per slab: with even ones alone
  // (bf16, B1 H4, us) L160 14.7 against 12.8 with five, L288 39.9 / 36.8, L416 90 / 85, L576 246 / 228, L701 420 / 396, L960
  // 929 / 888, L1152 1738 / 1625, L1601 4750 / 4500
  pl.S = L2 <= 512 ? 1 : L2 <= 1024 ? 2 : 4;
  if (L2 % (32 * pl.S) != 0) return false;
  pl.NKT = L2 / (32 * pl.S);
  // four waves per workgroup, two workgroups to a CU (see the kernel's comment); eight where a query block's keys are four slabs; rows of up to
  // 64 queries have two query blocks.  256 keys that do not lie next to each other in memory (heads
  // interleaved, or a transposed view: half a line each): the eight query blocks of a row in one workgroup, where such workgroups fill the chip, so that half as
  // many ask for a line (bf16, inputs not in the caches, us, four / eight waves: heads interleaved B2 H4 46.9 / 45.6, B4 H8 167.8 / 163.5, 240 keys
  // 154.5 / 153.3, transposed 164.1 / 161.9, a training pass 696 / 694; with inputs that stay in the caches equal at 256, 141 / 145 at 240;
  // contiguous B2 H4 42.0 / 42.4, B4 H8 146 / 150; 512 keys, heads interleaved, 1033 / 1069)
  // Two slabs of such keys, where four query blocks to a workgroup leave no more of them empty than two: the same (us, two / four query blocks:
  // transposed B1 H4 L640 294 / 292, L1024 1070 / 1046, heads interleaved L768 477 / 475, B2 H8 L890 2999 / 2963; L900 862 / 882, L960 944 / 954, contiguous
  // L640 1128 / 1138; with inputs that stay in the caches L640 286 / 296, L1024 999 / 1080).
  const int nblk = (row + 31) / 32;
  const bool four_blocks = scattered && L2 % 128 == 0 && nblk % 4 == 0;
  const bool row_of_eight = L2 == 256 && scattered && (long)B * H * ((L1 + 7) / 8) >= 256;
  pl.QB = pl.S == 2 && four_blocks ? 4 : pl.S > 1 || L2 <= 64 ? 2 : row_of_eight ? 8 : 4;
  pl.nqg = (row + 32 * pl.QB - 1) / (32 * pl.QB);
  pl.threads = 64 * pl.QB * pl.S;
  pl.KT = (L2 <= 64 || pl.S > 1) ? 64 : 128;
  pl.smem = (size_t)4 * 2 * pl.S * pl.KT * 32 * 2;  // four slots of a K and a V tile of KT keys per slab
  if (pl.S > 1) pl.smem += pl.S == 4 ? 8 * (3072 + 512) + 1024 : pl.S * pl.QB * (2048 + 512);  // the merge records
  pl.alias_scratch = 0;
  // two waves per SIMD: one, two or four workgroups per CU.  At least a row per 64 keys in a chunk: a workgroup's set-up
  // loads one bias row per query, so short rows can be spread thinner (B1 H4 L64: 14.9 us with 8 rows, 5 with 1)
  const int nch = balanced_chunks((long)B * H * pl.nqg, L1, 256 * 8 / (pl.QB * pl.S), pl.S > 1 ? 8 : L2 <= 64 ? 1 : L2 / 64);
  pl.rows_per_chunk = (L1 + nch - 1) / nch;
  pl.nchunks = (L1 + pl.rows_per_chunk - 1) / pl.rows_per_chunk;
  pl.fwd1 = 1;
  pl.valid = true;
  return true;
}

hipError_t launch_fwd1(const FwdParams& p, const FwdPlan& pl, int dtype, dim3 grid, dim3 block, hipStream_t st) {
  const bool tl = (p.L2 % (32 * pl.QB) != 0) || p.L2 != 32 * pl.NKT * pl.S || p.odd_bias;  // (the instances that mask a row's tail also read the bias entry by entry where they must)
  FTA_FWD1_CASE(2, 2, 2, 1)
  FTA_FWD1_CASE(5, 4, 4, 1) FTA_FWD1_CASE(7, 4, 4, 1) FTA_FWD1_CASE(9, 4, 4, 1) FTA_FWD1_CASE(11, 4, 4, 1)
  FTA_FWD1_CASE(13, 4, 4, 1) FTA_FWD1_CASE(15, 4, 4, 1)
  FTA_FWD1_CASE(4, 4, 4, 1) FTA_FWD1_CASE(6, 4, 4, 1) FTA_FWD1_CASE(8, 4, 4, 1) FTA_FWD1_CASE(10, 4, 4, 1)
  FTA_FWD1_CASE(8, 8, 4, 1)
  FTA_FWD1_CASE(12, 4, 4, 1) FTA_FWD1_CASE(14, 4, 4, 1) FTA_FWD1_CASE(16, 4, 4, 1)
  return launch_fwd1_slabs(p, pl, dtype, tl, grid, block, st);
}

}  // namespace fta
