// Backward: the launch plan and the dispatch of the stages.  Rows of up to 128 keys (D = 32: 192, with dropout 256) run the one-kernel form
// (fta_bwd_short.hip), longer ones the hand-scheduled kernels (fta_bwd_dq1.hip, fta_bwd_dkdv1.hip) or the general ones
// (fta_bwd_kernels.h, instances in fta_bwd_feat.hip).
#include <stdlib.h>

#include "fta_bwd_kernels.h"

namespace fta {

// ------------------------------------------------------------------------------------------------
// host side
// ------------------------------------------------------------------------------------------------
static BwdPlan plan_any_size(int B, int H, int L1, int L2, int D, int row, int feat) {
  BwdPlan pl{};
  pl.feat = feat != 0;
  pl.use_short = !forced_general() && plan_short(B, H, L1, row, D, feat, pl.sh);
  // (the two go together: the pipelined dQ kernel makes delta itself and hands the row constants on to the dK/dV one in
  // the packed form that only that one reads)
  // Their tiles end at the next multiple of 64 keys: the work grows with the square of that length.  A training step at B1
  // H4 D32 in fp16, tiles to the next multiple of 128 and key ranges of 512 + 256 -> this (us): L 257
  // 160 -> 143, 320 194 -> 169, 385 366 -> 328, 448 435 -> 395, 513 985 -> 886, 576 1114 -> 996, 704 1859 -> 1716, 1281
  // 11160 -> 10380.
  auto hand = [&](int lt) { pl.Lt = lt; return plan_dq1(B, H, L1, lt, row, D, pl.dq1) && plan_dkdv1(B, H, L1, lt, D, pl.dkdv1); };
  pl.use_hand = !pl.use_short && !feat && !forced_general() && (hand((row + 63) / 64 * 64) || hand(L2));
  if (pl.use_short || pl.use_hand) {
    pl.partial_bytes = (size_t)(pl.use_short ? pl.sh.nchunks : pl.dq1.nchunks) * B * H * L2 * L2 * sizeof(float);
    pl.aux_bytes = pl.use_short ? 0 : (size_t)B * H * L1 * L2 * 2 * sizeof(uint32_t);
    pl.valid = true;
    return pl;
  }
  // Dropout at D = 32 beyond 512 keys: key and query ranges of 256, 384 and 512, as even as the row divides, every one by
  // eight waves (four slabs of 64, 96 or 128 keys; two of 128, 192 or 256 queries).  Cut into the widest equal pieces that
  // divide the row, 640 keys take five launches of 128: steps at B1 H4 in bf16 of 576, 640, 896 and 1280 keys that way and as
  // below 3.09 / 1.85, 3.46 / 2.18, 7.54 / 5.65, 18.4 / 16.6 ms.
  // Longer rows at B1 H1: 1408 9.45 / 5.88, 1664 15.7 / 9.43, 1792 12.3 / 11.3, 2176 38.7 / 26.0, 2304 36.8 / 32.3, 3328 103 / 99.3, 3840 166 / 148,
  // 1152, 2560 and 4096 equal.  Five, seven and nine times 384 keys are the exception: in ranges of 384 dQ/dBias takes 2.67 us a key
  // at 1920, in ranges of 512, whose geometry comes from the arguments (known at compile time it spills), 3.03 (dK/dV 2.73 and 2.65), and a
  // step 1 to 4 % longer (1920 19.7 / 20.0, 2688 45.5 / 46.4, 3456 112 / 116); but dQ, too, is held in the tensors' type between launches,
  // and those are one or two fewer here.
  // dK and dV are held in the tensors' type from one query range to the next, a rounding at each.  So dK/dV takes rows that
  // 768 or 1024 divides in launches of as many queries, four slabs of 192 or 256: of 768, 1024, 2048, 2304 and
  // 3072 queries its relative error in bf16 is 2.37, 2.36, 2.64, 2.88 and 2.88e-3, in ranges of up to 512 2.65, 2.63, 3.11,
  // 3.40 and 3.53e-3; the steps are 1 to 3 % longer (768 3.60 / 3.53 ms, 1024 9.46 / 9.38, 1536 29.6 / 28.9, 2048 85.4 / 83.9).
  if (feat == 2 && D == 32 && L2 > 512 && L2 % 128 == 0 && L2 <= 512 * kMaxRanges) {
    pl.nranges = pl.nranges2 = even_ranges(L2 / 128, 4, 128, pl.range);
    const int nblk = (row + 31) / 32, sk = 4, qb = 2;
    int sj = 2, kb = 4;
    pl.NKT = pl.range[0] / 128; pl.SK = sk; pl.QB = qb; pl.KR = pl.range[0]; pl.nlaunch = pl.nranges;
    pl.NJT = pl.range[0] / 64; pl.JT = 64; pl.JR = pl.range[0]; pl.nlaunch2 = pl.nranges;
    for (int n = 0; n < pl.nranges; ++n) {
      const DropRange r = drop_range(pl.range[n]);
      if (r.smem > pl.smem) pl.smem = r.smem;
      if (r.smem2 > pl.smem2) pl.smem2 = r.smem2;
    }
    const int wide = L2 % 1024 == 0 ? 1024 : L2 % 768 == 0 ? 768 : 0;
    if (wide != 0) {
      const Ring r = dkdv_ring(32, wide / 128, 64, 4, 8);
      sj = 4; kb = 2;
      pl.nranges2 = 0; pl.NJT = wide / 128; pl.JR = wide; pl.nlaunch2 = L2 / wide;
      pl.ring2 = r.r; pl.nb2 = r.nb; pl.smem2 = dkdv_smem(32, pl.NJT, 64, 4, 8);
    }
    pl.SJ = sj; pl.KB = kb;
    pl.threads = pl.threads2 = 512;
    pl.nqg = (nblk + qb - 1) / qb;
    pl.nkg = (nblk + kb - 1) / kb;
    const int nch = balanced_chunks((long)B * H * pl.nqg, L1, 256), nch2 = balanced_chunks((long)B * H * pl.nkg, L1, 256);
    pl.rows_per_chunk = (L1 + nch - 1) / nch;
    pl.nchunks = (L1 + pl.rows_per_chunk - 1) / pl.rows_per_chunk;
    pl.rows_per_chunk2 = (L1 + nch2 - 1) / nch2;
    pl.nchunks2 = (L1 + pl.rows_per_chunk2 - 1) / pl.rows_per_chunk2;
    pl.delta_bytes = (size_t)B * H * L1 * L2 * sizeof(float);
    pl.partial_bytes = (size_t)pl.nchunks * B * H * L2 * L2 * sizeof(float);
    pl.aux_bytes = (size_t)B * H * L1 * L2 * 2 * sizeof(uint32_t);
    pl.valid = true;
    return pl;
  }
  const int nqb = L2 / 32;
  const size_t lds_max = 160 * 1024;
  // ---- dQ/dBias kernel: key range of at most 512 keys per launch, 128-key slabs
  int kr = 0;
  for (int c = 512; c >= 128; c -= 128)
    if (L2 % c == 0) { kr = c; break; }
  pl.KR = kr;
  pl.nlaunch = L2 / kr;
  // Dropout at D = 32, key ranges of 384 keys: four slabs of 96 keys instead of three of 128, so that the four SIMDs of a CU have
  // as many waves each, and the query (key) blocks that hold nothing of the row have no workgroup.  These are
  // workgroups of four waves, two to a CU (see fta_bwd_feat.hip).  Four slabs of 128 keys stay in one workgroup of eight: its stages of 64
  // keys leave no LDS for a second, and in stages of 32 keys four waves took longer (us a training step, four / eight waves in dQ/dBias:
  // B1 H4 L400 738 / 735, L450 in bf16 953 / 931, L512 in bf16 1048 / 1020, B2 H8 L420 in bf16 2957 / 2885, B4 H8 L512 8152 / 8047).
  const bool three = (feat == 2 && D == 32 && kr == 384);
  const int nblk = (feat == 2) ? (row + 31) / 32 : nqb;
  pl.NKT = three ? 3 : 4;
  pl.own_delta = three;
  pl.SK = kr / (32 * pl.NKT);
  int qb = (three ? 4 : 8) / pl.SK;
  if (qb < 1) qb = 1;
  while (qb > 1 && nqb % qb != 0) --qb;
  pl.QB = qb;
  pl.nqg = (nblk + qb - 1) / qb;
  pl.threads = 64 * pl.SK * pl.QB;
  const int G1 = (D == 32 && !three) ? 2 : 1;
  const int stage_rows = pl.SK * G1 * 32;
  const size_t slot1 = (size_t)2 * stage_rows * D * 2;
  const int steps1 = pl.NKT / G1;
  const size_t part1 = dq_records(D, pl.SK, pl.threads / 64);
  const size_t qtile1 = (size_t)2 * pl.QB * 32 * D * 2;  // Q and dO rows of the workgroup, one L1 row
  pl.ring = 0;
  for (int r = 4; r >= 3; --r) {
    const int nb = (r + steps1 - 1) / steps1;  // rows whose operand tiles can be in flight at once
    if (r * slot1 + nb * qtile1 + part1 <= lds_max / (three ? 2 : 1)) { pl.ring = r; pl.nb = nb; pl.smem = r * slot1 + nb * qtile1 + part1; break; }
  }
  pl.nchunks = balanced_chunks((long)B * H * pl.nqg, L1, three ? 512 : 256, least_rows(L2));
  pl.rows_per_chunk = (L1 + pl.nchunks - 1) / pl.nchunks;
  pl.nchunks = (L1 + pl.rows_per_chunk - 1) / pl.rows_per_chunk;
  // ---- dK/dV kernel: query slabs of at most 256 (D=32) / 128 (D=64) queries per wave (register
  // budget); up to SJ slabs share a workgroup, longer rows take several launches over query ranges
  // (the dropout instances with 256 queries per wave touch scratch memory twice per row; with 128, which halves the reuse of a
  // workgroup's K/V rows, a step took 4 % longer, also when the former spilled 42 registers)
  const int jwmax = (D == 32) ? 256 : 128;
  int jw = 0;
  for (int c = jwmax; c >= 128; c -= 128)
    if (L2 % c == 0) { jw = c; break; }
  // (dropout, lengths that three slabs of 128 queries would cut: two slabs of 192, as many waves for every SIMD)
  const bool two192 = (feat == 2 && D == 32 && jw == 128 && L2 % 384 == 0);
  if (two192) jw = row <= 320 ? 160 : 192;
  pl.NJT = jw / 32;
  const int nslab = two192 ? 2 : L2 / jw;
  const int sjmax = two192 ? 2 : 4;
  bool ok2 = false;
  for (int sj = (nslab < sjmax ? nslab : sjmax); sj >= 1 && !ok2; --sj) {
    if (nslab % sj != 0) continue;
    const bool four2 = (feat == 2 && D == 32 && sj == 2 && jw >= 160);
    int kb = (four2 ? 4 : 8) / sj;
    if (kb < 1) continue;
    while (kb > 1 && nqb % kb != 0) --kb;
    for (int jt = 64; jt >= 32 && !ok2; jt /= 2) {
      if (jw % jt != 0) continue;  // (160 queries: stages of 32)
      const int stage_rows2 = sj * jt;
      const size_t slot2 = (size_t)2 * stage_rows2 * D * 2 + (size_t)2 * stage_rows2 * 4;
      const size_t scratch2 = dkdv_shares(D, sj, sj * kb);
      const size_t ktile2 = (size_t)2 * kb * 32 * D * 2;  // K and V rows of the workgroup, one L1 row
      const int steps2 = (jw / 32) / (jt / 32);
      for (int r = 4; r >= 3 && !ok2; --r) {
        const int nb = (r + steps2 - 1) / steps2;
        if (r * slot2 + nb * ktile2 + scratch2 > lds_max / (four2 ? 2 : 1)) continue;
        pl.SJ = sj; pl.KB = kb; pl.nkg = (nblk + kb - 1) / kb; pl.threads2 = 64 * sj * kb; pl.JT = jt;
        pl.ring2 = r; pl.nb2 = nb; pl.smem2 = r * slot2 + nb * ktile2 + scratch2;
        pl.JR = sj * jw; pl.nlaunch2 = two192 ? 1 : L2 / pl.JR;
        ok2 = true;
      }
    }
  }
  pl.nchunks2 = balanced_chunks((long)B * H * (ok2 ? pl.nkg : 1), L1, feat == 2 && D == 32 && pl.threads2 == 256 ? 512 : 256, least_rows(L2));
  pl.rows_per_chunk2 = (L1 + pl.nchunks2 - 1) / pl.nchunks2;
  pl.nchunks2 = (L1 + pl.rows_per_chunk2 - 1) / pl.rows_per_chunk2;

  pl.delta_bytes = pl.own_delta ? 0 : (size_t)B * H * L1 * L2 * sizeof(float);
  pl.partial_bytes = (size_t)pl.nchunks * B * H * L2 * L2 * sizeof(float);
  pl.aux_bytes = (size_t)B * H * L1 * L2 * 2 * sizeof(uint32_t);
  pl.valid = ok2 && (pl.SK * pl.QB <= 8) && (pl.ring >= 3);
  return pl;
}

BwdPlan plan_bwd(int B, int H, int L1, int L2, int D, int row, int feat, size_t limit) {
  BwdPlan pl = plan_any_size(B, H, L1, L2, D, row, feat);
  if (!pl.valid || limit == 0 || pl.delta_bytes + pl.partial_bytes + pl.aux_bytes <= limit) return pl;
  // The chunks are as many as make the launch shortest, and each has a partial dBias of its own: as many as fit instead.
  int& nch = pl.use_short ? pl.sh.nchunks : pl.use_hand ? pl.dq1.nchunks : pl.nchunks;
  int& rows = pl.use_short ? pl.sh.rows_per_chunk : pl.use_hand ? pl.dq1.rows_per_chunk : pl.rows_per_chunk;
  const size_t one = pl.partial_bytes / nch, rest = pl.delta_bytes + pl.aux_bytes;
  if (rest + one > limit) return pl;
  const int most = (int)((limit - rest) / one);
  rows = (L1 + most - 1) / most;
  nch = (L1 + rows - 1) / rows;
  pl.partial_bytes = nch * one;
  return pl;
}

hipError_t launch_bwd(BwdParams p, const BwdPlan& pl, int D, int dtype, hipStream_t st, hipEvent_t* ev) {
  // ev (optional, 5 events): recorded before stage 0 and after each of the four stages
  auto mark = [&](int i) { if (ev != nullptr) (void)hipEventRecord(ev[i], st); };
  p.SK = pl.SK; p.QB = pl.QB; p.nqg = pl.nqg; p.nchunks = pl.nchunks; p.rows_per_chunk = pl.rows_per_chunk;
  p.ring = pl.ring; p.ring2 = pl.ring2; p.nb = pl.nb; p.nb2 = pl.nb2;
  p.SJ = pl.SJ; p.KB = pl.KB; p.nkg = pl.nkg; p.nchunks2 = pl.nchunks2; p.rows_per_chunk2 = pl.rows_per_chunk2;
  p.partial_scale = 1.0f;
  hipError_t e = hipSuccess;
  mark(0);
  if (pl.use_short) {
    // short rows, any options: one kernel
    mark(1);
    e = launch_short(p, pl.sh, D, dtype, pl.feat, st);  // (fp16 without dropout is planned at that level in precise mode only)
    if (e != hipSuccess) return e;
    p.nchunks = pl.sh.nchunks;
    mark(2);
    mark(3);
    e = launch_dbias_reduce(p, dtype, st);
    mark(4);
    return e;
  }
  if (!pl.use_hand) return launch_bwd_feat(p, pl, D, dtype, st, ev);
  if (p.drop.thresh != 0) return hipErrorInvalidConfiguration;  // (planned with other options)
  // The hand-scheduled kernels: fp16, its precise mode at D = 32, bf16.  bf16 at scales whose product with Q (and K),
  // rounded to 8 bits, would show in the gradients runs the instances that carry the product as a (hi, lo) pair.
  const bool nat = (p.nat != 0);
  const bool hilo = (dtype == kBF16 && bf16_scale_needs_split(p.scale)) || nat;
  mark(1);
  // 1. delta and the packed row constants, dQ, dBias partials (one launch per key range; later ranges accumulate into dQ)
  e = launch_dq1(p, pl.dq1, D, dtype, hilo, nat, st);
  if (e != hipSuccess) return e;
  p.nchunks = pl.dq1.nchunks;  // the reduction sums this many partial tiles
  mark(2);
  // 2. dK, dV
  e = launch_dkdv1(p, pl.dkdv1, D, dtype, hilo, nat, st);
  if (e != hipSuccess) return e;
  mark(3);
  // 3. dBias: sum the chunk partials
  if (dtype == kBF16) p.partial_scale = BF16::kOneHotInv;
  e = launch_dbias_reduce(p, dtype, st);
  mark(4);
  return e;
}

}  // namespace fta
