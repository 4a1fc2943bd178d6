// Backward: the instances of the general kernels (fta_bwd_kernels.h).  They run for dropout, for bf16 inputs and the precise
// mode of fp16 where the hand-scheduled kernels have no instances (plan_bwd knows), and in tests; dK/dV has 64
// queries per staged tile, or 32 (D = 64).
//
// Dropout is bound by the vector ALU (the mask alone is two generator calls and 16 compares per tile and lane), so what
// counts is instructions per score and that all four SIMDs of a CU have two waves.  B1 H4 L300 D32 bf16, dropout 0.25:
// dQ/dBias 223 us with three slabs of 128 keys (six waves) and 1/(1 - p) multiplied in per score, 161 with four slabs
// of 96 and the factor in the row constants; dK/dV 256 us with three slabs of 128 queries, each keep byte fetched from the
// lane that made it, 145 with two slabs of 192 and the bytes of a key group transposed once per tile.  With the geometry
// fixed at compile time where eight waves share the row: training passes of 386 to 325 us there (dQ/dBias 118), 350 to 299
// at B2 H4 L256 and 2.41 to 2.18 ms at B1 H8 L512 (dK/dV alone).
//
// Rows of 257 to 512 keys run in workgroups of four waves (dQ/dBias up to 384 keys, see plan_any_size: one query block in four
// slabs; dK/dV: two key blocks in two), two to a CU, whose priorities change in turns (see fta_fwd1_kernel): one's products and waits run beside the other's vector part, where eight waves of one
// workgroup meet at every stage, and a row's last group is at most one block short.  K and V, or Q and dO, are copied into LDS twice
// as often for it.  Training steps at B1 H4, us, before and after: L270 284 / 242, L300 in bf16 318 / 274, L330 372 / 337, L384 436 / 402, L400 787 / 735,
// L512 in bf16 1073 / 1020, B4 H8 L300 2262 / 2060; without the turns L300 302, L384 443.
#include "fta_bwd_kernels.h"

namespace fta {

hipError_t launch_dbias_reduce(const BwdParams& p, int dtype, hipStream_t st) {
  const int in_bh = p.L2 * ((p.L2 + 3) / 4);
  // shares of at least four chunks, until there are two waves for every SIMD
  int split = 1;
  while (split < 8 && (int64_t)p.B * p.H * in_bh * split < 2048 * 64 && p.nchunks >= 8 * split) split *= 2;
  const int per_bh = (in_bh + 256 / split - 1) / (256 / split);
  const dim3 grid((unsigned)(p.B * p.H * per_bh)), block(256);
  if (dtype == kBF16) hipLaunchKernelGGL(fta_dbias_reduce_kernel<BF16>, grid, block, 0, st, p, split, per_bh);
  else hipLaunchKernelGGL(fta_dbias_reduce_kernel<F16>, grid, block, 0, st, p, split, per_bh);
  return hipGetLastError();
}

template <class T, bool DROP>
static hipError_t bwd_feat_t(BwdParams p, const BwdPlan& pl, int D, hipStream_t st, hipEvent_t* ev) {
  auto mark = [&](int i) { if (ev != nullptr) (void)hipEventRecord(ev[i], st); };
  hipError_t e = hipSuccess;
  if (!pl.own_delta) {  // 0. delta and the {lse, delta} pairs
    const int64_t nthr = (int64_t)p.B * p.H * p.L1 * p.L2p * (D / 8);
    dim3 grid((unsigned)((nthr + 255) / 256)), block(256);
    if (D == 32) hipLaunchKernelGGL((fta_bwd_delta_kernel<T, 32>), grid, block, 0, st, p);
    else hipLaunchKernelGGL((fta_bwd_delta_kernel<T, 64>), grid, block, 0, st, p);
    if ((e = hipGetLastError()) != hipSuccess) return e;
  }
  mark(1);
  {  // 1. dQ, dBias partials
    dim3 grid((unsigned)(p.B * p.H * pl.nqg * pl.nchunks)), block((unsigned)pl.threads);
    if (pl.nranges > 0) {
      if constexpr (DROP)
        for (int n = 0, at = 0; n < pl.nranges; at += pl.range[n++]) {
          const DropRange r = drop_range(pl.range[n]);
          p.kr0 = at; p.ring = r.dq.r; p.nb = r.dq.nb;
          e = pl.range[n] == 512   ? launch_kernel(fta_bwd_dq_kernel<T, true, 32, 2>, p, grid, block, r.smem, st)
              : pl.range[n] == 384 ? launch_kernel(fta_bwd_dq_kernel<T, true, 32, 1, 3, 4>, p, grid, block, r.smem, st)
              : pl.range[n] == 256 ? launch_kernel(fta_bwd_dq_kernel<T, true, 32, 1, 2, 4>, p, grid, block, r.smem, st)
                                   : hipErrorInvalidConfiguration;
          if (e != hipSuccess) return e;
        }
    }
    for (int n = 0; n < (pl.nranges > 0 ? 0 : pl.nlaunch); ++n) {
      p.kr0 = n * pl.KR;
      e = hipErrorInvalidConfiguration;
      if (pl.own_delta) {  // key ranges of 384 keys with dropout: fixed geometry
        if constexpr (DROP)
          if (D == 32 && pl.NKT == 3 && pl.threads == 256 && pl.SK == 4 && pl.ring == dq_ring(32, 3, 1, 4, 4).r && pl.nb == dq_ring(32, 3, 1, 4, 4).nb)
            e = launch_kernel(fta_bwd_dq_kernel<T, true, 32, 1, 3, 4, 4>, p, grid, block, pl.smem, st);
      } else if (D == 32) {
        e = launch_kernel(fta_bwd_dq_kernel<T, DROP, 32, 2>, p, grid, block, pl.smem, st);
      } else {
        e = launch_kernel(fta_bwd_dq_kernel<T, DROP, 64, 1>, p, grid, block, pl.smem, st);
      }
      if (e != hipSuccess) return e;
    }
    p.kr0 = 0;
  }
  mark(2);
  {  // 2. dK, dV
    dim3 grid((unsigned)(p.B * p.H * pl.nkg * pl.nchunks2)), block((unsigned)pl.threads2);
    if (pl.nranges2 > 0) {
      if constexpr (DROP)
        for (int n = 0, at = 0; n < pl.nranges2; at += pl.range[n++]) {
          const DropRange r = drop_range(pl.range[n]);
          p.jr0 = at;
          e = pl.range[n] == 512   ? launch_kernel(fta_bwd_dkdv_kernel<T, true, 32, 8, 64, 2>, p, grid, block, r.smem2, st)
              : pl.range[n] == 384 ? launch_kernel(fta_bwd_dkdv_kernel<T, true, 32, 6, 64, 2>, p, grid, block, r.smem2, st)
              : pl.range[n] == 256 ? launch_kernel(fta_bwd_dkdv_kernel<T, true, 32, 4, 64, 2>, p, grid, block, r.smem2, st)
                                   : hipErrorInvalidConfiguration;
          if (e != hipSuccess) return e;
        }
    }
    for (int n = 0; n < (pl.nranges2 > 0 ? 0 : pl.nlaunch2); ++n) {
      p.jr0 = n * pl.JR;
      e = hipErrorInvalidConfiguration;
#define FTA_DKDV_FEAT_CASE(DD, NN, JJ) \
  if (e == hipErrorInvalidConfiguration && D == DD && pl.NJT == NN && pl.JT == JJ) \
    e = launch_kernel(fta_bwd_dkdv_kernel<T, DROP, DD, NN, JJ>, p, grid, block, pl.smem2, st);
      // fixed geometry: 384, 512, 768 and 1024 queries to a launch.  (Rows of up to 256 queries at D = 32 run the one-kernel
      // backward; <8, 64, 1> and <4, 64> are theirs where fta_debug_select_kernels asks for the general kernels)
      if constexpr (DROP) {
#define FTA_DKDV_FIX_CASE(NN, JJ, SS, WW)                                                                                        \
  if (D == 32 && pl.threads2 == 64 * WW && pl.NJT == NN && pl.JT == JJ && pl.SJ == SS && pl.ring2 == dkdv_ring(32, NN, JJ, SS, WW).r && \
      pl.nb2 == dkdv_ring(32, NN, JJ, SS, WW).nb)                                                                                \
    e = launch_kernel(fta_bwd_dkdv_kernel<T, true, 32, NN, JJ, SS, WW>, p, grid, block, pl.smem2, st);
        FTA_DKDV_FIX_CASE(5, 32, 2, 4) FTA_DKDV_FIX_CASE(6, 64, 2, 4) FTA_DKDV_FIX_CASE(8, 64, 1, 8) FTA_DKDV_FIX_CASE(8, 64, 2, 4)
        FTA_DKDV_FIX_CASE(6, 64, 4, 8) FTA_DKDV_FIX_CASE(8, 64, 4, 8)
#undef FTA_DKDV_FIX_CASE
      }
      if constexpr (!DROP) { FTA_DKDV_FEAT_CASE(32, 8, 64) }
      FTA_DKDV_FEAT_CASE(32, 4, 64)
      FTA_DKDV_FEAT_CASE(64, 4, 64) FTA_DKDV_FEAT_CASE(64, 4, 32)
#undef FTA_DKDV_FEAT_CASE
      if (e != hipSuccess) return e;
    }
    p.jr0 = 0;
  }
  mark(3);
  e = launch_dbias_reduce(p, T::is_bf16 ? kBF16 : kF16, st);  // 3. sums the chunk partials
  mark(4);
  return e;
}

hipError_t launch_bwd_feat(const BwdParams& p, const BwdPlan& pl, int D, int dtype, hipStream_t st, hipEvent_t* ev) {
  const bool drop = p.drop.thresh != 0;
  if (dtype == kF16) return drop ? bwd_feat_t<F16, true>(p, pl, D, st, ev) : bwd_feat_t<F16, false>(p, pl, D, st, ev);
  if (drop) return bwd_feat_t<BF16, true>(p, pl, D, st, ev);
  return bwd_feat_t<BF16, false>(p, pl, D, st, ev);
}

}  // namespace fta
