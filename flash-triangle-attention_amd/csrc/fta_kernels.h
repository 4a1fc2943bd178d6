// Kernel parameter blocks and launch plans shared by the kernels and the C-ABI layer.
#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>
#include <stdlib.h>

namespace fta {

typedef _Float16 half_t;

// Dropout on the attention weights.  Weight (b,h,i,j,k) is kept iff its random byte is >= thresh, so
// the keep probability is (256 - thresh)/256 and kept weights are scaled by 256/(256 - thresh).
struct DropParams {
  uint32_t seed_lo, seed_hi;
  uint32_t thresh;   // round(256 * p), 0..255; 0 = no dropout
  float scale;       // 256 / (256 - thresh)
};

enum ElemType { kF16 = 0, kBF16 = 1 };

struct FwdParams {
  const half_t* q; const half_t* k; const half_t* v; const half_t* bias;
  half_t* o; float* lse;
  int64_t qs[4], ks[4], vs[4], os[4];  // element strides (b,h,l1,l2)
  int64_t bs[3];                       // bias strides (b,h,j)
  int B, H, L1, L2;    // L2: the true row length
  int L2p;             // the length the tiles cover: the next supported multiple of 128 (== L2 where that is one)
  int odd_bias;        // bias rows may start off an 8-byte boundary (strides that are not multiples of 4): the bias
                       // is then read entry by entry where it must be, like the tail of a row
  int head_inner;      // the heads of a row are interleaved in memory (see work_id)
  int S;               // key slabs (waves sharing one query block)
  int QB;              // query blocks of 32 per workgroup
  int nqg;             // query groups = L2 / (32*QB)
  int nchunks;         // chunks of L1 rows
  int rows_per_chunk;
  int alias_scratch;   // the slab-merge records share an idle stage buffer (no LDS region of their own)
  float scale;
  DropParams drop;
};

struct FwdPlan {
  int NKT;             // 32-key tiles per wave slab
  int S, QB, nqg, nchunks, rows_per_chunk, threads, alias_scratch;
  int KT;              // keys per staged LDS tile (per slab)
  int L2p;             // the length the tiles cover (filled in by the C-ABI layer)
  int fwd1;            // 1: the hand-scheduled kernel of fta_fwd1_kernel.h runs (D = 32); 2: that of fta_fwd2.hip (D = 64)
  size_t smem;
  bool valid;
};

// How many chunks of L1 rows to cut a launch into: `base` workgroups exist per chunk, `slots`
// workgroups run on the chip at once (256 CUs times the workgroups of this kernel that fit a CU).
// The launch takes (rounds of workgroups) x (rows per chunk + what a workgroup spends before its
// first row: bias tile, pipeline fill, measured at about 5 rows' worth); the count that minimises
// that wins, with at least `least` rows per chunk.  (A launch of 2.25 rounds runs as long as one of 3;
// two rounds of half-length chunks lose to one round.)
inline int balanced_chunks(long base, int L1, long slots, int least = 8) {
  const int maxch = (L1 + least - 1) / least;
  int best = 1;
  long best_cost = -1;
  for (int nch = 1; nch <= maxch; ++nch) {
    const int rows = (L1 + nch - 1) / nch;
    const long chunks = (L1 + rows - 1) / rows;
    const long rounds = (base * chunks + slots - 1) / slots;
    const long cost = rounds * (rows + 5);
    if (best_cost < 0 || cost < best_cost) {
      best = nch;
      best_cost = cost;
    }
  }
  return best;
}

// The fewest rows of a chunk for rows of L2 keys: a workgroup's set-up loads one bias row per query, so that short rows
// can be spread thinner over the chip than eight to a workgroup.  B1 H4, us, eight -> this: forward at D = 64 of 48, 128, 192,
// 256, 384, 448 keys 23.8 -> 9.7, 23.6 -> 10.0, 48.4 -> 29.9, 51.2 -> 35.0, 114 -> 112, 216 -> 213; with dropout at D = 32 of
// 64, 192, 256, 384 24.1 -> 9.8, 50.4 -> 23.4, 42.2 -> 35.6, 114 -> 114; training steps at D = 32 (dK/dV) of 200, 256, 384, 448
// 92 -> 87, 98 -> 97, 256 -> 252, 402 -> 404, with dropout of 300, 384, 448 324 -> 312, 444 -> 445, 851 -> 852; at D = 64 of
// 160, 256, 384 141 -> 110, 166 -> 155, 518 -> 520, with dropout of 192, 256, 384 285 -> 217, 314 -> 284, 1205 -> 1206.  Where B * H
// fills the chip nothing changes (B4 H8 of 192, 256 and 384 keys within 0.7 %).  From 512 keys on it is eight.
inline int least_rows(int L2) { return L2 >= 512 ? 8 : L2 <= 128 ? 2 : L2 / 64; }

// ---- backward ---------------------------------------------------------------------------------

struct BwdParams {
  const half_t* q; const half_t* k; const half_t* v; const half_t* bias;
  const half_t* o; const float* lse; const half_t* dout;
  half_t* dq; half_t* dk; half_t* dv; half_t* dbias;
  float* delta;        // (B,H,L1,L2) fp32 workspace, written by the delta kernel, read by the general dQ kernel
  float* partial;      // (nchunks,B*H,L2,L2) fp32 workspace: per-chunk sums of dS over L1 rows
  uint32_t* aux;       // (B,H,L1,L2,2) workspace: the row constants lse and delta for the dK/dV kernel, as fp16 (hi,lo) splits
                       // of -lse (log2 domain) and -delta (hand-scheduled) or in fp32 (general)
  // (eight bytes that the hand-scheduled kernels do not read, in front of the strides: without them the compiler loads the
  // strides in larger pieces than it has scalar registers for, and 190 lane reads instead of 57 fetch them back in dq1)
  int dbias_f32;       // dbias is written as fp32 (B,H,L2,L2) instead of the element type
  float partial_scale; // what the reduction multiplies the summed partials by (1, or 128 behind the bf16
                       // hand-scheduled dQ/dBias kernel, whose one-hot selector is worth 2^-7: see kOneHotInv)
  int64_t qs[4], ks[4], vs[4], os[4], dos[4], dqs[4], dks[4], dvs[4];
  int64_t bs[3], dbs[3];
  int B, H, L1, L2;    // L2: the true row length; lse is (B,H,L1,L2)
  int L2p;             // the length the tiles cover (next supported multiple of 128); delta, partial and aux
                       // in the workspace are laid out with L2p
  float scale;
  // dQ/dBias kernel geometry
  int SK;              // 128-key slabs per workgroup (waves sharing one query block)
  int QB;              // query blocks of 32 per workgroup
  int nqg;             // query groups = L2 / (32*QB)
  int nchunks, rows_per_chunk;
  int kr0;             // first key of this launch's key range
  int ring;            // LDS ring slots of the K/V stage buffers
  int nb;              // LDS buffers for the per-row Q/dO tiles
  // dK/dV kernel geometry
  int SJ;              // query slabs (waves sharing one key block)
  int KB;              // key blocks of 32 per workgroup
  int nkg;             // key groups = L2 / (32*KB)
  int nchunks2, rows_per_chunk2;
  int jr0;             // first query of this launch's query range
  int ring2;           // LDS ring slots of the Q/dO stage buffers
  int nb2;             // LDS buffers for the per-row K/V tiles
  DropParams drop;
  int head_inner;      // the heads of a row are interleaved in memory (see work_id)
  int odd_bias;        // bias rows may start off an 8-byte boundary (strides that are not multiples of 4): the
                       // instances that mask a row's tail run, which read the bias entry by entry where they must
  int nat;             // (host side) the hand-scheduled backward kernels' precise instances run: exponents in
                       // natural units, scaled operands as (hi, lo) pairs
  int Lt;              // (host side) the length that the hand-scheduled kernels' tiles cover (see BwdPlan)
};


// Geometry of the one-wave-per-SIMD dK/dV kernel (a wave owns 32 keys against the launch's query range).
constexpr int kMaxRanges = 8;  // launches (key or query ranges) of a hand-scheduled backward stage: 4096 / 512
// Cuts `units` into the fewest ranges of at most `most` units, larger ones first and none more than a unit larger than
// another; the ranges, `unit` long each, go to `out` and their number is returned.
inline int even_ranges(int units, int most, int unit, int* out) {
  const int n = (units + most - 1) / most;
  for (int r = 0; r < n; ++r) out[r] = (units / n + (r < units % n ? 1 : 0)) * unit;
  return n;
}
struct Dq1Plan {
  int SK, QB, nqg, nchunks, rows_per_chunk, threads, KR, nlaunch, ring, nb;   // SK, QB, nqg, KR: of the first range
  int range[kMaxRanges];          // keys per launch
  size_t smem_range[kMaxRanges];
  size_t smem;                    // the largest
  int Lt;                         // the length its tiles cover (D = 64: the next multiple of 32 keys, `wide` of 128)
  bool wide;                      // D = 64: ranges of up to 512 keys in two slabs (fta_bwd_dq1w_kernel.h)
};
struct Dkdv1Plan {
  int NJT, JR, nlaunch, nkg, nchunks, rows_per_chunk, threads;   // NJT, JR: of the first range
  int range[kMaxRanges];          // queries per launch
  size_t smem_range[kMaxRanges];
  size_t smem;                    // the largest
};

// Geometry of the one-kernel backward for rows of up to 128 keys, at D = 32 192 (with dropout 256); a workgroup holds a whole row.
struct ShortPlan {
  int NT, nchunks, rows_per_chunk, threads;
  size_t smem;
};

struct BwdPlan {
  // dQ/dBias kernel
  int SK, QB, nqg, nchunks, rows_per_chunk, threads, KR, nlaunch, ring, nb;
  int NKT;             // 32-key tiles of a wave's slab
  size_t smem;
  // dK/dV kernel
  int NJT, JT, SJ, KB, nkg, nchunks2, rows_per_chunk2, threads2, JR, nlaunch2, ring2, nb2;
  size_t smem2;
  size_t delta_bytes, partial_bytes, aux_bytes;
  bool use_hand;       // the hand-scheduled one-wave-per-SIMD kernels run
  Dq1Plan dq1;
  Dkdv1Plan dkdv1;
  int nranges;         // dropout beyond 512 keys: ranges of their own geometry (see drop_range), else 0
  int nranges2;        // the same for dK/dV, 0 where it takes launches of JR queries
  int range[kMaxRanges];
  bool use_short;      // short rows: all gradients in one kernel
  ShortPlan sh;
  int L2p;             // the length the workspace is laid out with and the general kernels' tiles cover (filled in by the C-ABI layer)
  int Lt;              // the length the hand-scheduled kernels' tiles cover: the next multiple of 64, not of 128, where they have the instances
  bool own_delta;      // dropout: the dQ/dBias kernel forms delta and the row constants itself, no kernel runs in front of it
  bool feat;           // planned for the feature instances (bf16, dropout, precise fp16)
  bool valid;
};

// The hand-scheduled backward kernels round sm_scale * log2(e) * Q (and K) to the element type before
// the matrix core.  With bf16's 8 bits that rounding error grows with the scale (gradients: 4e-3
// relative-L2 at sm_scale = 1/sqrt(32), 1.7e-2 at 1.3 on N(0,1) inputs): beyond this scale the D = 32
// instances that carry the product as a (hi, lo) pair of bf16 values run (one more MFMA per contraction
// step of the score tile); D = 64 has no registers for the pair and takes the instances that apply the
// scale in fp32.
constexpr float kBf16PlainMaxScaleLog2 = 0.5f;
inline bool bf16_scale_needs_split(float sm_scale) { return !(fabsf(sm_scale) * 1.4426950408889634f <= kBf16PlainMaxScaleLog2); }

// Geometry of the one-wave-per-SIMD dQ/dBias kernel (256-key wave slabs).
bool plan_dq1(int B, int H, int L1, int L2, int row, int D, Dq1Plan& pl);
hipError_t launch_dq1(BwdParams p, const Dq1Plan& pl, int D, int dtype, bool hilo, bool nat, hipStream_t st);

bool plan_short(int B, int H, int L1, int L2, int D, int feat, ShortPlan& pl);
hipError_t launch_short(BwdParams p, const ShortPlan& pl, int D, int dtype, bool precise, hipStream_t st);

bool plan_dkdv1(int B, int H, int L1, int L2, int D, Dkdv1Plan& pl);
hipError_t launch_dkdv1(BwdParams p, const Dkdv1Plan& pl, int D, int dtype, bool hilo, bool nat, hipStream_t st);

// Stage buffers and row-operand buffers that a workgroup's share of LDS holds beside the exchange records, 160 KB for eight waves and
// 80 for four: of the dQ/dBias kernel with SK slabs
// of NKT tiles, G1 of them to a stage, and of the dK/dV kernel with SJ slabs of NJT tiles, JT queries to a stage
// (the kernels with that geometry fixed and the launch plan agree on it).
struct Ring { int r, nb; };
constexpr Ring fit_ring(int steps, int slot, int row, int records, int waves) {
  for (int r = 4; r >= 3; --r) {
    const int nb = (r + steps - 1) / steps;
    if (r * slot + nb * row + records <= waves * 20 * 1024) return Ring{r, nb};
  }
  return Ring{0, 0};
}
// (registers of its partial dQ that a wave publishes to the other slabs: all, at D = 64 those that they finish, of up to four slabs three quarters)
constexpr int dq_record_regs(int D) { return D == 32 ? 16 : 24; }
constexpr int dq_records(int D, int SK, int waves) { return SK > 1 ? waves * dq_record_regs(D) * 64 * 4 : 0; }
constexpr Ring dq_ring(int D, int NKT, int G1, int SK, int waves) {
  return fit_ring(NKT / G1, 4 * SK * G1 * 32 * D, 4 * (waves / SK) * 32 * D, dq_records(D, SK, waves), waves);
}
constexpr size_t dq_smem(int D, int NKT, int G1, int SK, int waves) {
  const Ring r = dq_ring(D, NKT, G1, SK, waves);
  return (size_t)r.r * (4 * SK * G1 * 32 * D) + (size_t)r.nb * (4 * (waves / SK) * 32 * D) + dq_records(D, SK, waves);
}
constexpr int dkdv_shares(int D, int SJ, int waves) { return (SJ - 1) * (waves / SJ) * 32 * (D / 32) * 64 * 4; }
constexpr Ring dkdv_ring(int D, int NJT, int JT, int SJ, int waves) {
  return fit_ring(NJT / (JT / 32), 4 * SJ * JT * D + 8 * SJ * JT, 4 * (waves / SJ) * 32 * D, dkdv_shares(D, SJ, waves), waves);
}

constexpr size_t dkdv_smem(int D, int NJT, int JT, int SJ, int waves) {
  const Ring r = dkdv_ring(D, NJT, JT, SJ, waves);
  return (size_t)r.r * (4 * SJ * JT * D + 8 * SJ * JT) + (size_t)r.nb * (4 * (waves / SJ) * 32 * D) + dkdv_shares(D, SJ, waves);
}

// One key range and one query range of the backward with dropout beyond 512 keys (D = 32): stage and row-operand
// buffers and LDS bytes of the dQ/dBias kernel with four slabs and of the dK/dV kernel with two.
struct DropRange { Ring dq, dkdv; size_t smem, smem2; };
inline DropRange drop_range(int len) {
  const int nkt = len / 128, g1 = nkt == 4 ? 2 : 1, njt = len / 64;
  return DropRange{dq_ring(32, nkt, g1, 4, 8), dkdv_ring(32, njt, 64, 2, 8), dq_smem(32, nkt, g1, 4, 8), dkdv_smem(32, njt, 64, 2, 8)};
}

// L2 is the length the tiles cover (a multiple of 128), `row` the true row length.
// `feat`: 0 the fp16 kernels; 1 the plan is for bf16 inputs or the precise mode, 2 for dropout (general
// kernels only, smaller instance sets).  `limit`: at most that many bytes of workspace (0: any number) if the partial dBias of
// one chunk fits.
BwdPlan plan_bwd(int B, int H, int L1, int L2, int D, int row, int feat, size_t limit = 0);
hipError_t launch_bwd(BwdParams p, const BwdPlan& pl, int D, int dtype, hipStream_t st, hipEvent_t* ev = nullptr);
hipError_t launch_dbias_reduce(const BwdParams& p, int dtype, hipStream_t st);
hipError_t launch_bwd_feat(const BwdParams& p, const BwdPlan& pl, int D, int dtype, hipStream_t st, hipEvent_t* ev);

// feat: the plan is for bf16 inputs or dropout, which have a smaller set of kernel instances
// (`row`: the true row length)
FwdPlan plan_fwd(int B, int H, int L1, int L2, int D, int row, bool feat, bool scattered = false);

// The kernels are gfx950 code objects: FTA_OK if the current device can run them (fta_api.hip).
int check_device();

// Launch helper shared by all kernels: raises the kernel's dynamic-LDS limit to `smem` bytes once
// per (kernel, device) -- the attribute call is not free and the limit only ever has to grow --
// then launches.  Defined in fta_api.hip.
hipError_t ensure_dynamic_lds(const void* kern, size_t smem);
template <class K, class P>
inline hipError_t launch_kernel(K kern, const P& p, dim3 grid, dim3 block, size_t smem, hipStream_t st) {
  hipError_t e = ensure_dynamic_lds(reinterpret_cast<const void*>(kern), smem);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(kern, grid, block, smem, st, p);
  return hipGetLastError();
}

// The backward runs the general kernels even where others apply (set through fta_debug_select_kernels, for tests).
bool forced_general();
hipError_t launch_fwd(FwdParams p, const FwdPlan& pl, int D, int dtype, hipStream_t st);
// The hand-scheduled forward (fta_fwd1_kernel.h): D = 32, tiled length 64 ... 1792, no dropout.
bool plan_fwd1(int B, int H, int L1, int L2, int D, int row, bool scattered, FwdPlan& pl);
hipError_t launch_fwd1(const FwdParams& p, const FwdPlan& pl, int dtype, dim3 grid, dim3 block, hipStream_t st);
hipError_t launch_fwd1_slabs(const FwdParams& p, const FwdPlan& pl, int dtype, bool tl, dim3 grid, dim3 block, hipStream_t st);
bool plan_fwd2(int B, int H, int L1, int L2, int D, FwdPlan& pl);
hipError_t launch_fwd2(const FwdParams& p, const FwdPlan& pl, int dtype, dim3 grid, dim3 block, hipStream_t st);
hipError_t launch_fwd_feat(const FwdParams& p, const FwdPlan& pl, int D, int dtype, dim3 grid, dim3 block, hipStream_t st);

}  // namespace fta
