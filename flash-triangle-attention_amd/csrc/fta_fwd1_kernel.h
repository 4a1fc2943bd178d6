// Forward, hand-scheduled variant (D = 32, tiled length 64 ... 1792; one key slab up to 512).
// Same mathematics and the same decomposition as fta_fwd_kernel (fta_fwd_kernel.h): a wave owns 32
// queries and all keys of a (b,h), keeps its bias tile in registers and walks a chunk of L1 rows;
// replaces upstream's _attn_fwd / _attn_fwd_inner (flash_tt_attn.py:49-109, :128-264).  What differs
// is the order of the instructions, which here is the order of the statements:
//   * the walk over 32-key tiles is software-pipelined inside each wave.  Iteration t issues the MFMAs
//     of O^T += V^T P^T for tile t-1 and of S^T = K Q^T for tile t+1 between the four blocks of
//     vector-ALU work of tile t, the LDS reads of the operands those MFMAs need one iteration ahead,
//     and one asynchronous copy of a later stage; nothing waits for a latency it has just started.
//     The pipeline runs across stage and row boundaries (a row is finished, normalised and stored
//     inside the first iteration of the next one);
//   * K/V stages of 128 keys live in a ring of four LDS slots; the barrier that publishes a stage sits
//     one tile before its first use, and the slot it frees is refilled one copy per iteration;
//   * per score the vector ALU does t = fma_mix(S, scale, bias) (fp32, bias exact from its fp16
//     pair), x = fma(t, log2e, -ref*log2e), p = exp2(x), and per pair one packing and one dot2 for the
//     row sum: no running maximum.  The reference `ref` is the maximum of the row's first tile plus a
//     margin; a later tile whose weights leave the 16-bit range shows in its own partial sum and is
//     redone, with O and l rescaled, by a slow path out of line (never taken at ordinary softmax
//     scales).
#pragma once
#include "fta_fwd_blocks.h"

namespace fta {

typedef float floatx4 __attribute__((ext_vector_type(4)));

// T: element type; NKT: 32-key tiles per row and slab (2 to 16: the score tiles alternate between two register
// tuples, and an odd count moves the next row's first tile from one to the other at the end of a row, 16 instructions
// where the tile it saves takes 64); TAIL: the row's true length L2 is shorter
// than the 32*NKT keys the tiles cover, or than the workgroups' query blocks (keys beyond it masked, queries
// beyond it computed on copies of the last one and not stored); W: waves (query blocks of 32) per workgroup: 4, or 2 for rows of up to 64
// keys, and 8 with several slabs (and for some rows of 256 keys, see plan_fwd1).
// Two waves share a SIMD either way.  With one slab they belong to independent workgroups, and the hardware lets the
// older one issue first whenever both are ready, which in a kernel bound by the vector ALU is nearly always: measured with
// a clock around every workgroup (B4 H8 L512), the older workgroup of a CU finished its 128 rows after 750 us and the
// younger one, left with a SIMD to itself that a lone wave cannot fill, after 1250.  So a wave's priority falls from half row to
// half row, in turns of two rows: the one that is ahead by less than two yields until the other has caught up (two rows apart they are equals
// again; and one that waits lets the other issue, whatever their priorities), and their barriers stay uncoupled.  Without / with it, us: B1 H4 L150
// 13.1 / 12.5, L200 20.4 / 18.4, L300 42.7 / 40.3, L384 66.8 / 63.0, L457 in bf16 113 / 109, B2 H4 L320 88.7 / 84, B4 H8 L128 31.7 / 31.9 (inputs in
// the caches 27.0 / 26.6), L192 89.7 / 85.6, L384 at scale 1.3 510 / 489.  One workgroup of eight
// waves, where the two waves of a SIMD meet at every stage barrier, gives B4 H8 L512 1037 and 1117 us (scale 1.3), B1 H4 L512 137.6; this 989,
// 1051 and 131.4.  Four steps over the whole chunk instead: 1027, 1087, 134.1; a step a row in turns of four: 984, 1055, 131.0, but 2 % more
// at 128 keys; four steps within a row: equal, 3 % more at 384 keys.
// S: key slabs.  Rows beyond 512 keys do not fit one wave's bias registers: S = 2 or 4 waves of a workgroup
// take the keys of one query block in slabs of 32*NKT and merge their (m, l, O) through LDS, in fp32, once per row:
// every slab finishes 16/S of the accumulator registers.  A stage then holds 64 keys of every slab.  Two slabs: workgroups of two query
// blocks, two to a CU, whose records of the merge leave out what a wave keeps (10 KB; with them whole a second workgroup does not fit LDS).
// Barriers of two workgroups do not couple, and a row's last query group is at most one block short; K and V are copied into LDS
// once for two query blocks instead of four.  B1 H4, us, one workgroup of four query blocks / two of two: L540 219 / 196, L660 in bf16 368 /
// 330, L701 in bf16 409 / 382, L768 at scale 1.3 523 / 489, L900 in bf16 813 / 762, L1000 996 / 980, B2 H4 L1024 2059 / 1988 (transposed: see plan_fwd1).
// (against the general kernel, rocprofv3, middle half of 60 launches: B1 H4 L701 bf16 656 -> 466 us, B1 H4 L1536 fp16
// 5200 -> 4100)
template <class T, int NKT, bool TAIL, int W, int G = 4, int S = 1>
__global__ void __attribute__((amdgpu_flat_work_group_size(64 * W, 64 * W), amdgpu_waves_per_eu(2, 2))) fta_fwd1_kernel(const FwdParams p) {
  static_assert(S == 4 ? W == 8 : W == 4 || (S == 2 && W == 8) || (S == 1 && W == 8 && NKT == 8) || (S == 1 && W == 2 && NKT == 2), "one or two waves per SIMD from the same workgroup");
  static_assert(S == 1 ? G == 4 || (G == 2 && NKT == 2) : G == 2, "stages of 128 keys; of 64 for such rows and for several slabs");
  static_assert(S == 1 || ((S == 2 || S == 4) && NKT >= 6), "slabs: four query blocks in two, or two in four; the merge takes the first three iterations of a row");
  constexpr int D = 32, KS = 2;
  constexpr int NCU = S * 2 * G / W;           // copies per wave and stage of K, and of V (a stage has 2*G pieces of 1 KB of each per slab)
  constexpr int KT = 32 * G;                   // keys per stage and slab
  constexpr int KW = 32 * NKT;                 // keys per slab
  constexpr int NST = (NKT + G - 1) / G;       // stages per row, the last one of NKT % G tiles where that is not 0
  constexpr int R = 4;                         // ring slots
  constexpr uint32_t TILE_B = S * KT * D * 2;  // bytes of a staged K (or V) tile: slab after slab
  constexpr uint32_t SLOT_B = 2 * TILE_B;      // K tile, then V tile
  static_assert(NKT >= 2 && NKT <= 16, "bias within the register budget");
  constexpr bool ODD = NKT % 2 != 0;
  // Stage w of a row: its tiles, and the copies a wave issues for it (of K, and as many of V).
  constexpr auto tiles_of = [](int w) { return (w + 1) * G <= NKT ? G : NKT - w * G; };
  // (several slabs: a slab's rows keep their place in a stage that is not full; what is not a tile of the slab is copied and not read)
  constexpr auto ncu_of = [=](int w) { return S > 1 ? NCU : (2 * tiles_of(w) + W - 1) / W; };
  // Iteration t issues the scores of tile tn = (t + 1) % NKT, and the tn % G-th share of the copies of the stage two
  // behind tile tn's: `first` to `end`, the K copies before the V copies.
  struct Share { int stage, first, end; };
  constexpr auto share_of = [=](int tn) {
    const int w = tn / G, fill = (w + 2) % NST, total = 2 * ncu_of(fill), per = (total + tiles_of(w) - 1) / tiles_of(w);
    const int a = (tn % G) * per;
    return Share{fill, a < total ? a : total, a + per < total ? a + per : total};
  };
  // copies issued between the request for the next row's Q and the last barrier of the row
  constexpr auto behind_q = [=]() {
    int n = 0;
    for (int tn = 1; tn < NKT; ++tn) n += share_of(tn).end - share_of(tn).first;
    return n;
  };

  extern __shared__ __attribute__((aligned(16))) char smem_raw[];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int hh = lane >> 5, l32 = lane & 31;

  const WorkId id = work_id(p.nqg, p.nchunks, p.H, p.head_inner);
  const int qg = id.group, chunk = id.chunk, b = id.b, h = id.h, bh = b * p.H + h;
  const int i0 = chunk * p.rows_per_chunk;
  const int nrows = min(p.rows_per_chunk, p.L1 - i0);
  if (nrows <= 0) return;  // whole workgroup leaves together

  const int slab = wave % S;
  const int q0 = (qg * (W / S) + wave / S) * 32;  // first query of this wave
  const int last = p.L2 - 1;
  const int qrow = TAIL ? min(q0 + l32, last) : q0 + l32;
  const bool qvalid = !TAIL || (q0 + l32 <= last);

  const half_t* qbase = p.q + b * p.qs[0] + h * p.qs[1];
  const half_t* kbase = p.k + b * p.ks[0] + h * p.ks[1];
  const half_t* vbase = p.v + b * p.vs[0] + h * p.vs[1];
  half_t* obase = p.o + b * p.os[0] + h * p.os[1];

  // ---- stage copies: a stage is 32*G K rows and 32*G V rows of 64 bytes, 1 KB per wave instruction,
  // NCU K and NCU V copies per wave; copy u of wave w carries the 16-byte pieces (w + W*u)*64 .. +63.
  // (S = 2: a copy covers rows of one slab, and a wave's next one the same rows of the other: one offset, and the slabs' distance in
  // the base.  With four slabs, where registers are left, that is 2 % slower)
  constexpr int NGO = S == 2 ? 1 : NCU;
  uint32_t goffk[NGO], goffv[NGO];
  constexpr bool CLAMP = TAIL || NKT % G != 0;
  [[maybe_unused]] uint32_t goffk_t[NGO], goffv_t[NGO];  // CLAMP: the row's last stage (rows beyond the last key are copies of it); S = 4: the last key's row
  [[maybe_unused]] const uint32_t ctail = (uint32_t)swz_slot<D>(lane >> 2, lane & 3) * 16u;  // S = 2: this lane's piece of a row, the same in every copy (16 rows each)
#pragma unroll
  for (int u = 0; u < NGO; ++u) {
    const int pidx = (wave + W * u) * 64 + lane, prow = pidx >> 2, chunkk = swz_slot<D>(prow, pidx & 3), row = (prow / KT) * KW + prow % KT;
    goffk[u] = (uint32_t)(((int64_t)row * p.ks[3] + chunkk * 8) * 2);
    goffv[u] = (uint32_t)(((int64_t)row * p.vs[3] + chunkk * 8) * 2);
    if constexpr (CLAMP && S != 2) {
      const int grow = S > 1 ? last : min((NST - 1) * KT + row, last) - (NST - 1) * KT;
      goffk_t[u] = (uint32_t)(((int64_t)grow * p.ks[3] + chunkk * 8) * 2);
      goffv_t[u] = (uint32_t)(((int64_t)grow * p.vs[3] + chunkk * 8) * 2);
    }
  }
  const uint32_t lds0 = lds_addr_of(smem_raw);
  const uint32_t wofs = (uint32_t)wave * 1024u;
  int64_t rstep_k = hold_scalar(p.ks[2] * 2), rstep_v = hold_scalar(p.vs[2] * 2);            // bytes from one row to the next
  int64_t sstep_k = hold_scalar(p.ks[3] * 2 * KT), sstep_v = hold_scalar(p.vs[3] * 2 * KT);  // from one stage to the next
  [[maybe_unused]] const int64_t ustep_k = (int64_t)KW * p.ks[3] * 2, ustep_v = (int64_t)KW * p.vs[3] * 2;
  // fill cursor: the stage the copies currently go to (row pointer, LDS slot); it runs ahead of the row
  // being computed and stops advancing at the chunk's last row (whose data is then copied again into
  // slots nothing reads any more: the loop stays free of "is there a next stage" branches)
  const char* kfill = (const char*)(kbase + (int64_t)i0 * p.ks[2]);
  const char* vfill = (const char*)(vbase + (int64_t)i0 * p.vs[2]);
  int fill_row = 0;
  uint32_t fill_lds = lds0 + wofs;  // LDS byte address of this wave's first copy in the slot being filled
  int fill_slot = 0;
  const char* kst = kfill;          // the stage's first K row / V row
  const char* vst = vfill;
  // begins stage number w (compile-time) of the fill row, or of the next row when w == 0 and `advance`
  auto fill_begin = [&](auto wc, bool advance) {
    constexpr int w = decltype(wc)::value;
    if constexpr (w == 0) {
      if (advance) {
        const bool more = fill_row + 1 < nrows;
        fill_row += more ? 1 : 0;
        kfill += more ? rstep_k : 0;
        vfill += more ? rstep_v : 0;
      }
    }
    kst = kfill + w * sstep_k;
    vst = vfill + w * sstep_v;
    fill_lds = lds0 + wofs + (uint32_t)fill_slot * SLOT_B;
    fill_slot = (fill_slot + 1) & (R - 1);
  };
  // S = 2: the smaller of `off` + `step` and this lane's piece of the last key's row (formed at every use: the sums would be kept over the rows)
  [[maybe_unused]] uint32_t lastk = (uint32_t)(last * p.ks[3] * 2), lastv = (uint32_t)(last * p.vs[3] * 2);
  auto clamped = [&](uint32_t off, uint32_t step, uint32_t lastrow) {
    uint32_t a, b;
    asm volatile("v_add_u32 %0, %2, %3\n\tv_add_u32 %1, %4, %5\n\tv_min_u32 %0, %0, %1" : "=&v"(a), "=&v"(b) : "s"(step), "v"(off), "s"(lastrow), "v"(ctail));
    return a;
  };
  // copy c (first the K copies, then the V copies) of the stage begun last, which is stage number w of
  // its row
  auto fill_copy = [&](auto wc, auto cc) {
    constexpr int w = decltype(wc)::value, c = decltype(cc)::value, nk = ncu_of(w);
    constexpr bool TL = S == 1 && CLAMP && (w == NST - 1);
    static_assert(c < 2 * nk, "a copy of the stage");
    if constexpr (S > 1 && (TAIL ? w >= NST - S : w * G + G > NKT)) {
      // (fewer than 64*S keys are missing, so the last slab ends in one of its last S stages; a stage that is not full
      // reaches beyond the last slab)
      if constexpr (S == 4) {
        if constexpr (c < nk) dma16s_at<(uint32_t)c * W * 1024u>(min(goffk[c] + (uint32_t)(w * sstep_k), goffk_t[c]), kfill, fill_lds);
        else dma16s_at<TILE_B + (uint32_t)(c - nk) * W * 1024u>(min(goffv[c - nk] + (uint32_t)(w * sstep_v), goffv_t[c - nk]), vfill, fill_lds);
      } else if constexpr (c < nk) dma16s_at<(uint32_t)c * W * 1024u>(clamped(goffk[0], (uint32_t)(w * sstep_k + c * ustep_k), lastk), kfill, fill_lds);
      else dma16s_at<TILE_B + (uint32_t)(c - nk) * W * 1024u>(clamped(goffv[0], (uint32_t)(w * sstep_v + (c - nk) * ustep_v), lastv), vfill, fill_lds);
    } else if constexpr (S == 2) {
      if constexpr (c < nk) dma16s_at<(uint32_t)c * W * 1024u>(goffk[0], kst + c * ustep_k, fill_lds);
      else dma16s_at<TILE_B + (uint32_t)(c - nk) * W * 1024u>(goffv[0], vst + (c - nk) * ustep_v, fill_lds);
    } else if constexpr (c < nk) dma16s_at<(uint32_t)c * W * 1024u>(TL ? goffk_t[c] : goffk[c], kst, fill_lds);
    else dma16s_at<TILE_B + (uint32_t)(c - nk) * W * 1024u>(TL ? goffv_t[c - nk] : goffv[c - nk], vst, fill_lds);
  };
  auto fill_share = [&](auto tc) {
    constexpr Share sh = share_of(decltype(tc)::value);
    static_for<sh.first, sh.end>([&](auto cc) { fill_copy(std::integral_constant<int, sh.stage>{}, cc); });
  };

  // ---- Q^T B-operand fragments of one row, straight into registers (contraction step ks holds
  // d = 16*ks + 8*hh .. +7); issued one row ahead, pending until a later barrier wait covers them
  const char* qcur = (const char*)(qbase + (int64_t)i0 * p.qs[2]);
  int64_t rstep_q = hold_scalar(p.qs[2] * 2);
  const uint32_t voff_q = (uint32_t)(((int64_t)qrow * p.qs[3] + 8 * hh) * 2);
  int q_row = 0;
  u32x4 qn[KS];
  auto q_issue = [&](bool advance) {
    if (advance) {
      const bool more = q_row + 1 < nrows;
      q_row += more ? 1 : 0;
      qcur += more ? rstep_q : 0;
    }
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
      asm volatile("global_load_dwordx4 %0, %1, %2" : "=v"(qn[ks]) : "v"(voff_q + 32u * ks), "s"(qcur) : "memory");
  };

  // ---- per-lane LDS addresses of the operand reads inside a slot
  FragOffsets<D> fo;
  fo.init(lane);
  uint32_t aK[KS], aT[2], aKc[KS], aTc[2];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) aK[ks] = lds0 + (uint32_t)(slab * KT * D + fo.a[ks]) * 2u;
#pragma unroll
  for (int x = 0; x < 2; ++x) aT[x] = lds0 + TILE_B + (uint32_t)(slab * KT * D + fo.t[0][x]) * 2u;
  int kslot = 0;  // slot the K reads are in (the V^T reads follow one tile later)

  const float scale = p.scale;
  const float lg2e = kLog2e;
  const uint32_t ones = T::is_bf16 ? 0x3F803F80u : 0x3C003C00u;

  // ---- prologue: stages 0 and 1 whole; the stationary bias (tile tt, register pair rg holds keys 32*tt + 8*rg +
  // 4*hh + 0..3 of query l32), which changes lanes in the ring slots that nothing is copied to yet; Q of row 0; behind
  // the barrier the first share of stage 2 (the one the iteration "before the first" would have issued)
  static_for<0, 2>([&](auto nc) {
    constexpr int n = decltype(nc)::value;
    fill_begin(std::integral_constant<int, n % NST>{}, n > 0);
    static_for<0, 2 * ncu_of(n % NST)>([&](auto cc) { fill_copy(std::integral_constant<int, n % NST>{}, cc); });
  });
  uint32_t bias_reg[NKT][8];
  static_assert(W * 4096 <= 2 * SLOT_B, "4 KB for every wave's bias");
  {
    const half_t* bias_bh = p.bias + b * p.bs[0] + h * p.bs[1];
    char* turn = smem_raw + 2 * SLOT_B + wave * 4096;
    auto sink = [&](int tt, int rg, u32x2 v) {
      bias_reg[tt][2 * rg] = v[0];
      bias_reg[tt][2 * rg + 1] = v[1];
    };
    load_bias_tiles<NKT / 2, 2, TAIL, NKT == 2>(bias_bh, p.bs[2], q0, p.L2, F16::kBeyond2, turn, lane, [=](int c) { return slab * KW + 64 * c; },
                                                fwd1_bias_pair<T>, sink);
    if constexpr (ODD)
      load_bias_tiles<1, 1, TAIL, false>(bias_bh, p.bs[2], q0, p.L2, F16::kBeyond2, turn, lane, [=](int) { return slab * KW + 32 * (NKT - 1); },
                                         fwd1_bias_pair<T>, [&](int, int rg, u32x2 v) { sink(NKT - 1, rg, v); });
  }
  q_issue(false);
  wait_vmem_all();
  __syncthreads();
  fill_begin(std::integral_constant<int, 2 % NST>{}, true);
  fill_share(std::integral_constant<int, 0>{});

  u32x4 qf[KS];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) qf[ks] = qn[ks];
  asm volatile("" : "+v"(qf[0]), "+v"(qf[1]));
  q_issue(true);  // row 1 (pending until the barrier of the row's last iteration)

  floatx16 s[2];
  floatx16 acc;
  uint32_t ph[8];
  u32x2 vtl[2], vth[2];  // V^T operands of the tile whose O^T MFMAs come next: two 16-key steps, as read
  u32x4 kf[KS];
#pragma unroll
  for (int r = 0; r < 16; ++r) acc[r] = 0.f;
#pragma unroll
  for (int r = 0; r < 8; ++r) ph[r] = 0u;
#pragma unroll
  for (int u = 0; u < 2; ++u) { vtl[u] = u32x2{0u, 0u}; vth[u] = u32x2{0u, 0u}; }
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) aKc[ks] = aK[ks];
#pragma unroll
  for (int x = 0; x < 2; ++x) aTc[x] = aT[x];
  {
    kf[0] = lds_issue_b128<0>(aKc[0]);
    kf[1] = lds_issue_b128<0>(aKc[1]);
    asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(kf[0]), "+v"(kf[1]));
    mfma_new_v<T>(s[0], as_half8(kf[0]), as_half8(qf[0]));
    mfma_acc_v<T>(s[0], as_half8(kf[1]), as_half8(qf[1]));
    asm volatile("s_nop 15\n\ts_nop 7" : "+v"(s[0]), "+v"(acc), "+v"(ph[0]), "+v"(ph[1]), "+v"(ph[2]), "+v"(ph[3]), "+v"(ph[4]),
                 "+v"(ph[5]), "+v"(ph[6]), "+v"(ph[7]));
  }
  asm volatile("" : "+v"(vtl[0]), "+v"(vtl[1]), "+v"(vth[0]), "+v"(vth[1]));

  float l = 0.f, m_ref = 0.f, nm = 0.f;   // running sum (this lane's half of the keys), reference (natural units), -ref*log2e
  float l_done = 1.f, m_done = 0.f;       // of the row whose O^T is being completed
  half_t* ocur = obase + (int64_t)i0 * p.os[2];
  float* lcur = p.lse + ((int64_t)bh * p.L1 + i0) * p.L2;
  const int64_t ostep = p.os[2];
  const uint32_t ooff = (uint32_t)(((int64_t)(q0 + l32) * p.os[3] + 8 * hh) * 2);  // bytes from the row's uniform base
  // (a store of more than 8 bytes reads its data registers for two more issue slots: nothing may rewrite them there, and
  // the compiler does not know that these statements are stores)
  auto store_lse = [&](float lse2) {
    if (hh == 0) {
      // (the byte offset is made here, from the lane number, once per row: the register file has no room to keep it)
      uint32_t lse_off;
      asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(lse_off));
      lse_off = (uint32_t)(q0 + (lse_off & 31u)) * 4u;
      asm volatile("global_store_dword %0, %1, %2" : : "v"(lse_off), "v"(lse2), "s"(lcur) : "memory");
    }
  };

  // Normalises and stores the finished row (`acc` complete): the two lanes of a query (hh = 0, 1) hold
  // alternating runs of four d values; one exchange per register pair gives each of them eight
  // consecutive ones, so the row goes out in 16-byte pieces: d = 16 pr + 8 hh .. +7.
  auto finish_row = [&]() {
    const float lt = sum_both_halves(l_done);
    const float inv = __builtin_amdgcn_rcpf(lt);
    if (qvalid) {
#pragma unroll
      for (int pr = 0; pr < 2; ++pr) {
        const uint32_t x0 = T::pack(acc[8 * pr] * inv, acc[8 * pr + 1] * inv), x1 = T::pack(acc[8 * pr + 2] * inv, acc[8 * pr + 3] * inv);
        const uint32_t y0 = T::pack(acc[8 * pr + 4] * inv, acc[8 * pr + 5] * inv), y1 = T::pack(acc[8 * pr + 6] * inv, acc[8 * pr + 7] * inv);
        auto r0 = __builtin_amdgcn_permlane32_swap(x0, y0, false, false);
        auto r1 = __builtin_amdgcn_permlane32_swap(x1, y1, false, false);
        const u32x4 piece = {(uint32_t)r0[0], (uint32_t)r1[0], (uint32_t)r0[1], (uint32_t)r1[1]};
        // (uniform row base + one 32-bit register of per-lane offset)
        if (pr == 0) asm volatile("global_store_dwordx4 %0, %1, %2\n\ts_nop 1" : : "v"(ooff), "v"(piece), "s"(ocur) : "memory");
        else asm volatile("global_store_dwordx4 %0, %1, %2 offset:32\n\ts_nop 1" : : "v"(ooff), "v"(piece), "s"(ocur) : "memory");
      }
      store_lse(m_done * kLog2e + __builtin_amdgcn_logf(lt));
    }
    ocur += ostep;
    lcur += p.L2;
  };

  // S > 1: the finished row's accumulator changes waves in two steps.  A wave's record holds the accumulator registers that
  // others finish, in groups of four, 1 KB each, and its (l, m) behind them; its own stay in registers.  S = 2: slab s finishes
  // registers 8*s .. +7.  S = 4: group s; group g of slab s is in place (g - s - 1) % 4 (its own goes to a place that nothing reads).
  constexpr uint32_t REC_B = (S == 4 ? 3072u : 2048u) + 512u;
  const uint32_t rec0 = lds0 + R * SLOT_B;
  [[maybe_unused]] float keep[16 / (S > 1 ? S : 4)];
  [[maybe_unused]] uint32_t ostride = (uint32_t)p.os[3] * 2u;
  if constexpr (S > 1) asm volatile("" : "+s"(ostride));
  auto lane_now = []() {  // (see store_lse)
    uint32_t l;
    asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(l));
    return l;
  };
  auto merge_give = [&]() {
    if constexpr (S > 1) {
      const uint32_t ln = lane_now(), rec = rec0 + (uint32_t)wave * REC_B;
      const float lt = sum_both_halves(l_done), m2 = m_done * kLog2e;
      auto half = [&](auto own) {
#pragma unroll
        for (int g = 0; g < 2; ++g) {
          constexpr int o = decltype(own)::value;
          const floatx4 v = {acc[8 - o + 4 * g], acc[9 - o + 4 * g], acc[10 - o + 4 * g], acc[11 - o + 4 * g]};
          asm volatile("ds_write_b128 %0, %1 offset:%2" : : "v"(rec + ln * 16u), "v"(v), "n"(g * 1024) : "memory");
#pragma unroll
          for (int e = 0; e < 4; ++e) keep[4 * g + e] = acc[o + 4 * g + e];
        }
      };
      if constexpr (S == 2) {
        if (slab == 0) half(std::integral_constant<int, 0>{});
        else half(std::integral_constant<int, 8>{});
      }
#pragma unroll
      for (int g = 0; g < (S == 4 ? 4 : 0); ++g) {
        const uint32_t at = (g == slab) ? rec0 + W * REC_B : rec + (uint32_t)((g - slab - 1) & 3) * 1024u;
        const floatx4 v = {acc[4 * g], acc[4 * g + 1], acc[4 * g + 2], acc[4 * g + 3]};
        asm volatile("ds_write_b128 %0, %1" : : "v"(at + ln * 16u), "v"(v) : "memory");
      }
      asm volatile("ds_write_b64 %0, %1 offset:%2" : : "v"(rec + ln * 8u), "v"(u32x2{__builtin_bit_cast(uint32_t, lt), __builtin_bit_cast(uint32_t, m2)}), "n"(REC_B - 512u) : "memory");
      if constexpr (S == 4) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float lo = (slab & 1) ? acc[4 + e] : acc[e], hi = (slab & 1) ? acc[12 + e] : acc[8 + e];
          keep[e] = (slab & 2) ? hi : lo;
        }
      }
    }
  };
  // (a stage barrier later)
  auto merge_take = [&]() {
    if constexpr (S > 1) {
      const uint32_t ln = lane_now(), team = rec0 + (uint32_t)(wave - slab) * REC_B;
      u32x2 st[S];  // (l, m) of every slab
#pragma unroll
      for (int x = 0; x < S; ++x) asm volatile("ds_read_b64 %0, %1 offset:%2" : "=v"(st[x]) : "v"(team + (uint32_t)x * REC_B + ln * 8u), "n"(REC_B - 512u) : "memory");
      if constexpr (S == 2) asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(st[0]), "+v"(st[1]));
      else asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(st[0]), "+v"(st[1]), "+v"(st[S - 2]), "+v"(st[S - 1]));
      float c[S], M = -INFINITY, tot = 0.f;
#pragma unroll
      for (int x = 0; x < S; ++x) {
        const uint32_t mw = st[x][1];
        M = __builtin_fmaxf(M, __builtin_bit_cast(float, mw));
      }
#pragma unroll
      for (int x = 0; x < S; ++x) {
        const uint32_t lw = st[x][0], mw = st[x][1];
        c[x] = exp2_fast(__builtin_bit_cast(float, mw) - M);
        tot += __builtin_bit_cast(float, lw) * c[x];
      }
      const float inv = __builtin_amdgcn_rcpf(tot);
      float o[16 / S];
      if constexpr (S == 2) {
        const float ck = slab ? c[1] : c[0], cx = slab ? c[0] : c[1];
        floatx4 a[2];
        asm volatile("ds_read_b128 %0, %2\n\tds_read_b128 %1, %2 offset:1024\n\ts_waitcnt lgkmcnt(0)" : "=&v"(a[0]), "=&v"(a[1]) : "v"(team + (uint32_t)(slab ^ 1) * REC_B + ln * 16u) : "memory");
#pragma unroll
        for (int e = 0; e < 8; ++e) o[e] = __builtin_fmaf(keep[e], ck, a[e / 4][e % 4] * cx) * inv;  // (the same rounding in every instance)
      } else {
        const float ck = (slab & 2) ? ((slab & 1) ? c[S - 1] : c[S - 2]) : ((slab & 1) ? c[S - 3] : c[S - 4]);
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] = keep[e] * ck;
#pragma unroll
        for (int x = 1; x < S; ++x) {  // from slab (slab + x) % 4, whose place for this slab's group is 3 - x
          const int from = (slab + x) & 3;
          const float cx = (from & 2) ? ((from & 1) ? c[S - 1] : c[S - 2]) : ((from & 1) ? c[S - 3] : c[S - 4]);
          floatx4 a;
          asm volatile("ds_read_b128 %0, %1\n\ts_waitcnt lgkmcnt(0)" : "=v"(a) : "v"(team + (uint32_t)from * REC_B + (uint32_t)(3 - x) * 1024u + ln * 16u) : "memory");
#pragma unroll
          for (int e = 0; e < 4; ++e) o[e] = __builtin_fmaf(a[e], cx, o[e]);
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] *= inv;
      }
      if (qvalid) {
        // (the byte offset is made here, like that of lse)
        const uint32_t off = (uint32_t)(q0 + (ln & 31u)) * ostride + (64u / S) * (uint32_t)slab + (16u / (S / 2)) * (ln >> 5);
        if constexpr (S == 2) {  // registers 8*slab .. +7: d = 16 slab + 8 hh .. +7 once the lanes of a query have swapped
          auto r0 = __builtin_amdgcn_permlane32_swap(T::pack(o[0], o[1]), T::pack(o[4], o[5]), false, false);
          auto r1 = __builtin_amdgcn_permlane32_swap(T::pack(o[2], o[3]), T::pack(o[6], o[7]), false, false);
          const u32x4 piece = {(uint32_t)r0[0], (uint32_t)r1[0], (uint32_t)r0[1], (uint32_t)r1[1]};
          asm volatile("global_store_dwordx4 %0, %1, %2\n\ts_nop 1" : : "v"(off), "v"(piece), "s"(ocur) : "memory");
        } else {
          asm volatile("global_store_dwordx2 %0, %1, %2" : : "v"(off), "v"(u32x2{T::pack(o[0], o[1]), T::pack(o[2], o[3])}), "s"(ocur) : "memory");
        }
        if (slab == 0) store_lse(M + __builtin_amdgcn_logf(tot));
      }
      ocur += ostep;
      lcur += p.L2;
    }
  };

#pragma nounroll
  for (int ir = 0; ir < nrows; ++ir) {
    static_for<0, NKT>([&](auto tc) {
      constexpr int t = decltype(tc)::value;
      constexpr int tn = (t + 1) % NKT;           // the tile whose scores this iteration produces
      constexpr bool PUB = (tn % G == 0);         // tile t+1 opens a stage: publish it first
      floatx16& sc = s[t & 1];
      floatx16& sn = s[(t + 1) & 1];
      if constexpr (W < 8 && t == 0) {  // (see W above)
        if (ir & 1) __builtin_amdgcn_s_setprio(1);
        else __builtin_amdgcn_s_setprio(3);
      }
      if constexpr (W < 8 && t == NKT / 2) {
        if (ir & 1) __builtin_amdgcn_s_setprio(0);
        else __builtin_amdgcn_s_setprio(2);
      }

      if constexpr (PUB) {
        // everything but the copies of the stage after it has landed (copies retire in order; the last wait of
        // a row also covers the Q loads of the next row, which fewer copies may separate from it)
        constexpr int ahead = 2 * ncu_of((tn / G + 1) % NST);
        constexpr int allowed = (t == NKT - 1 && behind_q() < ahead) ? behind_q() : ahead;
        static_assert(allowed <= 15, "low bits of vmcnt");
        // (S > 1, iteration 1: also this wave's record of the finished row is in LDS before the others pass the barrier;
        // behind a stage of one tile: also the V^T reads of the iteration before, from the stage whose slot is filled now)
        constexpr bool drain = (S > 1 && t == 1) || (t == NKT - 1 && tiles_of(NST - 1) == 1);
        __builtin_amdgcn_s_waitcnt((drain ? 0x0070 : 0x0F70) | allowed);
        __builtin_amdgcn_s_barrier();
        kslot = (kslot + 1) & (R - 1);
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) aKc[ks] = aK[ks] + (uint32_t)kslot * SLOT_B;
        fill_begin(std::integral_constant<int, share_of(tn).stage>{}, true);  // into the slot the barrier has freed
      }
      // K operands of tile t+1
      kf[0] = lds_issue_b128<(tn % G) * 32 * D * 2>(aKc[0]);
      kf[1] = lds_issue_b128<(tn % G) * 32 * D * 2>(aKc[1]);
      fill_share(std::integral_constant<int, tn>{});

      // O^T += V^T P^T of tile t-1, first 16 keys (the V^T operands were read one iteration ago)
      asm volatile("s_waitcnt lgkmcnt(2)" : "+v"(vtl[0]), "+v"(vth[0]), "+v"(vtl[1]), "+v"(vth[1]));
      {
        const half8_t va = as_half8(u32x4{vtl[0][0], vtl[0][1], vth[0][0], vth[0][1]});
        const half8_t pb = as_half8(u32x4{ph[0], ph[1], ph[2], ph[3]});
        if constexpr (t == 1) mfma_restart_v<T>(acc, va, pb);
        else mfma_acc_v<T>(acc, va, pb);
      }
      if constexpr (t == 0) {
        // the row's first tile fixes the reference: its maximum plus the margin
        FTA_PIN_V(sc);
        float mx = -INFINITY;
#pragma unroll
        for (int r = 0; r < 16; r += 2) {
          const uint32_t bb = bias_reg[0][r >> 1];
          const float x0 = __builtin_fmaf(sc[r], scale, F16::lo(bb)), x1 = __builtin_fmaf(sc[r + 1], scale, F16::hi(bb));
          mx = __builtin_fmaxf(__builtin_fmaxf(mx, x0), x1);
        }
        m_ref = max_both_halves(mx) + kFwd1Margin;
        nm = -m_ref * kLog2e;
        asm volatile("" : "+v"(nm));
      }
      float lt;
      fwd1_block4<T, 0>(sc[0], sc[1], sc[2], sc[3], bias_reg[t][0], bias_reg[t][1], scale, lg2e, nm, ones, ph[0], ph[1], lt);
      FTA_HOLD2(vtl[0], vth[0]);  // (no register an MFMA reads is given to anything else before the block behind it has run)
      {
        const half8_t va = as_half8(u32x4{vtl[1][0], vtl[1][1], vth[1][0], vth[1][1]});
        const half8_t pb = as_half8(u32x4{ph[4], ph[5], ph[6], ph[7]});
        mfma_acc_v<T>(acc, va, pb);
      }
      fwd1_block4<T, 1>(sc[4], sc[5], sc[6], sc[7], bias_reg[t][2], bias_reg[t][3], scale, lg2e, nm, ones, ph[2], ph[3], lt);
      FTA_HOLD2(vtl[1], vth[1]);
      FTA_HOLD4(ph[4], ph[5], ph[6], ph[7]);
      // V^T operands of tile t (for the next iteration)
      if constexpr (t % G == 0) {
#pragma unroll
        for (int x = 0; x < 2; ++x) aTc[x] = aT[x] + (uint32_t)(PUB ? (kslot - 1) & (R - 1) : kslot) * SLOT_B;  // (tile t opens the stage the K reads entered one tile ago)
      }
      vtl[0] = lds_issue_tr4<(t % G) * 32 * D * 2>(aTc[0]);
      vth[0] = lds_issue_tr4<(t % G) * 32 * D * 2>(aTc[1]);
      vtl[1] = lds_issue_tr4<(t % G) * 32 * D * 2 + 16 * D * 2>(aTc[0]);
      vth[1] = lds_issue_tr4<(t % G) * 32 * D * 2 + 16 * D * 2>(aTc[1]);
      if constexpr (t == 0) {
        // the previous row's O^T is complete (its last MFMA was issued two blocks ago)
        FTA_PIN_V(acc);
        if (ir > 0) {
          if constexpr (S == 1) finish_row(); else merge_give();
        }
      }
      if constexpr (t == 2 && S > 1) {
        if (ir > 0) merge_take();
      }
      // S^T of tile t+1
      asm volatile("s_waitcnt lgkmcnt(4)" : "+v"(kf[0]), "+v"(kf[1]));
      {
        const u32x4* qq = (t == NKT - 1) ? qn : qf;
        mfma_new_v<T>(sn, as_half8(kf[0]), as_half8(qq[0]));
        fwd1_block4<T, 1>(sc[8], sc[9], sc[10], sc[11], bias_reg[t][4], bias_reg[t][5], scale, lg2e, nm, ones, ph[4], ph[5], lt);
        FTA_HOLD2(kf[0], qq[0]);
        mfma_acc_v<T>(sn, as_half8(kf[1]), as_half8(qq[1]));
        fwd1_block4<T, 2>(sc[12], sc[13], sc[14], sc[15], bias_reg[t][6], bias_reg[t][7], scale, lg2e, nm, ones, ph[6], ph[7], lt);
        FTA_HOLD2(kf[1], qq[1]);
      }

      if constexpr (t == 0) {
        l = lt;  // (no weight of the first tile exceeds 2^-6)
      } else {
        if (__builtin_expect(__builtin_amdgcn_ballot_w64(!(lt <= kFwd1Limit)) != 0, 0)) {
          // Some weight of this tile left the 16-bit range: move the reference to this tile's maximum
          // plus the margin, rescale O and l, and redo the tile's weights from the scores.
          float mx = -INFINITY;
#pragma unroll
          for (int r = 0; r < 16; r += 2) {
            float x0, x1;
            fwd1_scaled_pair<T>(x0, x1, sc[r], sc[r + 1], scale, bias_reg[t][r >> 1]);
            mx = __builtin_fmaxf(__builtin_fmaxf(mx, x0), x1);
          }
          const float d = __builtin_fmaxf(max_both_halves(mx) + kFwd1Margin - m_ref, 0.f);
          const float alpha = exp2_fast(-d * kLog2e);
          l *= alpha;
          asm volatile("s_nop 15\n\ts_nop 15" : "+v"(acc));  // (the O^T MFMAs of this iteration have completed)
#pragma unroll
          for (int r = 0; r < 16; ++r) acc[r] *= alpha;
          m_ref += d;
          nm = -m_ref * kLog2e;
          lt = 0.f;
#pragma unroll
          for (int r = 0; r < 16; r += 2) {
            float x0, x1;
            fwd1_scaled_pair<T>(x0, x1, sc[r], sc[r + 1], scale, bias_reg[t][r >> 1]);
            const float p0 = exp2_fast(__builtin_fmaf(x0, kLog2e, nm)), p1 = exp2_fast(__builtin_fmaf(x1, kLog2e, nm));
            ph[r >> 1] = T::pack(p0, p1);
            lt = T::sum2(ph[r >> 1], lt);
          }
          // (the row sum's dot product is read by another opcode from here on: three slots; the packed weights by the matrix core: two)
          asm volatile("s_nop 3" : "+v"(acc), "+v"(lt), "+v"(ph[0]), "+v"(ph[1]), "+v"(ph[2]), "+v"(ph[3]), "+v"(ph[4]), "+v"(ph[5]),
                       "+v"(ph[6]), "+v"(ph[7]));
        }
        l += lt;
      }
    });
    // row change: the row's sums go to the side (its last O^T MFMAs are issued by the next iteration),
    // the Q fragments of the next row (landed: the last barrier wait covered them) become current, and
    // those of the row after are asked for
    l_done = l;
    m_done = m_ref;
    if constexpr (ODD) s[0] = s[1];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) qf[ks] = qn[ks];
    asm volatile("" : "+v"(qf[0]), "+v"(qf[1]));
    q_issue(true);
  }

  // ---- epilogue: the last tile's O^T MFMAs, the last row
  asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(vtl[0]), "+v"(vth[0]), "+v"(vtl[1]), "+v"(vth[1]), "+v"(kf[0]), "+v"(kf[1]));
  mfma_acc_v<T>(acc, as_half8(u32x4{vtl[0][0], vtl[0][1], vth[0][0], vth[0][1]}), as_half8(u32x4{ph[0], ph[1], ph[2], ph[3]}));
  mfma_acc_v<T>(acc, as_half8(u32x4{vtl[1][0], vtl[1][1], vth[1][0], vth[1][1]}), as_half8(u32x4{ph[4], ph[5], ph[6], ph[7]}));
  asm volatile("s_nop 15\n\ts_nop 7" : "+v"(acc));
  if constexpr (S == 1) {
    finish_row();
  } else {
    merge_give();
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // (the record is in LDS: the compiler does not know that the statements above write it)
    __syncthreads();
    merge_take();
  }
  wait_vmem_all();  // (no copy may still be in flight when the workgroup gives its LDS back)
}

}  // namespace fta

// Launches the instance (NKT, W, G, S) if it is the plan's.  (The instances that mask a row's tail, `tl`, also read the bias
// entry by entry where they must.)
#define FTA_FWD1_CASE(NN, WW, GG, SS)                                                                       \
  if (pl.NKT == NN && pl.QB * SS == WW && pl.KT == 32 * GG && pl.S == SS) {                                 \
    if (dtype == kBF16)                                                                                     \
      return tl ? launch_kernel(fta_fwd1_kernel<BF16, NN, true, WW, GG, SS>, p, grid, block, pl.smem, st)   \
                : launch_kernel(fta_fwd1_kernel<BF16, NN, false, WW, GG, SS>, p, grid, block, pl.smem, st); \
    return tl ? launch_kernel(fta_fwd1_kernel<F16, NN, true, WW, GG, SS>, p, grid, block, pl.smem, st)      \
              : launch_kernel(fta_fwd1_kernel<F16, NN, false, WW, GG, SS>, p, grid, block, pl.smem, st);    \
  }
