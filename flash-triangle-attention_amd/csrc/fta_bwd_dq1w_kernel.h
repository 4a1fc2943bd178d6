// dQ + dBias partials at head dim 64 with both halves of a key range of 256 to 512 keys in one workgroup: the schedule of
// fta_bwd_dq1_kernel.h (one wave per SIMD, order of the instructions as written) for two slabs.
//
//   * workgroup = 64 queries x 256 to 512 keys, wave = 32 queries x 4, 6 or 8 tiles of 32 keys.  dbias (128) and bias (64), the dQ sums
//     (32) and the K operands (16) live in accumulation registers;
//   * K/V stages of two tiles per slab (32 KB) in a ring of four: a stage is copied two barriers ahead of the one that publishes it.  A
//     barrier every second tile; it sits two tiles ahead of the published stage's first use and frees the slot of the stage before the current one;
//   * the registers of an operand are filled again right behind the MFMA that consumes it: 16 reads an iteration, in the order of
//     their use one iteration later, so that each wait leaves the last 12 in flight;
//   * slab s finishes d = 32 s .. +31 of the row: its operands of K^T are addressed so that acc[0] is its own half of d and
//     acc[1] the partner's, which goes through LDS once a row (the halves meet in fp32).  A wave writes its record in iteration 0 of the next row
//     and its partner reads it in iterations 2 and 3; barriers open every even iteration.  So write -> read has the barrier of iteration 2 between, and
//     read -> next row's write that of iteration 0.  The last row's record is written behind the loop: six and eight tiles have the
//     barrier of iteration 4 between the read and that, four tiles need one of their own there.
//
// Bound: matrix core and power (18 MFMAs a tile), issue (166 instructions) and memory in about equal parts: 1.40 to 1.45 ms at B2 H8 L512
// (averages of kernel traces over devices), 1200 cycles a tile.  Two launches over 256 keys each, of workgroups of 128 queries, read Q, dO, O and
// wrote dQ twice: 2 x 856 us on the device where this takes 1408.
#pragma once
#include "fta_bwd_dq1_kernel.h"

namespace fta {

typedef float floatx4 __attribute__((ext_vector_type(4)));

// Waits for all but the last N LDS reads and ties the registers of older ones to that point.
template <int N>
__device__ __forceinline__ void dq1w_wait_kt(u32x2 (&lo)[2], u32x2 (&hi)[2]) {
  asm volatile("s_waitcnt lgkmcnt(%4)" : "+v"(lo[0]), "+v"(hi[0]), "+v"(lo[1]), "+v"(hi[1]) : "n"(N));
}
template <int N>
__device__ __forceinline__ void dq1w_wait_k(u32x4 (&k)[4]) {
  asm volatile("s_waitcnt lgkmcnt(%4)" : "+a"(k[0]), "+a"(k[1]), "+a"(k[2]), "+a"(k[3]) : "n"(N));
}
template <int N>
__device__ __forceinline__ void dq1w_wait_v(u32x4 (&v)[4]) {
  asm volatile("s_waitcnt lgkmcnt(%4)" : "+v"(v[0]), "+v"(v[1]), "+v"(v[2]), "+v"(v[3]) : "n"(N));
}
// 16 bytes per lane to a uniform base plus a lane offset, with no 64-bit address per lane.  (The store reads its data for two slots more.)
template <int OFF>
__device__ __forceinline__ void store_dq_piece(uint32_t voff, u32x4 d, const void* base) {
  asm volatile("global_store_dwordx4 %0, %1, %2 offset:%3\n\ts_nop 1" ::"v"(voff), "v"(d), "s"(base), "n"(OFF) : "memory");
}
template <int OFF>
__device__ __forceinline__ void dq1w_put(uint32_t addr, floatx4 w) {
  asm volatile("ds_write_b128 %0, %1 offset:%2" ::"v"(addr), "v"(w), "n"(OFF) : "memory");
}
template <int N>
__device__ __forceinline__ void wait_vmem() {
  __builtin_amdgcn_s_waitcnt(0x0F70 | (N & 15) | ((N >> 4) << 14));
}

// NKT: 32-key tiles per slab.  LATER: earlier key ranges' launches left a partial dQ to add to.  Rows of any length and bias rows on any 2-byte
// boundary (keys beyond the row masked, queries beyond it computed on copies of the last one and not stored): instances for whole rows alone
// came out of the compiler with spilled registers and took 1384 us where these take 1360 (B2 H8 L512).
template <class T, int NKT, bool LATER>
__global__ void __launch_bounds__(256) fta_bwd_dq1w_kernel(const BwdParams p) {
  static_assert(NKT == 4 || NKT == 6 || NKT == 8, "whole stages of two tiles");
  constexpr int D = 64, KS = 4, DT = 2, SK = 2, QR = 64;
  constexpr int NST = NKT / 2, R = 4;           // stages per row, ring slots
  constexpr int SROWS = SK * 64;                // rows of a staged K (or V) tile
  constexpr uint32_t TILE_B = SROWS * D * 2, SLOT_B = 2 * TILE_B, QTILE_B = QR * D * 2;
  constexpr int NM = 18;                        // MFMAs per tile
  constexpr int SLAB = NKT * 32;
  constexpr int CF = NKT < 8 ? kA : kV;         // register file of the constant operands
  extern __shared__ __attribute__((aligned(16))) char smem_raw[];
  half_t* qbuf = reinterpret_cast<half_t*>(smem_raw + R * SLOT_B);  // Q rows, dO rows of one L1 row

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int slab = wave % SK, qb = wave / SK;
  const WorkId id = work_id(p.nqg, p.nchunks, p.H, p.head_inner);
  const int qg = id.group, chunk = id.chunk, b = id.b, h = id.h, bh = b * p.H + h;
  const int i0 = chunk * p.rows_per_chunk;
  const int nrows = min(p.rows_per_chunk, p.L1 - i0);
  if (nrows <= 0) return;
  const int q0 = qg * QR + qb * 32;
  const int key0 = p.kr0 + slab * SLAB;
  const float scale = p.scale, sl2 = p.scale * kLog2e;
  const int64_t step_k = hold_scalar(p.ks[2] * 2), step_v = hold_scalar(p.vs[2] * 2), step_q = hold_scalar(p.qs[2] * 2),
                step_do = hold_scalar(p.dos[2] * 2), step_o = hold_scalar(p.os[2] * 2), step_dq = hold_scalar(p.dqs[2] * 2),
                step_kst = hold_scalar(p.ks[3] * 128), step_vst = hold_scalar(p.vs[3] * 128);  // (from one stage to the next: 64 keys)
  const int step_lse = p.L2 * 4, step_aux = p.L2p * 8;
  auto advance = [](auto*& ptr, int64_t bytes) {
    using P = std::remove_reference_t<decltype(ptr)>;
    ptr = (P)((const char*)ptr + bytes);
  };

  // ---- staging: stage n = (row n / NST, part n % NST) lives in ring slot n % R.  Every wave issues four copies of a stage's K and of its V, and
  // two of a row's Q and of its dO; past the chunk's last row the row pointers stop, and the last row is copied again into slots that nothing reads.
  const int qrow0 = min(qg * QR, p.L2 - 1);  // (the window starts at a real row)
  int srow, schunk;                      // copy u of a wave brings row srow + 32 u of the stage
  uint32_t goffk, goffv;                 // (the first slab's copies: the second starts 32 rows further on)
  uint32_t goffq[2], goffdo[2];
  auto set_offsets = [&](int ln) {
    srow = wave * 8 + (ln >> 3);
    schunk = swz_slot<D>(srow, ln & 7) * 16;  // (the swizzle looks at the row's low four bits)
    goffk = (uint32_t)((int64_t)srow * p.ks[3] * 2 + schunk);
    goffv = (uint32_t)((int64_t)srow * p.vs[3] * 2 + schunk);
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int grow = min(qg * QR + srow + 32 * u, p.L2 - 1) - qrow0;
      goffq[u] = (uint32_t)((int64_t)grow * p.qs[3] * 2 + schunk);
      goffdo[u] = (uint32_t)((int64_t)grow * p.dos[3] * 2 + schunk);
    }
  };
  set_offsets(lane);
  // (The second slab may end beyond the row, whose last key is copied again; the first keys of every stage of both slabs' windows are real: the
  // tiles end less than 128 keys beyond the row, and a slab has 128 or more)
  const uint32_t kstride2 = (uint32_t)(p.ks[3] * 2), vstride2 = (uint32_t)(p.vs[3] * 2);
  const int klast = p.L2 - 1 - p.kr0;
  const uint32_t lds0 = lds_addr_of(smem_raw), ldsq = lds0 + R * SLOT_B, ldsx = ldsq + 2 * QTILE_B;
  const uint32_t wofs = (uint32_t)wave * 1024u;
  const half_t* kst = p.k + b * p.ks[0] + h * p.ks[1] + (int64_t)i0 * p.ks[2] + (int64_t)p.kr0 * p.ks[3];
  const half_t* vst = p.v + b * p.vs[0] + h * p.vs[1] + (int64_t)i0 * p.vs[2] + (int64_t)p.kr0 * p.vs[3];
  const half_t* krow = kst;
  const half_t* vrow = vst;
  const half_t* qcur = p.q + b * p.qs[0] + h * p.qs[1] + (int64_t)i0 * p.qs[2] + (int64_t)qrow0 * p.qs[3];
  const half_t* docur = p.dout + b * p.dos[0] + h * p.dos[1] + (int64_t)i0 * p.dos[2] + (int64_t)qrow0 * p.dos[3];
  int row_iss = 0, cur_slot = 0;
  uint32_t iss_dst = 0;
  auto stage_begin = [&](auto sc, bool first) {
    constexpr int s = decltype(sc)::value;
    if constexpr (s == 0) {
      if (!first && row_iss + 1 < nrows) {
        ++row_iss;
        advance(krow, step_k); advance(vrow, step_v);
      }
      kst = krow; vst = vrow;
    } else {
      advance(kst, step_kst); advance(vst, step_vst);
    }
    iss_dst = lds0 + (uint32_t)cur_slot * SLOT_B + wofs;
    cur_slot = (cur_slot + 1) % R;
  };
  auto kv_copy = [&](auto sc, auto cc) {  // copy c of stage s of a row
    constexpr int s = decltype(sc)::value, c = decltype(cc)::value, u = c % 4;
    constexpr bool isv = c >= 4;
    uint32_t off = isv ? goffv : goffk;
    const half_t* base = isv ? vst : kst;
    if constexpr (u == 1) advance(base, (isv ? step_vst : step_kst) >> 1);
    if constexpr (u >= 2) {
      int row = srow;
      asm volatile("" : "+v"(row));  // (formed here: kept for every copy, the offsets would not fit the registers)
      off = (uint32_t)min(row + (32 * u - 64 + SLAB), klast - 64 * s) * (isv ? vstride2 : kstride2) + (uint32_t)schunk;
    }
    dma16s_at<(isv ? TILE_B : 0u) + (uint32_t)u * 4096u>(off, uniform_ptr(base), iss_dst);
  };
  auto q_copy = [&](auto cc) {  // copy c of a row's Q and dO
    constexpr int c = decltype(cc)::value;
    dma16s_at<(c < 2 ? 0u : QTILE_B) + (uint32_t)(c % 2) * 4096u>(c < 2 ? goffq[c % 2] : goffdo[c % 2], uniform_ptr(c < 2 ? qcur : docur), ldsq + wofs);
  };

  // ---- prologue ------------------------------------------------------------------------------
  static_for<0, 4>(q_copy);
  static_for<0, R - 1>([&](auto nc) {
    constexpr int n = decltype(nc)::value;
    stage_begin(std::integral_constant<int, n % NST>{}, n == 0);
    static_for<0, 8>([&](auto cc) { kv_copy(std::integral_constant<int, n % NST>{}, cc); });
  });
  // stationary bias (times log2 e, MFMA B operands of S^T += E_u * bias^T_u)
  u32x4 bias4[NKT][2];
  {
    // while those copies fly; it changes lanes in the ring slot that nothing is copied to yet
    static_assert(4 * 4096 <= SLOT_B, "4 KB for every wave's bias");
    u32x2 even = {0u, 0u};
    const half_t* bias_bh = p.bias + b * p.bs[0] + h * p.bs[1];
    char* turn = smem_raw + (R - 1) * SLOT_B + wave * 4096;
    auto conv = [](uint32_t u) { return T::bias_log2(u); };
    auto sink = [&](int tt, int g, u32x2 v) {
      if (g % 2 == 0) { even = v; return; }
      u32x4& d = bias4[tt][g / 2];
      d = u32x4{even[0], even[1], v[0], v[1]};
      asm volatile("" : "+a"(d));  // parked in accumulation registers for the whole kernel
    };
    load_bias_tiles<NKT / 2, 2, true, false>(bias_bh, p.bs[2], q0, p.L2, F16::kBeyond2, turn, lane, [=](int c) { return key0 + 64 * c; }, conv, sink);
  }
  // What the row loop keeps per lane is formed behind the bias, whose 128 registers in flight would else push it into scratch memory.
  int ln = lane;
  asm volatile("" : "+v"(ln));
  set_offsets(ln);
  const int hh = ln >> 5, l32 = ln & 31;
  FragOffsets<D> fo;
  fo.init(ln);
  // dBias sums and one-hot selectors: see fta_bwd_dq1_kernel
  floatx16 dbacc[NKT];
#pragma unroll
  for (int tt = 0; tt < NKT; ++tt)
#pragma unroll
    for (int r = 0; r < 16; ++r) dbacc[tt][r] = 0.f;
  u32x4 E[2];
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const int rel = l32 - 16 * u;
    const bool valid = (rel >= 0) && (rel < 16) && (((rel >> 2) & 1) == hh);
    const int e = 4 * (rel >> 3) + (rel & 3);
    half8_t one;
#pragma unroll
    for (int x = 0; x < 8; ++x) one[x] = (valid && x == e) ? (half_t)1.0f : (half_t)0.0f;
    E[u] = __builtin_bit_cast(u32x4, one);
  }
  // (-lse and -delta sit in words 0 and 1 of one B operand; the factors of either in A operands of their own, see aug_ones)
  u32x4 onesS = {kLseOnes, 0u, 0u, 0u}, onesD = {0u, T::kDeltaOnes, 0u, 0u};
  if constexpr (CF == kA) asm volatile("s_nop 1" : "+a"(E[0]), "+a"(E[1]), "+a"(onesS), "+a"(onesD));
  else asm volatile("s_nop 1" : "+v"(E[0]), "+v"(E[1]), "+v"(onesS), "+v"(onesD));

  // O fragments and lse of a row, for its constants: straight into registers
  u32x4 of_n[KS];
  float lse_n = 0.f;
  const half_t* ocur = p.o + b * p.os[0] + h * p.os[1] + (int64_t)i0 * p.os[2];
  const float* lcur = p.lse + ((int64_t)bh * p.L1 + i0) * p.L2;
  const bool qvalid = q0 + l32 < p.L2;
  const int qread = min(q0 + l32, p.L2 - 1);
  const uint32_t voff_o = (uint32_t)(((int64_t)qread * p.os[3] + 8 * hh) * 2), voff_l = (uint32_t)qread * 4u;
  auto rowconst_issue = [&](int row) {
    if (row > 0 && row < nrows) { advance(ocur, step_o); advance(lcur, step_lse); }
    const void* ob = uniform_ptr(ocur);
    const void* lb = uniform_ptr(lcur);
    static_for<0, KS>([&](auto kc) { constexpr int ks = decltype(kc)::value; load_piece<kV, 32 * ks>(of_n[ks], voff_o, ob); });
    asm volatile("global_load_dword %0, %1, %2" : "=v"(lse_n) : "v"(voff_l), "s"(lb) : "memory");
  };

  half8_t qf[KS], dof[KS];
  u32x4 aug = {0u, 0u, 0u, 0u};
  uint32_t* auxcur = p.aux + (((int64_t)bh * p.L1 + i0) * p.L2p) * 2;
  const uint32_t voff_aux = (uint32_t)(q0 + l32) * 8u;
  const bool aux_wave = (slab == 0) && (p.kr0 == 0);
  auto row_operands = [&](int ir) {
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      qf[ks] = T::scale8(lds_frag<D>(qbuf, qb * 32, fo, ks), sl2);
      dof[ks] = lds_frag<D>(qbuf + QR * D, qb * 32, fo, ks);
    }
    asm volatile("" : "+v"(of_n[0]), "+v"(of_n[1]), "+v"(of_n[2]), "+v"(of_n[3]), "+v"(lse_n));  // (landed: a barrier's wait has covered them)
    float dpart = 0.f;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const u32x4 d4 = __builtin_bit_cast(u32x4, dof[ks]);
#pragma unroll
      for (int e = 0; e < 4; ++e) dpart = T::dot2(of_n[ks][e], d4[e], dpart);
    }
    const float nl = qvalid ? folded_lse(lse_n) : kBiasFloorLog2, nd = -sum_both_halves(dpart);
    const uint32_t ws = split_2048(nl), wd = T::delta_pair(nd);
    if (ir > 0 && ir < nrows) advance(auxcur, step_aux);
    if (aux_wave && hh == 0) {
      const u32x2 w = {ws, wd};
      const void* ab = uniform_ptr(auxcur);
      asm volatile("global_store_dwordx2 %0, %1, %2" ::"v"(voff_aux), "v"(w), "s"(ab) : "memory");
    }
    aug = u32x4{hh ? 0u : ws, hh ? 0u : wd, 0u, 0u};
    asm volatile("" : "+v"(aug));
  };

  floatx16 s_cur, dp_cur, s_nxt;
  uint32_t dsp_prev[8], dsp_cur[8];
  u32x4 kf[KS], vf[KS];           // K, V operands of the next tile
  u32x2 ktlo[2][DT], kthi[2][DT];  // K^T operands of the previous one
  floatx16 acc[DT];
  float keep[16];                  // this wave's half of the finished row
  u32x4 got[2];                    // the partner's share of half of that

  // per-lane LDS addresses of the operand reads inside this wave's part of a slot
  uint32_t aK[KS], aT[DT][2];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) aK[ks] = lds0 + (uint32_t)(slab * 64 * D + fo.a[ks]) * 2u;
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)  // (acc[0]: this slab's half of d)
#pragma unroll
    for (int x = 0; x < 2; ++x) aT[dt][x] = lds0 + (uint32_t)(slab * 64 * D + fo.t[dt][x]) * 2u;
  if (slab == 1)
#pragma unroll
    for (int x = 0; x < 2; ++x) { const uint32_t t = aT[0][x]; aT[0][x] = aT[1][x]; aT[1][x] = t; }
  const uint32_t xput = ldsx + (uint32_t)wave * 4096u + (uint32_t)ln * 16u, xget = ldsx + (uint32_t)(wave ^ 1) * 4096u + (uint32_t)ln * 16u;

  rowconst_issue(0);
  wait_vmem_all();
  __syncthreads();
  row_operands(0);
#pragma unroll
  for (int r = 0; r < 8; ++r) dsp_prev[r] = 0u;
#pragma unroll
  for (int u = 0; u < 2; ++u)
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) { ktlo[u][dt] = u32x2{0u, 0u}; kthi[u][dt] = u32x2{0u, 0u}; }
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[dt][r] = 0.f;
#pragma unroll
  for (int x = 0; x < 2; ++x) got[x] = u32x4{0u, 0u, 0u, 0u};
#pragma unroll
  for (int x = 0; x < 16; ++x) keep[x] = 0.f;
  {
    const half_t* cK = reinterpret_cast<const half_t*>(smem_raw) + slab * 64 * D;
    const half_t* cV = cK + TILE_B / 2;
    asm volatile("s_nop 1" : "+v"(qf[0]), "+v"(qf[1]), "+v"(qf[2]), "+v"(qf[3]));
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      if (ks == 0) {
        mfma_new_v<T>(s_cur, lds_frag<D>(cK, 0, fo, ks), qf[ks]);
        mfma_new_v<T>(dp_cur, lds_frag<D>(cV, 0, fo, ks), dof[ks]);
      } else {
        mfma_acc_v<T>(s_cur, lds_frag<D>(cK, 0, fo, ks), qf[ks]);
        mfma_acc_v<T>(dp_cur, lds_frag<D>(cV, 0, fo, ks), dof[ks]);
      }
    }
    mfma_rf<F16, CF, kA, kV, 1>(s_cur, E[0], bias4[0][0]);
    mfma_rf<F16, CF, kA, kV, 1>(s_cur, E[1], bias4[0][1]);
    mfma_rf<F16, CF, kV, kV, 1>(s_cur, onesS, aug);
    mfma_rf<T, CF, kV, kV, 1>(dp_cur, onesD, aug);
    asm volatile("s_nop 15\n\ts_nop 7" : "+v"(s_cur), "+v"(dp_cur));  // results land before anything reads them
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {  // K, V operands of tile 1, settled here
      kf[ks] = __builtin_bit_cast(u32x4, lds_frag<D>(cK, 32, fo, ks));
      vf[ks] = __builtin_bit_cast(u32x4, lds_frag<D>(cV, 32, fo, ks));
      asm volatile("" : "+a"(kf[ks]), "+v"(vf[ks]));
    }
  }

  // The finished row: the halves summed, scaled, rounded, what an earlier key range left added, and stored in 16-byte pieces (lane (query, hh) of
  // slab s gets d = 32 s + 16 y + 8 hh .. +7 of piece y).
  half_t* dqcur = p.dq + b * p.dqs[0] + h * p.dqs[1] + (int64_t)i0 * p.dqs[2];
  const uint32_t voff_dq = (uint32_t)(((int64_t)qread * p.dqs[3] + 32 * slab + 8 * hh) * 2);
  u32x4 old[2] = {u32x4{0u, 0u, 0u, 0u}, u32x4{0u, 0u, 0u, 0u}};
  auto old_issue = [&]() {
    const void* rb = uniform_ptr(dqcur);
    load_piece<kV, 0>(old[0], voff_dq, rb);
    load_piece<kV, 32>(old[1], voff_dq, rb);
  };
  auto store_piece = [&](auto yc) {
    constexpr int y = decltype(yc)::value;
    float a[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) a[e] = (keep[8 * y + e] + __builtin_bit_cast(float, (uint32_t)got[e / 4][e % 4])) * scale;
    uint32_t x0 = T::pack(a[0], a[1]), x1 = T::pack(a[2], a[3]), y0 = T::pack(a[4], a[5]), y1 = T::pack(a[6], a[7]);
    auto r0 = __builtin_amdgcn_permlane32_swap(x0, y0, false, false);
    auto r1 = __builtin_amdgcn_permlane32_swap(x1, y1, false, false);
    u32x4 out = {(uint32_t)r0[0], (uint32_t)r1[0], (uint32_t)r0[1], (uint32_t)r1[1]};
    if constexpr (LATER)
#pragma unroll
      for (int w = 0; w < 4; ++w) out[w] = T::add2(out[w], old[y][w]);
    const void* rb = uniform_ptr(dqcur);
    if (qvalid) store_dq_piece<32 * y>(voff_dq, out, rb);
  };
  auto take_own = [&]() {
    FTA_PIN_A(acc[0]);
#pragma unroll
    for (int x = 0; x < 16; ++x) keep[x] = acc[0][x];
#pragma unroll
    for (int x = 0; x < 16; ++x) asm volatile("" : "+v"(keep[x]));
  };
  auto give_other = [&]() {
    FTA_PIN_A(acc[1]);
    static_for<0, 4>([&](auto xc) {
      constexpr int x = decltype(xc)::value;
      dq1w_put<x * 1024>(xput, __builtin_shufflevector(acc[1], acc[1], 4 * x, 4 * x + 1, 4 * x + 2, 4 * x + 3));
    });
  };
  auto get_share = [&](auto yc) {
    constexpr int y = decltype(yc)::value;
    got[0] = lds_issue_b128<y * 2048>(xget);
    got[1] = lds_issue_b128<y * 2048 + 1024>(xget);
  };
  const bool stores_dq = q0 < p.L2;  // (this wave's part of a row is stored)

  int rd_slot = 0;  // ring slot that the K^T reads are in; K and V are read one ahead of it
#pragma nounroll
  for (int ir = 0; ir < nrows; ++ir) {
    static_for<0, NKT>([&](auto gc) {
      constexpr int g = decltype(gc)::value, per = g / 2;
      // -- every second tile: the stage that tile g + 2 starts is published, and the slot of the stage that ended refilled.  Waits for that stage's
      //    copies, issued two barriers ago: all but the eight (in a row's first period twelve) of the stage after it and what the last period stored;
      //    and, so that the slot is free, for the K^T operands of tile g - 1 (eight reads of later tiles behind them).
      if constexpr (g % 2 == 0) {
        constexpr int last = (per + NST - 1) % NST;                                            // the period before
        constexpr int kept = 8 + (last == 0 && NST > 2 ? 4 : 0);
        asm volatile("s_waitcnt lgkmcnt(8)" ::: "memory");
        if constexpr (last == 1 && NST == 4) {          // dQ, stored in iteration 3
          if (ir > 0 && stores_dq) wait_vmem<kept + 2>();
          else wait_vmem<kept>();
        } else if constexpr (last == NST - 1 && NST > 2) {  // the row constants, stored in the last iteration
          if (aux_wave) wait_vmem<kept + 1>();
          else wait_vmem<kept>();
        } else {
          wait_vmem<kept>();
        }
        __syncthreads();
        if constexpr (LATER && g == 2) asm volatile("" : "+v"(old[0]), "+v"(old[1]));  // (landed: twelve copies behind them)
        if constexpr (LATER && g == 0) old_issue();
        if constexpr (per == NST - 2) rowconst_issue(ir + 1);
        if constexpr (g == 2) get_share(std::integral_constant<int, 0>{});
        stage_begin(std::integral_constant<int, (per + 3) % NST>{}, false);
        if constexpr (g == 0)
          if (ir + 1 < nrows) { advance(qcur, step_q); advance(docur, step_do); }
      }
      if constexpr (g == NKT - 1) row_operands(ir + 1);

      // -- LDS reads, each behind the MFMA that consumes what the register holds: K^T of tile g (for the next iteration's dS of tile g), K and V
      //    of tile g + 2
      constexpr int gn = (g + 1) % NKT, g2 = (g + 2) % NKT;
      constexpr int offc = (g % 2) * 32 * D * 2, off2 = (g2 % 2) * 32 * D * 2;
      if constexpr (g % 2 == 0) {  // (the first iteration of a stage: K^T from its slot, K and V from the next one)
        const int kv_slot = (rd_slot + 1) % R;
        const uint32_t up_kv = kv_slot == 0 ? (uint32_t)(0 - (R - 1) * (int)SLOT_B) : SLOT_B;
        const uint32_t up_t = ir == 0 && g == 0 ? 0u : rd_slot == 0 ? (uint32_t)(0 - (R - 1) * (int)SLOT_B) : SLOT_B;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) aK[ks] += up_kv;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) { aT[dt][0] += up_t; aT[dt][1] += up_t; }
        rd_slot = kv_slot;
      }
      auto refill_kt = [&](auto uc, auto dc) {
        constexpr int u = decltype(uc)::value, dt = decltype(dc)::value;
        ktlo[u][dt] = lds_issue_tr4<offc + u * 16 * D * 2>(aT[dt][0]);
        kthi[u][dt] = lds_issue_tr4<offc + u * 16 * D * 2>(aT[dt][1]);
      };
      auto valu_pair = [&](auto kc) {
        constexpr int k = decltype(kc)::value;
        dsp_cur[k] = ds_pair<T, false>(s_cur[2 * k], s_cur[2 * k + 1], dp_cur[2 * k], dp_cur[2 * k + 1]);
      };
      // what follows MFMA m: its share of the vector-ALU work of tile g, and in the gaps a copy or a piece of the row change
      auto after = [&](auto mc) {
        constexpr int m = decltype(mc)::value;
        constexpr int pair_of[NM] = {-1, -1, 0, 1, 2, -1, 3, 4, 5, 6, -1, 7, -1, -1, -1, -1, -1, -1};
        if constexpr (pair_of[m] >= 0) valu_pair(std::integral_constant<int, pair_of[m]>{});
        constexpr int slot_of[NM] = {0, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1, 1, 2, 3, 4, 5, -1};
        constexpr int at = slot_of[m];
        if constexpr (at >= 0) {
          constexpr bool six = (per == 0);  // (a row's first period also brings the next row's Q and dO)
          constexpr int k = six ? at : at < 3 ? at : at == 4 ? 3 : -1;
          if constexpr (k >= 0) {
            constexpr int c = (g % 2) * (six ? 6 : 4) + k;
            constexpr int kv = NST > 2 ? c : six ? c - 4 : c, qc = NST > 2 ? c - 8 : c;  // (two stages a row: Q and dO first, the next barrier needs them)
            if constexpr (six && (NST > 2 ? c >= 8 : c < 4)) q_copy(std::integral_constant<int, qc>{});
            else kv_copy(std::integral_constant<int, (per + 3) % NST>{}, std::integral_constant<int, kv>{});
          }
        }
        if constexpr (g == 0 && m == 12) take_own();
        if constexpr (g == 0 && m == 14) give_other();
        if constexpr (g == 3 && (m == 12 || m == 17)) {
          // (the first half was read ahead of an iteration's sixteen, the second has the four of this one's V behind it)
          if constexpr (m == 12) asm volatile("" : "+v"(got[0]), "+v"(got[1]));
          else asm volatile("s_waitcnt lgkmcnt(4)" : "+v"(got[0]), "+v"(got[1]));
          if (ir > 0) store_piece(std::integral_constant<int, m == 17>{});
          if constexpr (m == 12) get_share(std::integral_constant<int, 1>{});
          else if (ir > 0) advance(dqcur, step_dq);
        }
      };
      // -- MFMAs that consume dS of tile g-1
      constexpr int gp = (g + NKT - 1) % NKT;
      static_for<0, 2>([&](auto uc) {
        constexpr int u = decltype(uc)::value;
        const u32x4 ds = {dsp_prev[4 * u], dsp_prev[4 * u + 1], dsp_prev[4 * u + 2], dsp_prev[4 * u + 3]};
        const half8_t db = as_half8(ds);
        mfma_rf<T, CF, kV, kA, (u == 0) ? 1 : 0>(dbacc[gp], E[u], ds);
        after(std::integral_constant<int, 3 * u>{});
        dq1w_wait_kt<12>(ktlo[u], kthi[u]);
        static_for<0, DT>([&](auto dc) {
          constexpr int dt = decltype(dc)::value;
          const half8_t kt = as_half8(u32x4{ktlo[u][dt][0], ktlo[u][dt][1], kthi[u][dt][0], kthi[u][dt][1]});
          if constexpr (g == 1 && u == 0) mfma_restart_a<T>(acc[dt], kt, db);
          else mfma_acc_a_late<T>(acc[dt], kt, db);  // (its operand may just have been put together)
          refill_kt(uc, dc);
          after(std::integral_constant<int, 3 * u + 1 + dt>{});
        });
      });
      // -- MFMAs that produce S^T of tile g+1; behind the last vector-ALU pair those that produce dP^T, in the registers that dP^T of tile g
      //    leaves (three tiles in registers instead of four, which would not fit)
      dq1w_wait_k<12>(kf);
      static_for<0, KS>([&](auto kc) {
        constexpr int ks = decltype(kc)::value;
        mfma_rf<T, kA, kV, kV, (ks == 0) ? 3 : 0>(s_nxt, kf[ks], __builtin_bit_cast(u32x4, qf[ks]));
        kf[ks] = lds_issue_b128_a<off2>(aK[ks]);
        after(std::integral_constant<int, 6 + ks>{});
      });
      mfma_rf<F16, CF, kA, kV, 0>(s_nxt, E[0], bias4[gn][0]);
      after(std::integral_constant<int, 10>{});
      mfma_rf<F16, CF, kA, kV, 0>(s_nxt, E[1], bias4[gn][1]);
      after(std::integral_constant<int, 11>{});
      mfma_rf<F16, CF, kV, kV, 0>(s_nxt, onesS, aug);
      after(std::integral_constant<int, 12>{});
      dq1w_wait_v<12>(vf);
      static_for<0, KS>([&](auto kc) {
        constexpr int ks = decltype(kc)::value;
        if constexpr (ks == 0) mfma_new_v<T>(dp_cur, as_half8(vf[ks]), dof[ks]);
        else mfma_acc_v<T>(dp_cur, as_half8(vf[ks]), dof[ks]);
        vf[ks] = lds_issue_b128<off2 + (int)TILE_B>(aK[ks]);
        after(std::integral_constant<int, 13 + ks>{});
      });
      mfma_rf<T, CF, kV, kV, 0>(dp_cur, onesD, aug);
      after(std::integral_constant<int, 17>{});
      FTA_PIN_V(s_nxt);  // no copy of the new tile may be placed before this point
      FTA_PIN_V(dp_cur);
      s_cur = s_nxt;
#pragma unroll
      for (int r = 0; r < 8; ++r) dsp_prev[r] = dsp_cur[r];
    });
    // (nothing may copy registers with reads still in flight: settle them before the loop turns)
    dq1w_wait_kt<0>(ktlo[0], kthi[0]);
    dq1w_wait_kt<0>(ktlo[1], kthi[1]);
    dq1w_wait_k<0>(kf);
    dq1w_wait_v<0>(vf);
  }

  // ---- epilogue: dS of the last tile, the last dQ row, the dBias tile -----------------------------
  asm volatile("s_nop 7" : "+v"(s_cur), "+v"(dp_cur));  // (the look-ahead MFMAs still write their tile)
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const half8_t db = as_half8(u32x4{dsp_prev[4 * u], dsp_prev[4 * u + 1], dsp_prev[4 * u + 2], dsp_prev[4 * u + 3]});
    dbacc[NKT - 1] = T::mfma(as_half8(E[u]), db, dbacc[NKT - 1]);
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) acc[dt] = T::mfma(as_half8(u32x4{ktlo[u][dt][0], ktlo[u][dt][1], kthi[u][dt][0], kthi[u][dt][1]}), db, acc[dt]);
  }
  if constexpr (LATER) old_issue();
  if constexpr (NKT == 4) __syncthreads();  // (the partner has read the record of the row before: no barrier of the loop lies behind iteration 3)
  {
    float* out = reinterpret_cast<float*>(smem_raw + R * SLOT_B + 2 * QTILE_B) + wave * 1024 + ln * 4;
    const float* in = reinterpret_cast<const float*>(smem_raw + R * SLOT_B + 2 * QTILE_B) + (wave ^ 1) * 1024 + ln * 4;
#pragma unroll
    for (int x = 0; x < 16; ++x) keep[x] = acc[0][x];
#pragma unroll
    for (int x = 0; x < 16; ++x) out[(x / 4) * 256 + x % 4] = acc[1][x];
    wait_vmem_all();  // (no copy may still be in flight when the workgroup gives its LDS back)
    __syncthreads();
    if constexpr (LATER) asm volatile("" : "+v"(old[0]), "+v"(old[1]));
    static_for<0, 2>([&](auto yc) {
      constexpr int y = decltype(yc)::value;
      got[0] = *reinterpret_cast<const u32x4*>(in + 2 * y * 256);
      got[1] = *reinterpret_cast<const u32x4*>(in + (2 * y + 1) * 256);
      store_piece(yc);
    });
  }

  float* part = p.partial + (((int64_t)chunk * p.B * p.H + bh) * p.L2p + (q0 + l32)) * p.L2p + key0 + 4 * hh;
#pragma unroll
  for (int tt = 0; tt < NKT; ++tt)
#pragma unroll
    for (int rg = 0; rg < 4; ++rg) {
      // (bf16: the selector of the MFMA is worth 2^-7, see kOneHotInv; the reduction scales the sums back)
      float4 w = {dbacc[tt][4 * rg], dbacc[tt][4 * rg + 1], dbacc[tt][4 * rg + 2], dbacc[tt][4 * rg + 3]};
      *reinterpret_cast<float4*>(part + tt * 32 + rg * 8) = w;
    }
}

template <class T>
inline hipError_t launch_dq1w_range(const BwdParams& p, int range, dim3 grid, size_t smem, hipStream_t st) {
  // (a first range is the row's longest: 384 keys at least)
  if (range == 512 && p.kr0 == 0) return launch_kernel(fta_bwd_dq1w_kernel<T, 8, false>, p, grid, dim3(256), smem, st);
  if (range == 384 && p.kr0 == 0) return launch_kernel(fta_bwd_dq1w_kernel<T, 6, false>, p, grid, dim3(256), smem, st);
  if (range == 512) return launch_kernel(fta_bwd_dq1w_kernel<T, 8, true>, p, grid, dim3(256), smem, st);
  if (range == 384) return launch_kernel(fta_bwd_dq1w_kernel<T, 6, true>, p, grid, dim3(256), smem, st);
  if (range == 256 && p.kr0 != 0) return launch_kernel(fta_bwd_dq1w_kernel<T, 4, true>, p, grid, dim3(256), smem, st);
  return hipErrorInvalidConfiguration;
}

hipError_t launch_dq1w_bf16(const BwdParams& p, int range, dim3 grid, size_t smem, hipStream_t st);  // (fta_bwd_dq1_bf16.hip)

}  // namespace fta
