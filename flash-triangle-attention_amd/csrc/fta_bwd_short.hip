// Backward for short rows: all four gradients in one kernel.  Up to 128 keys; at D = 32 up to 192, with dropout 256.
//
// The long-row backward is two kernels because a bias gradient needs one workgroup to keep its rectangle of
// (query, key) pairs across the L1 rows while dQ needs every key of a row and dK, dV every query: at 512 keys
// the rectangle alone is the register file of a CU.  At 128 keys it is 64 KB, at 256 half of the register file, so a
// workgroup holds a whole row: wave w owns query block w and keeps the fp32 dBias sums of its 32 queries against all keys in
// registers, the row's Q, K, V and dO sit in LDS, each is read from memory once, and S, dP and the
// exponentials are formed once (the two-kernel form reads the row twice and recomputes all of them).
//
// Scores are computed transposed (S^T = K Q^T: keys on accumulator rows, the query on the lane), which makes dS^T the B
// operand of dQ^T += K^T dS^T as it stands.  dV and dK contract over the queries instead: there a wave owns key block w and
// takes the tile (queries of wave q, keys of block w) from wave q.  The row goes in NT rounds: in round r wave w
// works on keys (w + r) % NT, writes P and dS as 16-bit row-major tiles into its slot of the exchange buffer, and after
// the round's barrier reads those of wave (w - r) % NT with transposing LDS reads.  Two buffers, so one barrier per round
// (one buffer and two barriers beyond 192 keys, where LDS ends).
//
// Everything per score is in fp32 on the vector ALU (scale, bias, row constants unrounded).  The precise mode of fp16
// is an instance that rounds P and dS to nearest on their way into the matrix core instead of toward zero; dropout
// replays the forward's mask.
//
// Up to 128 keys (two waves per SIMD, from two or more workgroups) the bias stays in registers beside the sums, and one
// workgroup's loads run under the other's products.  Bound: memory (eight tensors of 64 bytes per pair and head against some 130
// vector instructions per 32 x 32 tile, about half of the memory time at 128 keys).  B4 H8 L128 D32 fp16: 70 us; the delta,
// dQ/dBias and dK/dV kernels took 14 + 70 + 51.  A wave goes ahead of the other workgroup's on its SIMD while it is in the
// vector part of a round, so that the two do not stand in the same part: B4 H8 L128 training step 104.6 -> 102.8 us, with
// dropout 0.25 123.9 -> 116.8.  (One workgroup per CU, whose waves meet in every round: 3 % slower with it at 256 keys and dropout.)
//
// Beyond 128 keys a CU holds one workgroup of five to eight waves, so that it has to overlap by itself: two sets of row tiles
// in LDS, the next row's coming in during the first four rounds.  The bias has no registers left: a wave packs its
// tiles, converted and in the order of the rounds, where it will write its part of the partial bias gradient at the end, and loads
// a tile of 2 KB per round (from L2, a round ahead).  Bound: the chain of a round (exchange read, S and dP, exponentials,
// exchange write, barrier), 1.8 us (260 us for 24 rows of six rounds) for two tiles per SIMD of which the vector ALU is busy 40 % and the matrix core 15.
// Backward kernels, two (dQ/dBias, dK/dV) -> this, us: B4 H8 L192 fp16 346 -> 260, B1 H4 L192 51 -> 43; training steps B4 H8
// L160 332 -> 227, L192 441 -> 339, B1 H4 L192 with dropout 220 -> 83, B2 H4 L256 with dropout 300 -> 236.  B1 H4 L224
// 85 -> 85 and B2 H4 L256 160 -> 174: without dropout the two kernels take over at 192 keys (their tiles then fill whole slabs
// of 256, and this one's waves have the second barrier).
// Measured and left: the two waves of a SIMD half a round apart (L192 339 -> 404), the own Q and dO in registers (as fast).
#include <type_traits>

#include "fta_kernels.h"
#include "fta_common.h"

namespace fta {

// (a pointer whose address was made by hand is generic, and its loads would wait for LDS, too)
template <class V>
__device__ __forceinline__ V global_load(const void* base, uint32_t byte) {
  return *reinterpret_cast<const __attribute__((address_space(1))) V*>(reinterpret_cast<uintptr_t>(base) + byte);
}

// NT: blocks of 32 queries (and keys) that a row takes, one wave each.
template <class T, int D, int NT, bool DROP, bool NEAREST>
__global__ void __launch_bounds__(64 * NT) __attribute__((amdgpu_waves_per_eu(D == 32 ? 2 : 1))) fta_bwd_short_kernel(const BwdParams p) {
  constexpr int KS = D / 16, DT = D / 32;
  constexpr bool LATE = NT > 6;          // (no registers: operands are read later)
  constexpr int ROWS = 32 * NT;
  constexpr int TILE = ROWS * D;         // elements of a staged tensor row
  constexpr int XT = 32 * 32;            // elements of an exchanged tile
  constexpr bool AHEAD = NT > 4;         // (D = 32) one workgroup per CU: the next row's tiles come in under this row's products
  constexpr bool STREAM = NT > 4;        // the bias is read again in every row
  constexpr int XB = NT > 6 ? 1 : 2;     // exchange buffers
  extern __shared__ __attribute__((aligned(16))) char smem_raw[];
  half_t* const stage = reinterpret_cast<half_t*>(smem_raw);  // [buffer][Q, K, V, dO]
  half_t* const xchg = stage + (AHEAD ? 8 : 4) * TILE;         // [buffer][wave][P, dS]

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int hh = lane >> 5, l32 = lane & 31;
  const WorkId id = work_id(1, p.nchunks, p.H, p.head_inner);
  const int chunk = id.chunk, b = id.b, h = id.h, bh = b * p.H + h;
  const int i0 = chunk * p.rows_per_chunk;
  const int nrows = min(p.rows_per_chunk, p.L1 - i0);
  if (nrows <= 0) return;  // whole workgroup leaves together

  const int last = p.L2 - 1;
  const int j = wave * 32 + l32;         // this lane's query, and its key in the dK, dV part
  const bool valid = j <= last;
  const int jc = valid ? j : last;

  FragOffsets<D> fo;
  FragOffsets<32> fx;                    // (the same offsets at D = 32)
  fo.init(lane);
  fx.init(lane);

  // bias (in registers or packed in memory, see above) in the order of the rounds: tile r holds keys of block (wave + r) % NT.  It is
  // loaded behind the first row's copies, which saves a latency at the start (training passes, in front of them / behind: B4 H8 L128 99.1 / 96.9 us,
  // B2 H8 L192 in bf16 154.6 / 150.6).  The values are the forward's,
  // of the kernel that made lse (hand-scheduled at D = 32 without dropout, else the general one): where every key of a
  // query is masked the weights are differences to that very floor.
  constexpr bool FWD1 = (D == 32 && !DROP);
  typedef typename std::conditional<FWD1, F16, T>::type BT;
  uint32_t bias_reg[STREAM ? 1 : NT][8];
  float* part = p.partial + ((int64_t)chunk * p.B * p.H + bh) * p.L2p * p.L2p;
  char* packed = reinterpret_cast<char*>(part + (int64_t)wave * 32 * p.L2p);
  float dbacc[NT][16];
#pragma unroll
  for (int r = 0; r < NT; ++r)
#pragma unroll
    for (int e = 0; e < 16; ++e) dbacc[r][e] = 0.f;

  // copies of one row: TILE / 512 pieces of 1 KB per tensor, dealt to the waves; rows beyond the last are copies of it
  constexpr int NC = TILE / 512 / NT;    // per wave and tensor
  const uint32_t lds0 = lds_addr_of(smem_raw) + (uint32_t)wave * 1024u;
  u32x4 of[KS];
  float lse_n = 0.f;
  // (every per-lane offset is formed here from the lane number, per row: kept over the rows they spill, and a reload
  // waits for all copies in flight)
  auto copies = [&](const half_t* base, const int64_t (&st)[4], int t, int i, int buf) {
    uint32_t ln = (uint32_t)lane, lim = (uint32_t)last;
    asm volatile("" : "+v"(ln), "+s"(lim));
    const void* sb = uniform_ptr(base + b * st[0] + h * st[1] + (int64_t)i * st[2]);
#pragma unroll
    for (int u = 0; u < NC; ++u) {
      const uint32_t row = (uint32_t)((wave + NT * u) * (512 / D)) + ln / (D / 8);
      const uint32_t c = (uint32_t)swz_slot<D>((int)row, (int)(ln % (D / 8)));
      dma16s(min(row, lim) * (uint32_t)(2 * st[3]) + c * 16u, sb, lds0 + (uint32_t)((4 * buf + t) * TILE * 2 + u * NT * 1024));
    }
  };
  auto fetch = [&](int t, int i, int buf) {
    if (t == 0) copies(p.q, p.qs, 0, i, buf);
    if (t == 1) copies(p.k, p.ks, 1, i, buf);
    if (t == 2) copies(p.v, p.vs, 2, i, buf);
    if (t == 3) copies(p.dout, p.dos, 3, i, buf);
  };
  auto fetch_o = [&](int i) {
    uint32_t ln = (uint32_t)lane, lim = (uint32_t)last;
    asm volatile("" : "+v"(ln), "+s"(lim));
    const uint32_t jl = min((uint32_t)wave * 32u + (ln & 31u), lim);
    const void* ob = uniform_ptr(p.o + b * p.os[0] + h * p.os[1] + (int64_t)i * p.os[2]);
    const uint32_t oo = jl * (uint32_t)(2 * p.os[3]) + (ln >> 5) * 16u;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) of[ks] = global_load<u32x4>(ob, oo + 32 * ks);
    lse_n = global_load<float>(uniform_ptr(p.lse + ((int64_t)bh * p.L1 + i) * p.L2), jl * 4u);
  };
  float delta, nl;
  auto row_constants = [&](const half_t* tdo) {
    delta = 0.f;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const u32x4 g = __builtin_bit_cast(u32x4, lds_frag<D>(tdo, wave * 32, fo, ks));
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        delta = __builtin_fmaf(T::lo(of[ks][e]), T::lo(g[e]), delta);
        delta = __builtin_fmaf(T::hi(of[ks][e]), T::hi(g[e]), delta);
      }
    }
    delta = sum_both_halves(delta);
    nl = valid ? -lse_n : -INFINITY;  // (queries beyond the end: weights exactly 0)
  };

  const float scale = p.scale;
  u32x4 bn[2];
  auto fetch_bias = [&](int r) {
    uint32_t ln = (uint32_t)lane;
    asm volatile("" : "+v"(ln) : : "memory");
    const void* sb = uniform_ptr(packed);
    bn[0] = global_load<u32x4>(sb, ln * 16u + r * 2048);
    bn[1] = global_load<u32x4>(sb, ln * 16u + r * 2048 + 1024);
  };
  for (int t = 0; t < 4; ++t) fetch(t, i0, 0);
  {  // (the first row's, by loads that the compiler waits for: they may be kept over the bias)
    const half_t* ob = p.o + b * p.os[0] + h * p.os[1] + (int64_t)i0 * p.os[2] + (int64_t)jc * p.os[3] + 8 * hh;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) of[ks] = *reinterpret_cast<const u32x4*>(ob + 16 * ks);
    lse_n = p.lse[((int64_t)bh * p.L1 + i0) * p.L2 + jc];
  }
  load_bias_tiles<NT, 1, true, true>(p.bias + b * p.bs[0] + h * p.bs[1], p.bs[2], wave * 32, p.L2, BT::kBeyond2,
                                     reinterpret_cast<char*>(xchg + wave * 2 * XT), lane, [=](int c) { return (wave + c) % NT * 32; },
                                     [](uint32_t u) { return FWD1 ? fwd1_bias_pair<T>(u) : T::finite2(u); },
                                     [&](int r, int g, u32x2 v) {
                                       if constexpr (STREAM) {
                                         *reinterpret_cast<u32x2*>(packed + r * 2048 + (g / 2) * 1024 + lane * 16 + (g % 2) * 8) = v;
                                       } else {
                                         bias_reg[r][2 * g] = v[0];
                                         bias_reg[r][2 * g + 1] = v[1];
                                       }
                                     });
  if constexpr (STREAM) {
    wait_vmem_all();
    fetch_bias(0);
  }
  if constexpr (AHEAD) {
    wait_vmem_all();
    __syncthreads();
    row_constants(stage + 3 * TILE);
  }
  for (int ir = 0; ir < nrows; ++ir) {
    const int i = i0 + ir, buf = AHEAD ? ir & 1 : 0;
    const half_t *tq = stage + buf * 4 * TILE, *tk = tq + TILE, *tv = tk + TILE, *tdo = tv + TILE;
    if constexpr (!AHEAD) {
      wait_vmem_all();
      __syncthreads();
      row_constants(tdo);
    }
    floatx16 aq[DT], ak[DT], av[DT];
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int e = 0; e < 16; ++e) { aq[dt][e] = 0.f; ak[dt][e] = 0.f; av[dt][e] = 0.f; }
    int w = wave;
    asm volatile("" : "+s"(w));  // (LDS addresses are formed in each round: kept over the rows they would take 80 registers)
    // dV and dK of the keys that this wave owns, from what wave qb left in round r - 1
    half8_t xp[2], xd[2], xo[2][DT], xq[2][DT];
    auto theirs = [&](int r, int w) {
      int qb = w - (r - 1);
      qb = qb < 0 ? qb + NT : qb;
      const half_t* x = xchg + ((r - 1) % XB * NT + qb) * 2 * XT;
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        xp[u] = lds_frag_t<32>(x, 16 * u, fx, 0);
        xd[u] = lds_frag_t<32>(x + XT, 16 * u, fx, 0);
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) {
          xo[u][dt] = lds_frag_t<D>(tdo, qb * 32 + 16 * u, fo, dt);
          xq[u][dt] = lds_frag_t<D>(tq, qb * 32 + 16 * u, fo, dt);
        }
      }
    };
    auto take = [&]() {
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) {
          av[dt] = T::mfma(xo[u][dt], xp[u], av[dt]);
          ak[dt] = T::mfma(xq[u][dt], xd[u], ak[dt]);
        }
    };
#pragma unroll
    for (int r = 0; r < NT; ++r) {
      asm volatile("" : "+s"(w));
      int kb = w + r;
      kb = kb >= NT ? kb - NT : kb;
      if constexpr (STREAM) {
#pragma unroll
        for (int e = 0; e < 8; ++e) bias_reg[0][e] = bn[e / 4][e % 4];
      }
      half_t* mine = xchg + (r % XB * NT + w) * 2 * XT;
      if constexpr (!AHEAD) __builtin_amdgcn_s_setprio(0);
      if (r > 0) theirs(r, w);
      half8_t fa[KS], fb[KS];
      auto scores = [&]() {
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {  // (Q and dO from LDS in every round: the registers for their fragments are not there)
          fa[ks] = lds_frag<D>(tk, kb * 32, fo, ks);
          fb[ks] = lds_frag<D>(tq, w * 32, fo, ks);
        }
      };
      if constexpr (!LATE) scores();
      __builtin_amdgcn_sched_barrier(0);
      if (r > 0) take();
      if constexpr (LATE) scores();
      floatx16 s, dp;
#pragma unroll
      for (int e = 0; e < 16; ++e) { s[e] = 0.f; dp[e] = 0.f; }
      half8_t ga[KS], gb[KS];
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        ga[ks] = lds_frag<D>(tv, kb * 32, fo, ks);
        gb[ks] = lds_frag<D>(tdo, w * 32, fo, ks);
      }
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) s = T::mfma(fa[ks], fb[ks], s);
      auto dots = [&]() {
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) dp = T::mfma(ga[ks], gb[ks], dp);
      };
      if constexpr (!LATE) dots();
      [[maybe_unused]] uint32_t keep[4];
      if constexpr (DROP) keep_bits4_shared(p.drop, (uint32_t)(bh * p.L1 + i), j, kb * 32 + 4 * hh, keep);
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (!AHEAD) __builtin_amdgcn_s_setprio(1);
      uint32_t t16[8];
#pragma unroll
      for (int e = 0; e < 16; e += 2) {
        uint32_t& bb = bias_reg[STREAM ? 0 : r][e >> 1];
        asm volatile("" : "+v"(bb));  // (converted where it is used: kept in fp32 over the rows it would take twice the registers)
        const float p0 = s[e] = exp2_fast(__builtin_fmaf(__builtin_fmaf(s[e], scale, BT::lo(bb)), kLog2e, nl));
        const float p1 = s[e + 1] = exp2_fast(__builtin_fmaf(__builtin_fmaf(s[e + 1], scale, BT::hi(bb)), kLog2e, nl));
        float w0 = p0, w1 = p1;
        if constexpr (DROP) {
          w0 = keep_byte(p.drop, keep[e >> 2], e & 3) ? p0 * p.drop.scale : 0.f;
          w1 = keep_byte(p.drop, keep[e >> 2], (e & 3) + 1) ? p1 * p.drop.scale : 0.f;
        }
        t16[e >> 1] = NEAREST ? T::pack(w0, w1) : T::pack_fast(w0, w1);
      }
      if constexpr (AHEAD)
        if (r < 4 && ir + 1 < nrows) fetch(r, i + 1, buf ^ 1);
      if constexpr (STREAM) fetch_bias((r + 1) % NT);
      if (AHEAD && r == NT - 1 && NT <= 6) fetch_o(min(i + 1, i0 + nrows - 1));
      // hand P and dS to the wave that owns these keys: row l32 (query), 4 keys at 8 g + 4 hh
      auto hand = [&](half_t* to) {
#pragma unroll
        for (int g = 0; g < 4; ++g) *reinterpret_cast<u32x2*>(to + swz_off<32>(l32, g) + 4 * hh) = u32x2{t16[2 * g], t16[2 * g + 1]};
      };
      if (XB == 1 && r > 0) __syncthreads();  // (everybody has read the last round's)
      hand(mine);
      if constexpr (LATE) dots();
      half8_t ft[2][DT];
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) ft[u][dt] = lds_frag_t<D>(tk, kb * 32 + 16 * u, fo, dt);
#pragma unroll
      for (int e = 0; e < 16; e += 2) {
        float e0 = dp[e], e1 = dp[e + 1];
        if constexpr (DROP) {
          e0 = keep_byte(p.drop, keep[e >> 2], e & 3) ? e0 * p.drop.scale : 0.f;
          e1 = keep_byte(p.drop, keep[e >> 2], (e & 3) + 1) ? e1 * p.drop.scale : 0.f;
        }
        const float d0 = s[e] * (e0 - delta), d1 = s[e + 1] * (e1 - delta);
        dbacc[r][e] += d0;
        dbacc[r][e + 1] += d1;
        asm volatile("" : "+v"(dbacc[r][e]), "+v"(dbacc[r][e + 1]));  // (here: else the sums are made at the row's end, from addends kept until then)
        t16[e >> 1] = NEAREST ? T::pack(d0, d1) : T::pack_fast(d0, d1);
      }
      hand(mine + XT);
      if (AHEAD && r == NT - 1 && NT > 6) fetch_o(min(i + 1, i0 + nrows - 1));
      // dQ^T += K^T dS^T
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const half8_t db = as_half8(u32x4{t16[4 * u], t16[4 * u + 1], t16[4 * u + 2], t16[4 * u + 3]});
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) aq[dt] = T::mfma(ft[u][dt], db, aq[dt]);
      }
      __syncthreads();
    }
    theirs(NT, w);
    take();
    if constexpr (AHEAD) wait_vmem_all();
    __syncthreads();                      // the row's tiles have been read by everybody (AHEAD: and the next row's are there)
    if constexpr (AHEAD) {
      row_constants(stage + ((buf ^ 1) * 4 + 3) * TILE);
    } else if (ir + 1 < nrows) {
      for (int t = 0; t < 4; ++t) fetch(t, i + 1, 0);
      fetch_o(i + 1);
    }
    // rows of dQ, dK, dV: one exchange between the lane halves per register pair gives each lane eight consecutive d
    uint32_t ln = (uint32_t)lane;
    asm volatile("" : "+v"(ln));
    const uint32_t jl = (uint32_t)wave * 32u + (ln & 31u);
    auto put = [&](half_t* base, const int64_t (&st)[4], const floatx16 (&acc)[DT], float f) {
      const void* row = uniform_ptr(base + b * st[0] + h * st[1] + (int64_t)i * st[2]);
      const uint32_t off = jl * (uint32_t)(2 * st[3]) + (ln >> 5) * 16u;
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          const floatx16& a = acc[dt];
          const uint32_t x0 = T::pack(a[8 * u] * f, a[8 * u + 1] * f), x1 = T::pack(a[8 * u + 2] * f, a[8 * u + 3] * f);
          const uint32_t y0 = T::pack(a[8 * u + 4] * f, a[8 * u + 5] * f), y1 = T::pack(a[8 * u + 6] * f, a[8 * u + 7] * f);
          auto r0 = __builtin_amdgcn_permlane32_swap(x0, y0, false, false);
          auto r1 = __builtin_amdgcn_permlane32_swap(x1, y1, false, false);
          const u32x4 piece = {(uint32_t)r0[0], (uint32_t)r1[0], (uint32_t)r0[1], (uint32_t)r1[1]};
          if (jl <= (uint32_t)last) {
            // (the store reads its data for two more issue slots)
            asm volatile("global_store_dwordx4 %0, %1, %2 offset:%3\n\ts_nop 1" ::"v"(off), "v"(piece), "s"(row), "n"(64 * dt + 32 * u) : "memory");
          }
        }
    };
    put(p.dq, p.dqs, aq, scale);
    put(p.dk, p.dks, ak, scale);
    put(p.dv, p.dvs, av, 1.0f);
  }
  // partial dBias of this chunk
  part += (int64_t)j * p.L2p;
#pragma unroll
  for (int r = 0; r < NT; ++r) {
    int kb = wave + r;
    kb = kb >= NT ? kb - NT : kb;
#pragma unroll
    for (int g = 0; g < 4; ++g)
      *reinterpret_cast<float4*>(part + kb * 32 + 8 * g + 4 * hh) =
          make_float4(dbacc[r][4 * g], dbacc[r][4 * g + 1], dbacc[r][4 * g + 2], dbacc[r][4 * g + 3]);
  }
}

// ---- host side -----------------------------------------------------------------------------------------
bool plan_short(int B, int H, int L1, int L2, int D, int feat, ShortPlan& pl) {
  if (L2 > (D == 64 ? 128 : feat == 2 ? 256 : 192)) return false;
  pl = ShortPlan{};
  pl.NT = (L2 + 31) / 32;
  pl.threads = 64 * pl.NT;
  pl.smem = (size_t)(pl.NT > 4 ? 8 : 4) * 32 * pl.NT * D * 2 + (size_t)(pl.NT > 6 ? 1 : 2) * pl.NT * 2 * 32 * 32 * 2;
  // D = 32: two waves per SIMD; D = 64 (more registers): one
  const long slots = (pl.NT > 4 ? 1 : (D == 32 ? 8 : 4) / pl.NT) * 256;
  const int nch = balanced_chunks((long)B * H, L1, slots, 2);
  pl.rows_per_chunk = (L1 + nch - 1) / nch;
  pl.nchunks = (L1 + pl.rows_per_chunk - 1) / pl.rows_per_chunk;
  return true;
}

hipError_t launch_short(BwdParams p, const ShortPlan& pl, int D, int dtype, bool precise, hipStream_t st) {
  p.nchunks = pl.nchunks;
  p.rows_per_chunk = pl.rows_per_chunk;
  const dim3 grid((unsigned)(p.B * p.H * pl.nchunks)), block((unsigned)pl.threads);
  const bool drop = p.drop.thresh != 0;
#define FTA_SHORT_DROP(DD, NN)                                                                                             \
  if (D == DD && pl.NT == NN && drop)                                                                                      \
    return dtype == kBF16 ? launch_kernel(fta_bwd_short_kernel<BF16, DD, NN, true, true>, p, grid, block, pl.smem, st)     \
                          : launch_kernel(fta_bwd_short_kernel<F16, DD, NN, true, true>, p, grid, block, pl.smem, st);
#define FTA_SHORT_CASE(DD, NN)                                                                                             \
  FTA_SHORT_DROP(DD, NN)                                                                                                   \
  if (D == DD && pl.NT == NN) {                                                                                            \
    if (dtype == kBF16) return launch_kernel(fta_bwd_short_kernel<BF16, DD, NN, false, true>, p, grid, block, pl.smem, st); \
    return precise ? launch_kernel(fta_bwd_short_kernel<F16, DD, NN, false, true>, p, grid, block, pl.smem, st)            \
                   : launch_kernel(fta_bwd_short_kernel<F16, DD, NN, false, false>, p, grid, block, pl.smem, st);          \
  }
  FTA_SHORT_CASE(32, 1) FTA_SHORT_CASE(32, 2) FTA_SHORT_CASE(32, 3) FTA_SHORT_CASE(32, 4) FTA_SHORT_CASE(32, 5) FTA_SHORT_CASE(32, 6)
  FTA_SHORT_DROP(32, 7) FTA_SHORT_DROP(32, 8)
  FTA_SHORT_CASE(64, 1) FTA_SHORT_CASE(64, 2) FTA_SHORT_CASE(64, 3) FTA_SHORT_CASE(64, 4)
#undef FTA_SHORT_CASE
#undef FTA_SHORT_DROP
  return hipErrorInvalidConfiguration;
}

}  // namespace fta
