// Backward for short rows (up to 128 keys): all four gradients in one kernel.
//
// The long-row backward is two kernels because a bias gradient needs one workgroup to keep its rectangle of
// (query, key) pairs across the L1 rows while dQ needs every key of a row and dK, dV every query: at 512 keys
// the rectangle alone is the register file of a CU.  At 128 keys it is 64 KB, so a workgroup holds a whole row:
// wave w owns query block w and keeps the bias and the fp32 dBias sums of its 32 queries against all keys in
// registers, the row's Q, K, V and dO sit in LDS, each is read from memory once, and S, dP and the
// exponentials are formed once (the two-kernel form reads the row twice and recomputes all of them).
//
// Scores are computed transposed (S^T = K Q^T: keys on accumulator rows, the query on the lane), which makes dS^T the B
// operand of dQ^T += K^T dS^T as it stands.  dV and dK contract over the queries instead: there a wave owns key block w and
// takes the tile (queries of wave q, keys of block w) from wave q.  The row goes in NT rounds: in round r wave w
// works on keys (w + r) % NT, writes P and dS as 16-bit row-major tiles into its slot of the exchange buffer, and after
// the round's barrier reads those of wave (w - r) % NT with transposing LDS reads.  Two buffers, so one barrier per round.
//
// Everything per score is in fp32 on the vector ALU (scale, bias, row constants unrounded).  The precise mode of fp16
// is an instance that rounds P and dS to nearest on their way into the matrix core instead of toward zero; dropout
// replays the forward's mask.
//
// Bound: memory (eight tensors of 64 bytes per pair and head against some 130 vector instructions per 32 x 32 tile,
// about half of the memory time at 128 keys).  Two workgroups of four waves share a CU, one's loads under the other's
// products.  The bias gradient's sums are made where their addends are (an empty asm statement holds them there): moved to
// the end of the row, as the compiler would have it, they keep every addend of the row in registers, and at 128 keys in
// scratch.  B4 H8 L128 D32 fp16: 70 us (87 with the sums at the row's end); the delta, dQ/dBias and dK/dV kernels took
// 14 + 70 + 51.
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
  constexpr int ROWS = 32 * NT;
  constexpr int TILE = ROWS * D;         // elements of a staged tensor row
  constexpr int XT = 32 * 32;            // elements of an exchanged tile
  extern __shared__ __attribute__((aligned(16))) char smem_raw[];
  half_t* tq = reinterpret_cast<half_t*>(smem_raw);
  half_t *tk = tq + TILE, *tv = tk + TILE, *tdo = tv + TILE;
  half_t* xchg = tdo + TILE;             // [buffer][wave][P, dS]

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

  // stationary bias, in the order of the rounds: tile r holds keys of block (wave + r) % NT.  The values are the forward's,
  // of the kernel that made lse (hand-scheduled at D = 32 without dropout, else the general one): where every key of a
  // query is masked the weights are differences to that very floor.
  constexpr bool FWD1 = (D == 32 && !DROP);
  typedef typename std::conditional<FWD1, F16, T>::type BT;
  uint32_t bias_reg[NT][8];
  float dbacc[NT][16];
  load_bias_tiles<NT, 1, true, true>(p.bias + b * p.bs[0] + h * p.bs[1], p.bs[2], wave * 32, p.L2, BT::kBeyond2,
                                     reinterpret_cast<char*>(xchg + wave * 2 * XT), lane, [=](int c) { return (wave + c) % NT * 32; },
                                     [](uint32_t u) { return FWD1 ? fwd1_bias_pair<T>(u) : T::finite2(u); },
                                     [&](int r, int g, u32x2 v) {
                                       bias_reg[r][2 * g] = v[0];
                                       bias_reg[r][2 * g + 1] = v[1];
                                     });
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
  auto fetch = [&](int i) {
    uint32_t ln = (uint32_t)lane, lim = (uint32_t)last;
    asm volatile("" : "+v"(ln), "+s"(lim));
    auto copies = [&](const half_t* base, const int64_t (&st)[4], int t) {
      const void* sb = uniform_ptr(base + b * st[0] + h * st[1] + (int64_t)i * st[2]);
#pragma unroll
      for (int u = 0; u < NC; ++u) {
        const uint32_t row = (uint32_t)((wave + NT * u) * (512 / D)) + ln / (D / 8);
        const uint32_t c = (uint32_t)swz_slot<D>((int)row, (int)(ln % (D / 8)));
        dma16s(min(row, lim) * (uint32_t)(2 * st[3]) + c * 16u, sb, lds0 + (uint32_t)(t * TILE * 2 + u * NT * 1024));
      }
    };
    copies(p.q, p.qs, 0);
    copies(p.k, p.ks, 1);
    copies(p.v, p.vs, 2);
    copies(p.dout, p.dos, 3);
    const uint32_t jl = min((uint32_t)wave * 32u + (ln & 31u), lim);
    const void* ob = uniform_ptr(p.o + b * p.os[0] + h * p.os[1] + (int64_t)i * p.os[2]);
    const uint32_t oo = jl * (uint32_t)(2 * p.os[3]) + (ln >> 5) * 16u;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) of[ks] = global_load<u32x4>(ob, oo + 32 * ks);
    lse_n = global_load<float>(uniform_ptr(p.lse + ((int64_t)bh * p.L1 + i) * p.L2), jl * 4u);
  };

  const float scale = p.scale;
  fetch(i0);
  for (int ir = 0; ir < nrows; ++ir) {
    const int i = i0 + ir;
    wait_vmem_all();
    __syncthreads();
    float delta = 0.f;
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
    const float nl = valid ? -lse_n : -INFINITY;  // (queries beyond the end: weights exactly 0)
    floatx16 aq[DT], ak[DT], av[DT];
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int e = 0; e < 16; ++e) { aq[dt][e] = 0.f; ak[dt][e] = 0.f; av[dt][e] = 0.f; }
    int w = wave;
    asm volatile("" : "+s"(w));  // (LDS addresses are formed in each round: kept over the rows they would take 80 registers)
#pragma unroll
    for (int r = 0; r < NT; ++r) {
      asm volatile("" : "+s"(w));
      int kb = w + r;
      kb = kb >= NT ? kb - NT : kb;
      int qb = w - r;
      qb = qb < 0 ? qb + NT : qb;
      floatx16 s, dp;
#pragma unroll
      for (int e = 0; e < 16; ++e) { s[e] = 0.f; dp[e] = 0.f; }
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {  // (Q and dO from LDS in every round: the registers for their fragments are not there)
        s = T::mfma(lds_frag<D>(tk, kb * 32, fo, ks), lds_frag<D>(tq, w * 32, fo, ks), s);
        dp = T::mfma(lds_frag<D>(tv, kb * 32, fo, ks), lds_frag<D>(tdo, w * 32, fo, ks), dp);
      }
      [[maybe_unused]] uint32_t keep[4];
      if constexpr (DROP) keep_bits4_shared(p.drop, (uint32_t)(bh * p.L1 + i), j, kb * 32 + 4 * hh, keep);
      uint32_t pp[8], ds[8];
#pragma unroll
      for (int e = 0; e < 16; e += 2) {
        uint32_t& bb = bias_reg[r][e >> 1];
        asm volatile("" : "+v"(bb));  // (converted where it is used: kept in fp32 over the rows it would take twice the registers)
        float p0 = exp2_fast(__builtin_fmaf(__builtin_fmaf(s[e], scale, BT::lo(bb)), kLog2e, nl));
        float p1 = exp2_fast(__builtin_fmaf(__builtin_fmaf(s[e + 1], scale, BT::hi(bb)), kLog2e, nl));
        float e0 = dp[e], e1 = dp[e + 1], w0 = p0, w1 = p1;
        if constexpr (DROP) {
          const bool k0 = keep_byte(p.drop, keep[e >> 2], e & 3), k1 = keep_byte(p.drop, keep[e >> 2], (e & 3) + 1);
          w0 = k0 ? p0 * p.drop.scale : 0.f;
          w1 = k1 ? p1 * p.drop.scale : 0.f;
          e0 = k0 ? e0 * p.drop.scale : 0.f;
          e1 = k1 ? e1 * p.drop.scale : 0.f;
        }
        const float d0 = p0 * (e0 - delta), d1 = p1 * (e1 - delta);
        dbacc[r][e] += d0;
        dbacc[r][e + 1] += d1;
        if constexpr (D == 32) asm volatile("" : "+v"(dbacc[r][e]), "+v"(dbacc[r][e + 1]));  // (D = 64 has the registers)
        pp[e >> 1] = NEAREST ? T::pack(w0, w1) : T::pack_fast(w0, w1);
        ds[e >> 1] = NEAREST ? T::pack(d0, d1) : T::pack_fast(d0, d1);
      }
      // dQ^T += K^T dS^T
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const half8_t db = as_half8(u32x4{ds[4 * u], ds[4 * u + 1], ds[4 * u + 2], ds[4 * u + 3]});
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) aq[dt] = T::mfma(lds_frag_t<D>(tk, kb * 32 + 16 * u, fo, dt), db, aq[dt]);
      }
      // hand P and dS to the wave that owns these keys: row l32 (query), 4 keys at 8 g + 4 hh
      half_t* mine = xchg + ((r & 1) * NT + w) * 2 * XT;
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int off = swz_off<32>(l32, g) + 4 * hh;
        *reinterpret_cast<u32x2*>(mine + off) = u32x2{pp[2 * g], pp[2 * g + 1]};
        *reinterpret_cast<u32x2*>(mine + XT + off) = u32x2{ds[2 * g], ds[2 * g + 1]};
      }
      __syncthreads();
      const half_t* theirs = xchg + ((r & 1) * NT + qb) * 2 * XT;
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const half8_t fp = lds_frag_t<32>(theirs, 16 * u, fx, 0), fd = lds_frag_t<32>(theirs + XT, 16 * u, fx, 0);
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) {
          av[dt] = T::mfma(lds_frag_t<D>(tdo, qb * 32 + 16 * u, fo, dt), fp, av[dt]);
          ak[dt] = T::mfma(lds_frag_t<D>(tq, qb * 32 + 16 * u, fo, dt), fd, ak[dt]);
        }
      }
    }
    __syncthreads();                      // the row's tiles have been read by everybody
    if (ir + 1 < nrows) fetch(i + 1);
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
  float* part = p.partial + (((int64_t)chunk * p.B * p.H + bh) * p.L2p + j) * p.L2p;
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
bool plan_short(int B, int H, int L1, int L2, int D, ShortPlan& pl) {
  if (L2 > 128) return false;
  pl = ShortPlan{};
  pl.NT = (L2 + 31) / 32;
  pl.threads = 64 * pl.NT;
  pl.smem = (size_t)4 * 32 * pl.NT * D * 2 + (size_t)2 * pl.NT * 2 * 32 * 32 * 2;
  // D = 32: two waves per SIMD; D = 64 (more registers): one
  const long slots = (D == 32 ? 8 : 4) / pl.NT * 256;
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
#define FTA_SHORT_CASE(DD, NN)                                                                                             \
  if (D == DD && pl.NT == NN) {                                                                                            \
    if (dtype == kBF16)                                                                                                    \
      return drop ? launch_kernel(fta_bwd_short_kernel<BF16, DD, NN, true, true>, p, grid, block, pl.smem, st)             \
                  : launch_kernel(fta_bwd_short_kernel<BF16, DD, NN, false, true>, p, grid, block, pl.smem, st);           \
    if (drop) return launch_kernel(fta_bwd_short_kernel<F16, DD, NN, true, true>, p, grid, block, pl.smem, st);            \
    return precise ? launch_kernel(fta_bwd_short_kernel<F16, DD, NN, false, true>, p, grid, block, pl.smem, st)            \
                   : launch_kernel(fta_bwd_short_kernel<F16, DD, NN, false, false>, p, grid, block, pl.smem, st);          \
  }
  FTA_SHORT_CASE(32, 1) FTA_SHORT_CASE(32, 2) FTA_SHORT_CASE(32, 3) FTA_SHORT_CASE(32, 4)
  FTA_SHORT_CASE(64, 1) FTA_SHORT_CASE(64, 2) FTA_SHORT_CASE(64, 3) FTA_SHORT_CASE(64, 4)
#undef FTA_SHORT_CASE
  return hipErrorInvalidConfiguration;
}

}  // namespace fta
