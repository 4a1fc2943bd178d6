// The AlphaFold2 triangle-attention block around the attention kernels, forward and backward:
//
//   forward    blk_proj_kernel   layer norm, q/k/v/bias/gate projections of a pair row, sigmoid of the gate
//              (attention)
//              blk_out_kernel    gate * o, output projection
//   backward   blk_dout_kernel   gradient through the output projection and the gate: dO and d(gate logits)
//              (attention backward)
//              blk_dx_kernel     sum of the five projections' input gradients, layer norm backward: dz
//              blk_wgrad_kernel  all weight gradients, as partial sums over chunks of pair rows
//              blk_reduce_kernel, blk_norm_grad_kernel  the partials summed in a fixed order
//
// What bounds them: memory.  A pair row is 128 channels in and 4 x 128 out, 2*128*516 operations against
// 1.3 KB in bf16: 100 flop per byte where the chip balances at 250.  So each tensor is read once per kernel
// (z by the sections of wgrad: once from memory, then from the die's L2) and everything that can be formed from a row in registers is: the normalised row never goes to memory (it
// is formed again where the backward needs it), nor do gate * o or the five input gradients before they
// are summed.  The kernels out and dout let a wave own 32 pair rows: lane l holds row l % 32 as
// the B operands of its MFMAs (8 channels per 16-wide contraction step and lane half), an accumulator tile (32
// output channels x 32 rows) is written as two 16-byte pieces per lane, and the weights are the A operands, all of
// them in LDS in operand order, read with one conflict-free ds_read_b128 per contraction step, no barrier after they
// are loaded.  proj and dx have four to five times the weights: there the waves of a workgroup keep them in registers,
// one or two tiles of output channels each, and share the rows through LDS (see "staged row tiles" below).
//
// fp32 blocks: the fp32 matrix instructions run at a sixteenth of the bf16 ones' rate and bounded every kernel (training pass
// at 192 x 192 pairs: 283 us in these kernels).  So an fp32 operand is taken apart into three bf16 ones, x = x1 + x2 + x3, which
// hold its 24 bits, and a product of two is six bf16 products summed in fp32 (x1 y1, x1 y2, x2 y1, x1 y3, x2 y2, x3 y1; what is
// left out is below 2^-24 of the product).  Activations are taken apart where they enter LDS, weights on their way into
// registers or LDS.  Against 64 bits (relative L2, 192 x 192 pairs, fp32 instructions / three parts): gate 8.0e-8 / 7.1e-8, out
// 1.6e-7 / 1.3e-7, dz 2.9e-7 / 2.3e-7, weight gradients 4.0e-7 / 1.8e-7 (wo) to 3.6e-7 (wb): the matrix core sums 16 products
// at once, the fp32 instruction two.  Infinity, and values that round to it in
// bf16 (beyond 3.39e38), have no three parts: a tile whose sums are not all finite is formed again by the fp32 instruction,
// so that infinities come out as they went in.  Nothing is rounded to 16 bits in memory that was not before (q, k, v, bias, o and their gradients).
// us per kernel at 192 x 192 pairs, before and after: proj 69 / 47, out 32 / 26, dout 29 / 28, dx 57 / 48, wgrad 82 / 50; a
// training pass 352 / 265 (256 x 256: 498 / 394, 321 x 321: 838 / 670), inference 112 / 82 (457 x 457: 505 / 387).  A workgroup there has few
// rows, so that what it waits for before the first of them counts: with every load that the first row needs asked for at once, row blocks dealt to the
// workgroups in turn and dx's operands read a step ahead proj 41, out 19, dout 21, dx 40, wgrad 46; a training pass 246 (beside 272; 150 x 150: 181
// beside 200, 256 x 256: 383 beside 413, 321 x 321: 645 beside 690), inference 73 beside 84 (457 x 457: 374 beside 384).
//
// Measured, AlphaFold2's block (C 128, 4 heads of 32) at 384 x 384 pairs in bf16: a training pass 3.64 ms as separate
// library calls around the attention, 0.47 with these; us per kernel (rocprofv3, median of 40 launches): proj 49, out
// 26, dout 37, dx 46, wgrad 62, reduce 10, norm_grad 5.
#include "fta_block.h"

#include <type_traits>

#include "fta.h"

#include "fta_common.h"
#include "fta_kernels.h"
#include "fta_pipe.h"

namespace fta {
namespace {

// ---- operand fragments: 8 consecutive contraction elements per lane -----------------------------------
template <bool F32> struct Frag;
template <> struct Frag<false> { u32x4 w; };
template <> struct Frag<true> { float v[8]; };
template <bool F32> struct Store { typedef uint16_t type; };
template <> struct Store<true> { typedef float type; };

// The same as matrix core operands: the 16-bit values as they are, fp32 ones as three planes of bf16, largest first.
template <bool F32> struct Op { u32x4 p[F32 ? 3 : 1]; };
template <bool HERE = false>
__device__ __forceinline__ Op<false> to_op(const Frag<false>& f) { return Op<false>{{f.w}}; }
// (HERE: in place, every time.  Weights are the same in every pass of a loop, and their planes, taken out of it, do not fit
// the registers.)
template <bool HERE = false>
__device__ __forceinline__ Op<true> to_op(const Frag<true>& f) {
  Op<true> o;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    float a = f.v[2 * e], b = f.v[2 * e + 1];
#pragma unroll
    for (int n = 0; n < 3; ++n) {  // (the differences are exact)
      uint32_t w;
      if constexpr (HERE) {
        // (two idle slots behind the last of them, in front of an MFMA that the compiler may put there)
        if (n == 0 && e < 3) asm volatile("v_cvt_pk_bf16_f32 %0, %1, %2" : "=v"(w) : "v"(a), "v"(b));
        else if (n == 0) asm volatile("v_cvt_pk_bf16_f32 %0, %1, %2\n\ts_nop 1" : "=v"(w) : "v"(a), "v"(b));
        else w = BF16::pack(a, b);
      } else {
        w = BF16::pack(a, b);
      }
      // (the compiler would convert each half once more by itself, to subtract it)
      if (n < 2) asm("" : "+v"(w));
      o.p[n][e] = w;
      a -= BF16::lo(w);
      b -= BF16::hi(w);
    }
  }
  return o;
}
template <class A, int PA = 3, bool LONG = false, int PB = 3>
__device__ __forceinline__ floatx16 mma(const Op<false>& a, const Op<false>& b, floatx16 c) {
  return A::mfma(as_half8(a.p[0]), as_half8(b.p[0]), c);
}
// (PA, PB: planes of `a` and `b` that are not zero: two hold the 11 bits of an fp16 value.  LONG: a sum over many steps; the small
// products are summed by themselves first, so that the long sum is rounded twice a step and not six times)
template <class A, int PA = 3, bool LONG = false, int PB = 3>
__device__ __forceinline__ floatx16 mma(const Op<true>& a, const Op<true>& b, floatx16 c) {
  constexpr int at[6][2] = {{2, 0}, {0, 2}, {1, 1}, {0, 1}, {1, 0}, {0, 0}};
  floatx16 t = c;
  if constexpr (LONG)
#pragma unroll
    for (int r = 0; r < 16; ++r) t[r] = 0.f;
#pragma unroll
  for (int n = 0; n < (LONG ? 5 : 6); ++n)
    if (at[n][0] < PA && at[n][1] < PB) t = BF16::mfma(as_half8(a.p[at[n][0]]), as_half8(b.p[at[n][1]]), t);
  if constexpr (LONG) {
    c = BF16::mfma(as_half8(a.p[0]), as_half8(b.p[0]), c);
#pragma unroll
    for (int r = 0; r < 16; ++r) t[r] += c[r];
  }
  return t;
}

// A tile of sums that are not all finite (for the whole wave): three parts of an infinite operand, or of a finite one that
// rounds to infinity in bf16, sum to NaN whatever the product is.  The waves keep a flag, and one that has seen such a tile
// forms all of its tiles again behind its loop, from the operands in memory, where the registers of the loop are free.
__device__ __forceinline__ bool not_finite(const floatx16& c) {
  float s = 0.f;
#pragma unroll
  for (int r = 0; r < 16; ++r) s = __builtin_fmaf(c[r], 0.f, s);
  return __builtin_amdgcn_ballot_w64(s != 0.f) != 0;
}
// One contraction step by the fp32 matrix instruction: element e of the two lane halves is one pair.
__device__ __forceinline__ floatx16 mma_f32(const float (&a)[8], const float (&b)[8], floatx16 c) {
#pragma unroll
  for (int e = 0; e < 8; ++e) c = __builtin_amdgcn_mfma_f32_32x32x2f32(a[e], b[e], c, 0, 0, 0);
  return c;
}

template <class A>
__device__ __forceinline__ void unpack(const Frag<false>& f, float (&x)[8]) {
#pragma unroll
  for (int e = 0; e < 4; ++e) { x[2 * e] = A::lo(f.w[e]); x[2 * e + 1] = A::hi(f.w[e]); }
}
template <class A>
__device__ __forceinline__ void unpack(const Frag<true>& f, float (&x)[8]) {
#pragma unroll
  for (int e = 0; e < 8; ++e) x[e] = f.v[e];
}
template <class A>
__device__ __forceinline__ void pack(const float (&x)[8], Frag<false>& f) {
#pragma unroll
  for (int e = 0; e < 4; ++e) f.w[e] = A::pack(x[2 * e], x[2 * e + 1]);
}
template <class A>
__device__ __forceinline__ void pack(const float (&x)[8], Frag<true>& f) {
#pragma unroll
  for (int e = 0; e < 8; ++e) f.v[e] = x[e];
}

// 8 consecutive elements of memory (16-byte aligned)
template <bool F32>
__device__ __forceinline__ Frag<F32> load8(const void* base, int64_t elem) {
  Frag<F32> f;
  if constexpr (F32) {
    const float4* s = reinterpret_cast<const float4*>(static_cast<const float*>(base) + elem);
    const float4 a = s[0], b = s[1];
    f.v[0] = a.x; f.v[1] = a.y; f.v[2] = a.z; f.v[3] = a.w;
    f.v[4] = b.x; f.v[5] = b.y; f.v[6] = b.z; f.v[7] = b.w;
  } else {
    f.w = *reinterpret_cast<const u32x4*>(static_cast<const uint16_t*>(base) + elem);
  }
  return f;
}
template <bool F32>
__device__ __forceinline__ void store8(void* base, int64_t elem, const Frag<F32>& f) {
  if constexpr (F32) {
    float4* d = reinterpret_cast<float4*>(static_cast<float*>(base) + elem);
    d[0] = make_float4(f.v[0], f.v[1], f.v[2], f.v[3]);
    d[1] = make_float4(f.v[4], f.v[5], f.v[6], f.v[7]);
  } else {
    *reinterpret_cast<u32x4*>(static_cast<uint16_t*>(base) + elem) = f.w;
  }
}
template <class A, bool F32>
__device__ __forceinline__ float load1(const void* base, int64_t elem) {
  if constexpr (F32) return static_cast<const float*>(base)[elem];
  else return A::lo((uint32_t) static_cast<const uint16_t*>(base)[elem]);
}
template <class A, bool F32>
__device__ __forceinline__ void store1(void* base, int64_t elem, float x) {
  if constexpr (F32) static_cast<float*>(base)[elem] = x;
  else static_cast<uint16_t*>(base)[elem] = (uint16_t)A::pack(x, 0.f);
}

// Fragments in LDS: one 16-byte plane (two for fp32) of 64 lanes per fragment, so that a wave's read is
// one contiguous kilobyte.
template <bool F32> constexpr int kFragBytes = F32 ? 2048 : 1024;
template <bool F32>
__device__ __forceinline__ Frag<F32> frag_read(const char* frags, int idx, int lane) {
  Frag<F32> f;
  const char* s = frags + (size_t)idx * kFragBytes<F32> + lane * 16;
  if constexpr (F32) {
    const float4 a = *reinterpret_cast<const float4*>(s), b = *reinterpret_cast<const float4*>(s + 1024);
    f.v[0] = a.x; f.v[1] = a.y; f.v[2] = a.z; f.v[3] = a.w;
    f.v[4] = b.x; f.v[5] = b.y; f.v[6] = b.z; f.v[7] = b.w;
  } else {
    f.w = *reinterpret_cast<const u32x4*>(s);
  }
  return f;
}
template <bool F32>
__device__ __forceinline__ void frag_write(char* frags, int idx, int lane, const Frag<F32>& f) {
  char* d = frags + (size_t)idx * kFragBytes<F32> + lane * 16;
  if constexpr (F32) {
    *reinterpret_cast<float4*>(d) = make_float4(f.v[0], f.v[1], f.v[2], f.v[3]);
    *reinterpret_cast<float4*>(d + 1024) = make_float4(f.v[4], f.v[5], f.v[6], f.v[7]);
  } else {
    *reinterpret_cast<u32x4*>(d) = f.w;
  }
}
template <bool F32>
__device__ __forceinline__ Frag<F32> frag_zero() {
  Frag<F32> f;
  if constexpr (F32) {
#pragma unroll
    for (int e = 0; e < 8; ++e) f.v[e] = 0.f;
  } else {
    f.w = u32x4{0, 0, 0, 0};
  }
  return f;
}

// Operands in LDS: a 16-byte plane of 64 lanes each, three for fp32.
template <bool F32> constexpr int kOpBytes = F32 ? 3072 : 1024;
// (PL: the fp32 planes that are not zero)
template <bool F32, int PL = 3>
__device__ __forceinline__ Op<F32> op_read(const char* ops, int idx, int lane) {
  Op<F32> o;
  const char* s = ops + (size_t)idx * kOpBytes<F32> + lane * 16;
#pragma unroll
  for (int n = 0; n < (F32 ? PL : 1); ++n) o.p[n] = *reinterpret_cast<const u32x4*>(s + n * 1024);
  return o;
}
template <bool F32, int PL = 3>
__device__ __forceinline__ void op_write(char* ops, int idx, int lane, const Op<F32>& o) {
  char* d = ops + (size_t)idx * kOpBytes<F32> + lane * 16;
#pragma unroll
  for (int n = 0; n < (F32 ? PL : 1); ++n) *reinterpret_cast<u32x4*>(d + n * 1024) = o.p[n];
}

// An accumulator tile (lane: column l % 32; register r: row 8*(r/4) + 4*hh + r%4) as two runs of eight
// consecutive rows per lane: out[u][e] is row 16*u + 8*hh + e.
__device__ __forceinline__ void rows8(const floatx16& acc, float (&out)[2][8]) {
#pragma unroll
  for (int u = 0; u < 2; ++u)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float a = acc[8 * u + r], b = acc[8 * u + 4 + r];
      auto s = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(uint32_t, a), __builtin_bit_cast(uint32_t, b), false, false);
      out[u][r] = __builtin_bit_cast(float, (uint32_t)s[0]);
      out[u][4 + r] = __builtin_bit_cast(float, (uint32_t)s[1]);
    }
}

// The two runs of a lane's row on their way to memory or back.  An access of run u by all lanes takes 32 bytes out of every row, a half
// or a quarter of the lines it touches.  So the lanes of rows r and r + 16 exchange (the second half of theirs for the first of the other's):
// a lane then has one part of both rows, and an access takes 64 consecutive bytes of each of 16 rows.  at0, at1: the elements
// of rows r % 16 and 16 + r % 16 where the lane half's runs begin (row_pair).
__device__ __forceinline__ void swap16(uint32_t& a, uint32_t& b) {
  auto s = __builtin_amdgcn_permlane16_swap(a, b, false, false);
  a = s[0];
  b = s[1];
}
__device__ __forceinline__ void row_pair(int64_t at, int64_t& at0, int64_t& at1) {
  uint32_t lo0 = (uint32_t)at, lo1 = lo0, hi0 = (uint32_t)((uint64_t)at >> 32), hi1 = hi0;
  swap16(lo0, lo1);
  swap16(hi0, hi1);
  at0 = (int64_t)((uint64_t)hi0 << 32 | lo0);
  at1 = (int64_t)((uint64_t)hi1 << 32 | lo1);
}
template <bool F32>
__device__ __forceinline__ void load_runs(const void* base, int64_t at0, int64_t at1, int lane, Frag<F32>& f0, Frag<F32>& f1) {
  const int odd = (lane >> 4) & 1;
  if constexpr (F32) {
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const uint32_t* d = static_cast<const uint32_t*>(base) + 16 * u + 4 * odd;
      const u32x4 a = *reinterpret_cast<const u32x4*>(d + at0), b = *reinterpret_cast<const u32x4*>(d + at1);
      Frag<F32>& f = u == 0 ? f0 : f1;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        uint32_t x = a[e], y = b[e];
        swap16(x, y);
        f.v[e] = __builtin_bit_cast(float, x);
        f.v[4 + e] = __builtin_bit_cast(float, y);
      }
    }
  } else {
    const uint16_t* d = static_cast<const uint16_t*>(base) + 16 * odd;
    const u32x4 a = *reinterpret_cast<const u32x4*>(d + at0), b = *reinterpret_cast<const u32x4*>(d + at1);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      uint32_t x = a[e], y = b[e];
      swap16(x, y);
      f0.w[e] = x;
      f1.w[e] = y;
    }
  }
}
template <bool F32>
__device__ __forceinline__ void store_runs(void* base, int64_t at0, int64_t at1, int lane, Frag<F32> (&f)[2]) {
  const int odd = (lane >> 4) & 1;
  if constexpr (F32) {
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      uint32_t w[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) w[e] = __builtin_bit_cast(uint32_t, f[u].v[e]);
#pragma unroll
      for (int e = 0; e < 4; ++e) swap16(w[e], w[4 + e]);
      uint32_t* d = static_cast<uint32_t*>(base) + 16 * u + 4 * odd;
      *reinterpret_cast<u32x4*>(d + at0) = u32x4{w[0], w[1], w[2], w[3]};
      *reinterpret_cast<u32x4*>(d + at1) = u32x4{w[4], w[5], w[6], w[7]};
    }
  } else {
    u32x4 a = f[0].w, b = f[1].w;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      uint32_t x = a[e], y = b[e];
      swap16(x, y);
      a[e] = x;
      b[e] = y;
    }
    uint16_t* d = static_cast<uint16_t*>(base) + 16 * odd;
    *reinterpret_cast<u32x4*>(d + at0) = a;
    *reinterpret_cast<u32x4*>(d + at1) = b;
  }
}

__device__ __forceinline__ floatx16 zero16() {
  floatx16 v;
#pragma unroll
  for (int e = 0; e < 16; ++e) v[e] = 0.f;
  return v;
}

template <bool F32>
__device__ __forceinline__ float sigmoid(float x) {
  if constexpr (F32) {
    // (a quarter of 1 + exp(-x), whose reciprocal is not subnormal, and one Newton step; the division takes 4 us more of a training
    // pass of 275 at 192 x 192 pairs)
    const float d = __builtin_fmaf(expf(-x), 0.25f, 0.25f), r = __builtin_amdgcn_rcpf(d);
    return d < INFINITY ? 0.25f * __builtin_fmaf(__builtin_fmaf(-d, r, 1.0f), r, r) : 0.25f * r;
  }
  else return __builtin_amdgcn_rcpf(1.0f + exp2_fast(-kLog2e * x));
}

// q / L for q < 2^24 (L <= 4096): the fp32 quotient is off by one at most.
__device__ __forceinline__ uint32_t div_by_length(uint32_t q, uint32_t L, float inv_l) {
  uint32_t i = (uint32_t)((float)q * inv_l);
  const int r = (int)(q - i * L);
  i -= r < 0 ? 1u : 0u;
  i += r >= (int)L ? 1u : 0u;
  return i;
}

// 32 pair rows of one batch entry: which ones, and where this lane's row is.
struct RowBlock {
  int b;          // batch entry (wave-uniform)
  uint32_t p;     // this lane's row: i * L + j, the last one of the batch entry beyond the end
  uint32_t i, j;
};
__device__ __forceinline__ RowBlock row_block(const BlockParams& p, int blk, int lane) {
  RowBlock r;
  r.b = blk / p.nper;
  r.p = min((uint32_t)(blk - r.b * p.nper) * 32u + (uint32_t)(lane & 31), (uint32_t)p.LL - 1u);
  r.i = div_by_length(r.p, (uint32_t)p.L, 1.0f / (float)p.L);
  r.j = r.p - r.i * (uint32_t)p.L;
  return r;
}
__device__ __forceinline__ int64_t pair_off(const int64_t (&s)[3], const RowBlock& r) { return r.b * s[0] + r.i * s[1] + r.j * s[2]; }
// element of (b, h, i, j, d = 0) in a (B, H, L, L, D) tensor
__device__ __forceinline__ int64_t head_off(const BlockParams& p, const RowBlock& r, int h) {
  return (((int64_t)r.b * p.H + h) * p.LL + r.p) * p.D;
}

// Sum over the 8 or 16 neighbouring lanes that hold a pair row of 64 or 128 channels (DPP moves: quads, then
// mirrored half rows, then mirrored rows).
template <int LANES>
__device__ __forceinline__ float row_sum(float x) {
  auto add = [](float v, auto sel) {
    return v + __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), decltype(sel)::value, 0xF, 0xF, true));
  };
  x = add(x, std::integral_constant<int, 0xB1>{});   // lanes 1 0 3 2
  x = add(x, std::integral_constant<int, 0x4E>{});   // lanes 2 3 0 1
  x = add(x, std::integral_constant<int, 0x141>{});  // half row mirrored
  if constexpr (LANES == 16) x = add(x, std::integral_constant<int, 0x140>{});  // row mirrored
  return x;
}

// 1 / sqrt(x): the instruction's result, good to one unit in the last place, and one Newton step.  x * y is off by 2^-24 of it at most,
// half of which reaches the result, and its rounding adds 2^-24: 1.5 * 2^-24, where a root and a division, 25 instructions,
// round twice (a training pass at 384 x 384 pairs in bf16: 513 us with the instruction alone and with this, 527 with those).
__device__ __forceinline__ float inv_sqrt(float x) {
  const float y = __builtin_amdgcn_rsqf(x);
  const float z = __builtin_fmaf(0.5f * y, __builtin_fmaf(-(x * y), y, 1.0f), y);
  return x < INFINITY ? z : y;
}

// Layer norm without its parameters: v holds 8 of the row's C channels, the neighbouring lanes the others.
// Mean first, then the squared deviations, in fp32.
template <int C>
__device__ __forceinline__ void normalise(float (&v)[8], float eps, float& mean, float& rstd) {
  float s = 0.f;
#pragma unroll
  for (int e = 0; e < 8; ++e) s += v[e];
  mean = row_sum<C / 8>(s) * (1.0f / C);
  s = 0.f;
#pragma unroll
  for (int e = 0; e < 8; ++e) { v[e] -= mean; s = __builtin_fmaf(v[e], v[e], s); }
  rstd = inv_sqrt(row_sum<C / 8>(s) * (1.0f / C) + eps);
#pragma unroll
  for (int e = 0; e < 8; ++e) v[e] *= rstd;
}

// ---- staged row tiles ---------------------------------------------------------------------------------
// The kernels whose weights fill the registers (proj, dx) share the rows between the waves instead: a stage of
// rows is loaded in whole 128-byte lines (a thread takes 8 consecutive elements of a row, neighbouring threads the
// next ones), and sits in LDS as MFMA B operands, one 16-byte slot per (row, 8 elements) and plane.  Slot
// of row r, piece c of a 32-row sub-block: ((c / 2) * 64 + (r ^ (c % 16)) + 32 * (c % 2)): the XOR spreads the
// pieces of a row, which neighbouring threads write at once, over the banks.
template <bool F32, int PL = 3>
__device__ __forceinline__ void piece_write(char* blk, int r, int c, const Frag<F32>& f) {
  op_write<F32, PL>(blk, c / 2, (r ^ (c % 16)) + 32 * (c % 2), to_op(f));
}
template <bool F32, int PL = 3>
__device__ __forceinline__ Op<F32> piece_frag(const char* blk, int ks, int l32, int hh) {
  return op_read<F32, PL>(blk, ks, (l32 ^ ((2 * ks + hh) % 16)) + 32 * hh);
}

// (fp32) A tile of projections by the fp32 instruction: the lane's pair row at element `row` of z, its weight row at
// element `wrow` of w.
template <int C>
__device__ __forceinline__ floatx16 proj_tile_f32(const BlockParams& p, int64_t row, const void* w, int64_t wrow, int hh) {
  float s = 0.f;
#pragma clang loop unroll(disable)
  for (int c = 0; c < C; c += 8) {
    const Frag<true> z = load8<true>(p.z, row + c);
#pragma unroll
    for (int e = 0; e < 8; ++e) s += z.v[e];
  }
  const float mean = s * (1.0f / C);
  s = 0.f;
#pragma clang loop unroll(disable)
  for (int c = 0; c < C; c += 8) {
    const Frag<true> z = load8<true>(p.z, row + c);
#pragma unroll
    for (int e = 0; e < 8; ++e) s = __builtin_fmaf(z.v[e] - mean, z.v[e] - mean, s);
  }
  const float rstd = 1.0f / __builtin_sqrtf(s * (1.0f / C) + p.eps);
  floatx16 acc = zero16();
#pragma clang loop unroll(disable)
  for (int c = 8 * hh; c < C; c += 16) {
    Frag<true> z = load8<true>(p.z, row + c);
    const Frag<true> g = load8<true>(p.gamma, c), b = load8<true>(p.beta, c), a = load8<true>(w, wrow + c);
#pragma unroll
    for (int e = 0; e < 8; ++e) z.v[e] = __builtin_fmaf((z.v[e] - mean) * rstd, g.v[e], b.v[e]);
    acc = mma_f32(a.v, z.v, acc);
  }
  return acc;
}

// ---- forward: layer norm and projections --------------------------------------------------------------
// A wave keeps the weights of one or two tiles of 32 output channels (4*HD/32 tiles of q, k, v, gate over eight
// waves) in registers, 64 of them; the bias heads are one more tile, its weights in LDS, that the waves take
// turns at.  The next stage's loads and its layer norm overlap this stage's products (two stage buffers).
// fp32: a tile's three planes take 96 registers, so that a wave keeps one tile and two workgroups of the same die share the
// output tiles of a row (each reads and normalises it); the bias heads are dot products of the threads that hold the row, in
// the first of the two (a tile more for one of eight waves that meet at every stage's barrier costs half as much
// again): 47 us at 192 x 192 pairs.  With both tiles' weights in fp32 and taken apart at every use, proj took 55, by fp32
// matrix instructions 69.
template <class A, bool F32, int C, int HD>
__global__ void __launch_bounds__(512) blk_proj_kernel(BlockParams p) {
  constexpr int PARTS = F32 ? HD / 64 : 1;           // workgroups that share a row's tiles
  constexpr int KS = C / 16, NT = HD / 64 / PARTS;   // NT: tiles per wave
  constexpr int TR = F32 ? 32 : 64, RS = TR / 32;    // rows per stage (fp32: half, so that few rows still load the CUs evenly)
  constexpr int NP = (TR * C / 8 + 511) / 512;       // pieces per thread
  constexpr int SUB = KS * kOpBytes<F32>, BUF = RS * SUB;
  extern __shared__ char smem[];
  char* wbf = smem + 2 * BUF;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), l32 = lane & 31, hh = lane >> 5;
  float* bgs = reinterpret_cast<float*>(wbf + SUB);
  float* msk = bgs + HD;  // what the mask adds to the bias of a stage's rows, two buffers
  // (the parts of a row are a multiple of the dies apart where the launch fills the chip)
  const int teams = (int)gridDim.x / PARTS, part = (int)blockIdx.x / teams;
  auto tile_of = [=](int t) { return (t * 8 + wave) * PARTS + part; };  // (the gate's tiles, which have the sigmoid besides, spread over waves and parts)
  const int c8 = (tid % (C / 8)) * 8;
  const int LL = (int)p.LL, nst = (LL + TR - 1) / TR, ntot = p.B * nst;
  const float inv_l = 1.0f / (float)p.L;
  Frag<F32> z[NP];
  float mrow;
  const void* mask = p.mask != nullptr ? p.mask : p.gamma;  // (loaded either way, see the stores)
  int zst = 0;  // the stage in z
  auto fetch = [&](int st) {
    const int b = st / nst, p0 = (st - b * nst) * TR;
    zst = st;
    {
      const uint32_t q = (uint32_t)min(p0 + (F32 ? tid / (C / 8) : tid) % TR, LL - 1), i = div_by_length(q, (uint32_t)p.L, inv_l);
      mrow = load1<A, F32>(mask, p.mask != nullptr ? (int64_t)b * p.L + (q - i * (uint32_t)p.L) : 0);
    }
#pragma unroll
    for (int n = 0; n < NP; ++n) {
      const uint32_t q = (uint32_t)min(p0 + (tid + 512 * n) / (C / 8), LL - 1);
      const uint32_t i = div_by_length(q, (uint32_t)p.L, inv_l), j = q - i * (uint32_t)p.L;
      z[n] = load8<F32>(p.z, b * p.zs[0] + (int64_t)i * p.zs[1] + (int64_t)j * p.zs[2] + c8);
    }
  };
  float wbv[F32 ? 4 : 1][8];  // (fp32) the bias heads' weights of this thread's channels (of the last head for heads there are not)
  float gam[8], bet[8];
  auto put = [&](int buffer) {
    char* buf = smem + buffer * BUF;
    // 0 marks padded key positions, which no query may attend to
    const float add = p.mask != nullptr ? (mrow - 1.0f) * 30000.0f : 0.f;
    if (!F32 && tid < TR) msk[buffer * TR + tid] = add;
#pragma unroll
    for (int n = 0; n < NP; ++n) {
      const int row = (tid + 512 * n) / (C / 8);
      float v[8], mean, rstd;
      unpack<A>(z[n], v);
      normalise<C>(v, p.eps, mean, rstd);
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = __builtin_fmaf(v[e], gam[e], bet[e]);
      if constexpr (F32) {
        if (part == 0) {
          const int b = zst / nst, q = min((zst - b * nst) * TR + row, LL - 1), h = c8 / 8;
          float own = 0.f;
#pragma unroll
          for (int g = 0; g < 4; ++g) {
            float s = 0.f;
#pragma unroll
            for (int e = 0; e < 8; ++e) s = __builtin_fmaf(v[e], wbv[g][e], s);
            s = row_sum<C / 8>(s);
            own = h == g ? s : own;
          }
          if (h < p.H && row < TR) store1<A, false>(p.bias, ((int64_t)b * p.H + h) * LL + q, own + add);
        }
      }
      Frag<F32> f;
      pack<A>(v, f);
      if (TR * C / 8 >= 512 || row < TR) piece_write<F32>(buf + (row / 32) * SUB, row % 32, c8 / 8, f);
    }
  };
  // Every load that the first stage waits for is issued here, with no branch and no other load's result in between.
  // (With a pointer per lane, the bias heads' weights under a branch each and the gate's bias behind the weights, four latencies followed
  // each other and a workgroup's first products began after 27k of its 86k cycles at 192 x 192 pairs in fp32.)
  int st = (int)blockIdx.x - part * teams;
  fetch(min(st, ntot - 1));
#pragma unroll
  for (int e = 0; e < 8; ++e) { gam[e] = load1<A, F32>(p.gamma, c8 + e); bet[e] = load1<A, F32>(p.beta, c8 + e); }
  if constexpr (F32) {
#pragma unroll
    for (int h = 0; h < 4; ++h)
#pragma unroll
      for (int e = 0; e < 8; ++e) wbv[h][e] = load1<A, F32>(p.wb, min(h, p.H - 1) * C + c8 + e);
  }
  Frag<F32> wraw[NT][KS];
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    const int n0 = tile_of(t) * 32, sec = n0 / HD;  // (a tile is of one projection)
    const void* ws = p.w[sec];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) wraw[t][ks] = load8<F32>(ws, (int64_t)(n0 - sec * HD + l32) * C + ks * 16 + hh * 8);
  }
  static_assert(KS <= 8 && HD <= 512, "a wave has one step of the bias heads' weights, a thread one entry of the gate's bias");
  [[maybe_unused]] Frag<F32> wbr;
  if constexpr (!F32) wbr = load8<F32>(p.wb, (int64_t)min(l32, p.H - 1) * C + min(wave, KS - 1) * 16 + hh * 8);
  const float bg = load1<A, F32>(p.bg != nullptr ? p.bg : p.gamma, p.bg != nullptr ? min(tid, HD - 1) : 0);
  if (st < ntot) {
    put(0);
    fetch(min(st + teams, ntot - 1));
  }
  Op<F32> w[NT][KS];
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) w[t][ks] = to_op(wraw[t][ks]);
  if constexpr (!F32)
    if (wave < KS) op_write<F32>(wbf, wave, lane, to_op(l32 < p.H ? wbr : frag_zero<F32>()));
  if (tid < HD) bgs[tid] = p.bg != nullptr ? bg : 0.f;
  __syncthreads();
  // the tile of channels n .. n + 31 of pair rows q0 .. q0 + 31
  // (rows beyond the end repeat the last one, and store the same values to the same place: with no branch
  // around the stores the waits for the next stage's loads do not have to wait for them as well)
  auto store_tile = [&](const floatx16& acc, int n, int b, int q0) {
    const int sec = n / HD, col = n - sec * HD, h = col / p.D;
    const int64_t off = ((int64_t)b * p.H + h) * LL * p.D + (col - h * p.D) + hh * 8;
    const int64_t at0 = off + (int64_t)min(q0 + (lane & 15), LL - 1) * p.D, at1 = off + (int64_t)min(q0 + 16 + (lane & 15), LL - 1) * p.D;
    float y[2][8];
    rows8(acc, y);
    if (sec == 3) {
      Frag<F32> f[2];
#pragma unroll
      for (int u = 0; u < 2; ++u) {
#pragma unroll
        for (int e = 0; e < 8; ++e) y[u][e] = sigmoid<F32>(y[u][e] + bgs[col + 16 * u + 8 * hh + e]);
        pack<A>(y[u], f[u]);
      }
      store_runs<F32>(p.gate, at0, at1, lane, f);
    } else {
      Frag<false> f[2];
#pragma unroll
      for (int u = 0; u < 2; ++u) pack<A>(y[u], f[u]);
      store_runs<false>(p.qkv[sec], at0, at1, lane, f);
    }
  };
  [[maybe_unused]] bool bad = false;
  [[maybe_unused]] const int st0 = st;
  auto products = [&](int st, int it) {
    const char* buf = smem + (it & 1) * BUF;
    const int b = st / nst, p0 = (st - b * nst) * TR;
#pragma unroll
    for (int rs = 0; rs < RS; ++rs) {
      floatx16 acc[NT];
#pragma unroll
      for (int t = 0; t < NT; ++t) acc[t] = zero16();
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        const Op<F32> x = piece_frag<F32>(buf + rs * SUB, ks, l32, hh);
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[t] = mma<A>(w[t][ks], x, acc[t]);
      }
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        if constexpr (F32) bad = bad || not_finite(acc[t]);
        store_tile(acc[t], tile_of(t) * 32, b, p0 + rs * 32);
      }
      if (!F32 && wave == ((RS * it + rs) & 7)) {
        floatx16 ab = zero16();
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
          ab = mma<A>(op_read<F32>(wbf, ks, lane), piece_frag<F32>(buf + rs * SUB, ks, l32, hh), ab);
        const float add = msk[(it & 1) * TR + rs * 32 + l32];
        const int q = min(p0 + rs * 32 + l32, LL - 1);
        if (hh == 0)
#pragma unroll
          for (int h = 0; h < 4; ++h)
            if (h < p.H) store1<A, false>(p.bias, ((int64_t)b * p.H + h) * LL + q, ab[h] + add);
      }
    }
  };
  // Half of the waves (one of the two that share a SIMD) prepare the next stage first and multiply then, the others the other
  // way round, so that one wave's products run beside the other's layer norm.
  auto prepare = [&](int st, int it) {
    put((it + 1) & 1);
    fetch(min(st + 2 * teams, ntot - 1));  // (behind the last stage: once more the last rows, which nobody waits for)
  };
  int it = 0;
  for (; st + teams < ntot; st += teams, ++it) {
    if (wave >= 4) prepare(st, it);
    products(st, it);
    if (wave < 4) prepare(st, it);
    __syncthreads();
  }
  if (st < ntot) products(st, it);
  if constexpr (F32)
    if (bad)
#pragma clang loop unroll(disable)
      for (st = st0; st < ntot; st += teams) {
        const int b = st / nst, q0 = (st - b * nst) * TR, q = min(q0 + l32, LL - 1);
        const uint32_t i = div_by_length((uint32_t)q, (uint32_t)p.L, inv_l), j = (uint32_t)q - i * (uint32_t)p.L;
#pragma clang loop unroll(disable)
        for (int t = 0; t < NT; ++t) {
          const int n = tile_of(t) * 32, sec = n / HD;
          store_tile(proj_tile_f32<C>(p, b * p.zs[0] + (int64_t)i * p.zs[1] + (int64_t)j * p.zs[2], p.w[sec], (int64_t)(n - sec * HD + l32) * C, hh), n, b, q0);
        }
      }
}

// ---- forward: gating and output projection ------------------------------------------------------------
// The first item (a column group of a row block) of a wave, in steps of all waves: neighbouring waves take the groups of a row block, then
// comes the next workgroup, so that where the items are no multiple of the waves, the last ones are spread over all CUs.  (Workgroup after
// workgroup, the first 32 of 256 had two items per wave and the others one at 192 x 192 pairs in fp32: out 24.0 / 19.4 us, dout 24.4 / 21.2;
// at 384 x 384 in bf16 27.0 / 25.9 and 39.2 / 36.5.)
__device__ __forceinline__ int first_item(int cg, int nwg, int wave) {
  return __builtin_amdgcn_readfirstlane(((wave / cg) * nwg + (int)blockIdx.x) * cg + wave % cg);
}
template <class A, bool F32, int C, int HD>
__global__ void __launch_bounds__(512) blk_out_kernel(BlockParams p) {
  constexpr int KS = HD / 16, NT = C / 32;
  extern __shared__ char smem[];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), l32 = lane & 31, hh = lane >> 5;
  constexpr int NW = 8, NF = NT * KS / NW;  // waves; weight fragments that a wave brings
  static_assert(NT * KS % NW == 0 && C <= 64 * NW, "shares of the weights");
  float* bos = reinterpret_cast<float*>(smem + (size_t)NT * KS * kOpBytes<F32>);
  // The weights and the first rows are asked for together (a fragment at a time, and the rows behind the barrier, were six latencies in
  // a row: at 192 x 192 pairs a wave has one or two row blocks)
  Frag<F32> wf[NF];
#pragma unroll
  for (int n = 0; n < NF; ++n) {
    const int idx = wave + NW * n;
    wf[n] = load8<F32>(p.wo, (int64_t)((idx / KS) * 32 + l32) * HD + (idx % KS) * 16 + hh * 8);
  }
  float bo = load1<A, F32>(p.bo != nullptr ? p.bo : p.wo, p.bo != nullptr ? min(tid, C - 1) : 0);
  const int nitems = p.B * p.nper * p.cg, step = (int)gridDim.x * NW;
  int item = first_item(p.cg, (int)gridDim.x, wave);
  Frag<F32> gt[KS];
  Frag<false> o[KS];
  RowBlock rb = row_block(p, min(item, nitems - 1) / p.cg, lane);
  auto fetch = [&]() {
#pragma unroll
    for (int ks = 0; ks < KS; ks += 2) {
      const int h = ks * 16 / p.D;
      int64_t at0, at1;
      row_pair(head_off(p, rb, h) + (ks * 16 - h * p.D) + hh * 8, at0, at1);
      load_runs<F32>(p.gate, at0, at1, lane, gt[ks], gt[ks + 1]);
      load_runs<false>(p.o, at0, at1, lane, o[ks], o[ks + 1]);
    }
  };
  fetch();
  asm volatile("" : "+v"(bo));  // (not asked for under the branch below)
#pragma unroll
  for (int n = 0; n < NF; ++n) op_write<F32>(smem, wave + NW * n, lane, to_op(wf[n]));
  if (tid < C) bos[tid] = p.bo != nullptr ? bo : 0.f;
  __syncthreads();
  if (item >= nitems) return;
  auto store_tile = [&](const floatx16& acc, int t, const RowBlock& r) {
    const int64_t oo = pair_off(p.outs, r) + hh * 8;
    float y[2][8];
    rows8(acc, y);
#pragma unroll
    for (int u = 0; u < 2; ++u) {
#pragma unroll
      for (int e = 0; e < 8; ++e) y[u][e] += bos[t * 32 + 16 * u + 8 * hh + e];
      Frag<F32> f;
      pack<A>(y[u], f);
      store8<F32>(p.out, oo + t * 32 + 16 * u, f);  // (rows beyond the end: once more the last one)
    }
  };
  [[maybe_unused]] bool bad = false;
  [[maybe_unused]] const int item0 = item;
  for (; item < nitems; item += step) {
    const RowBlock cur = rb;
    const int g = item % p.cg;
    Op<F32> x[KS];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      float a[8], b[8];
      unpack<A>(gt[ks], a);
      unpack<A>(o[ks], b);
#pragma unroll
      for (int e = 0; e < 8; ++e) a[e] *= b[e];
      Frag<F32> f;
      pack<A>(a, f);
      x[ks] = to_op(f);
    }
    if (item + step < nitems) {
      rb = row_block(p, (item + step) / p.cg, lane);
      fetch();
    }
    for (int t = g; t < NT; t += p.cg) {
      floatx16 acc = zero16();
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) acc = mma<A>(op_read<F32>(smem, t * KS + ks, lane), x[ks], acc);
      if constexpr (F32) bad = bad || not_finite(acc);
      store_tile(acc, t, cur);
    }
  }
  if constexpr (F32)
    if (bad)
#pragma clang loop unroll(disable)
      for (item = item0; item < nitems; item += step) {
        const RowBlock cur = row_block(p, item / p.cg, lane);
#pragma clang loop unroll(disable)
        for (int t = item % p.cg; t < NT; t += p.cg) {
          floatx16 acc = zero16();
#pragma clang loop unroll(disable)
          for (int ks = 0; ks < KS; ++ks) {
            const int h = ks * 16 / p.D;
            const int64_t off = head_off(p, cur, h) + (ks * 16 - h * p.D) + hh * 8;
            Frag<true> v = load8<true>(p.gate, off);
            float b[8];
            unpack<A>(load8<false>(p.o, off), b);
#pragma unroll
            for (int e = 0; e < 8; ++e) v.v[e] *= b[e];
            acc = mma_f32(load8<true>(p.wo, (int64_t)(t * 32 + l32) * HD + ks * 16 + hh * 8).v, v.v, acc);
          }
          store_tile(acc, t, cur);
        }
      }
}

// ---- backward: output projection and gate -------------------------------------------------------------
// d(gate * o) = Wo^T dout; dO = that * gate, d(gate logit) = that * o * gate * (1 - gate).  Workgroups behind
// the first nwg pack the transposed projection weights that blk_dx_kernel reads.
template <class A, bool F32, int C, int HD>
__global__ void __launch_bounds__(512) blk_dout_kernel(BlockParams p) {
  constexpr int KS = C / 16, NT = HD / 32;
  extern __shared__ char smem[];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), l32 = lane & 31, hh = lane >> 5;
  constexpr int NW = 8, NF = NT * KS / NW;  // (as in blk_out_kernel)
  static_assert(NT * KS % NW == 0, "shares of the weights");
  if ((int)blockIdx.x >= p.nwg) {
    constexpr int ksall = 4 * HD / 16 + 1;
    const int npack = (int)gridDim.x - p.nwg;
    for (int idx = ((int)blockIdx.x - p.nwg) * NW + wave; idx < (C / 32) * ksall; idx += npack * NW) {
      const int ct = idx / ksall, ks = idx % ksall, c = ct * 32 + l32;
      float v[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const int n = ks * 16 + hh * 8 + e, s = n / HD;
        v[e] = s < 4 ? load1<A, F32>(p.w[s], (int64_t)(n - s * HD) * C + c)
                     : (n - 4 * HD < p.H ? load1<A, F32>(p.wb, (int64_t)(n - 4 * HD) * C + c) : 0.f);
      }
      Frag<F32> f;
      pack<A>(v, f);
      frag_write<F32>(static_cast<char*>(p.wt), idx, lane, f);
    }
    return;
  }
  float wv[NF][8];
#pragma unroll
  for (int n = 0; n < NF; ++n)
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int idx = wave + NW * n;
      wv[n][e] = load1<A, F32>(p.wo, (int64_t)((idx % KS) * 16 + hh * 8 + e) * HD + (idx / KS) * 32 + l32);
    }
  const int nitems = p.B * p.nper * p.cg, step = p.nwg * NW;
  int item = first_item(p.cg, p.nwg, wave);
  Frag<F32> f[KS];  // the next row block
  RowBlock rb = row_block(p, min(item, nitems - 1) / p.cg, lane);
  auto fetch = [&]() {
    const int64_t so = pair_off(p.douts, rb) + hh * 8;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) f[ks] = load8<F32>(p.dout, so + ks * 16);
  };
  fetch();
#pragma unroll
  for (int n = 0; n < NF; ++n) {
    Frag<F32> fw;
    pack<A>(wv[n], fw);
    op_write<F32>(smem, wave + NW * n, lane, to_op(fw));
  }
  __syncthreads();
  if (item >= nitems) return;
  auto head_at = [&](int t, const RowBlock& r) { const int h = t * 32 / p.D; return head_off(p, r, h) + (t * 32 - h * p.D) + hh * 8; };
  auto operands = [&](int t, const RowBlock& r, Frag<F32> (&gt)[2], Frag<false> (&o)[2]) {
    int64_t at0, at1;
    row_pair(head_at(t, r), at0, at1);
    load_runs<F32>(p.gate, at0, at1, lane, gt[0], gt[1]);
    load_runs<false>(p.o, at0, at1, lane, o[0], o[1]);
  };
  auto store_tile = [&](const floatx16& acc, int t, const RowBlock& r, const Frag<F32> (&gt)[2], const Frag<false> (&o)[2]) {
    int64_t at0, at1;
    row_pair(head_at(t, r), at0, at1);
    float y[2][8];
    rows8(acc, y);
    Frag<false> fo[2];
    Frag<F32> fd[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      float a[8], b[8], d[8];
      unpack<A>(gt[u], a);
      unpack<A>(o[u], b);
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        d[e] = y[u][e] * b[e] * a[e] * (1.0f - a[e]);
        y[u][e] *= a[e];
      }
      pack<A>(y[u], fo[u]);
      pack<A>(d, fd[u]);
    }
    store_runs<false>(p.dog, at0, at1, lane, fo);  // (rows beyond the end: once more the last one)
    store_runs<F32>(p.dgp, at0, at1, lane, fd);
  };
  [[maybe_unused]] bool bad = false;
  [[maybe_unused]] const int item0 = item;
  for (; item < nitems; item += step) {
    const RowBlock cur = rb;
    const int g = item % p.cg;
    Op<F32> x[KS];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) x[ks] = to_op(f[ks]);
    if (item + step < nitems) {
      rb = row_block(p, (item + step) / p.cg, lane);
      fetch();
    }
    for (int t = g; t < NT; t += p.cg) {
      Frag<F32> gt[2];
      Frag<false> o[2];
      operands(t, cur, gt, o);
      floatx16 acc = zero16();
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) acc = mma<A>(op_read<F32>(smem, t * KS + ks, lane), x[ks], acc);
      if constexpr (F32) bad = bad || not_finite(acc);
      store_tile(acc, t, cur, gt, o);
    }
  }
  if constexpr (F32)
    if (bad)
#pragma clang loop unroll(disable)
      for (item = item0; item < nitems; item += step) {
        const RowBlock cur = row_block(p, item / p.cg, lane);
        const int64_t so = pair_off(p.douts, cur) + hh * 8;
#pragma clang loop unroll(disable)
        for (int t = item % p.cg; t < NT; t += p.cg) {
          Frag<F32> gt[2];
          Frag<false> o[2];
          operands(t, cur, gt, o);
          floatx16 acc = zero16();
#pragma clang loop unroll(disable)
          for (int ks = 0; ks < KS; ++ks) {
            float w[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) w[e] = load1<A, F32>(p.wo, (int64_t)(ks * 16 + hh * 8 + e) * HD + t * 32 + l32);
            acc = mma_f32(w, load8<true>(p.dout, so + ks * 16).v, acc);
          }
          store_tile(acc, t, cur, gt, o);
        }
      }
}

// ---- backward: input gradient and layer norm ----------------------------------------------------------
// dx = sum of the five projections' input gradients, one product with 4*HD + 16 contraction elements (the bias
// heads padded to one 16-wide step).  A wave keeps the transposed weights of 32 channels in registers (132 of them in
// bf16; fp32: half of the contraction as fp32, 136, taken apart at every use because its planes, 204, do not fit beside
// the rest), the rows' gradients go through LDS once, and dx comes back through LDS in fp32 (one plane per share of the
// contraction) to the threads that hold the rows of z in the layer norm's layout: 8 channels of a row each, so that dz
// leaves in whole lines.
template <class A, bool F32, int C, int HD>
__global__ void __launch_bounds__(512) blk_dx_kernel(BlockParams p) {
  constexpr int TR = F32 ? 32 : 64, RS = TR / 32, NT = C / 32;
  constexpr int SPLIT = 8 / (RS * NT);                   // shares of the contraction
  constexpr int KH = HD / 16, KALL = 4 * KH + 1, KW = (KALL + SPLIT - 1) / SPLIT;
  constexpr int NP = TR * HD / 8 / 512;                  // pieces per thread of a section
  constexpr int NZ = (TR * C / 8 + 511) / 512;           // pieces of z
  constexpr int SUB = KALL * kOpBytes<F32>;
  constexpr int XROW = C + 4;                            // floats per row of a dx plane
  static_assert(NP >= 1 || F32, "pieces");
  constexpr int NPP = NP > 0 ? NP : 1;
  extern __shared__ char smem[];
  float* dxs = reinterpret_cast<float*>(smem + RS * SUB);
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), l32 = lane & 31, hh = lane >> 5;
  const int ct = wave % NT, rs = (wave / NT) % RS, share = wave / (NT * RS);
  const int c8 = (tid % (C / 8)) * 8;
  float gam[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) gam[e] = load1<A, F32>(p.gamma, c8 + e);

  const int LL = (int)p.LL, nst = (LL + TR - 1) / TR, ntot = p.B * nst;
  const float inv_l = 1.0f / (float)p.L;
  Frag<F32> z[NZ], dg[NPP];
  Frag<false> d[3][NPP];
  uint16_t rd[4];
  auto fetch = [&](int st) {
    const int b = st / nst, p0 = (st - b * nst) * TR;
#pragma unroll
    for (int n = 0; n < NPP; ++n) {
      const int pc = tid + 512 * n, e8 = (pc % (HD / 8)) * 8, h = e8 / p.D;
      const int q = min(p0 + pc / (HD / 8), LL - 1);
      const int64_t off = (((int64_t)b * p.H + h) * LL + q) * p.D + (e8 - h * p.D);
#pragma unroll
      for (int s = 0; s < 3; ++s) d[s][n] = load8<false>(p.dqkv[s], off);
      dg[n] = load8<F32>(p.dgp, off);
    }
#pragma unroll
    for (int h = 0; h < 4; ++h) rd[h] = static_cast<const uint16_t*>(p.db)[((int64_t)b * p.H + min(h, p.H - 1)) * LL + min(p0 + tid % TR, LL - 1)];
  };
  // (rows beyond the end, or beyond the stage, repeat the last one and store the same values there)
  auto pair_off_of = [&](const int64_t (&s)[3], int st, int n) {
    const int b = st / nst, r = (st - b * nst) * TR + min((tid + 512 * n) / (C / 8), TR - 1);
    const uint32_t q = (uint32_t)min(r, LL - 1), i = div_by_length(q, (uint32_t)p.L, inv_l), j = q - i * (uint32_t)p.L;
    return b * s[0] + (int64_t)i * s[1] + (int64_t)j * s[2] + c8;
  };
  auto put = [&]() {
#pragma unroll
    for (int n = 0; n < NPP; ++n) {
      const int pc = tid + 512 * n, row = pc / (HD / 8), c = pc % (HD / 8);
      if (NP >= 1 || row < TR) {
        char* blk = smem + (row / 32) * SUB;
#pragma unroll
        for (int s = 0; s < 3; ++s) {
          Frag<F32> f;
          if constexpr (F32) unpack<A>(d[s][n], f.v);
          else f = d[s][n];
          piece_write<F32, 2>(blk, row % 32, s * (HD / 8) + c, f);
        }
        piece_write<F32>(blk, row % 32, 3 * (HD / 8) + c, dg[n]);
      }
    }
    if (tid < 2 * TR) {  // (the second half of the step: zeros)
      float v[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
      if (tid < TR)
#pragma unroll
        for (int h = 0; h < 4; ++h) v[h] = h < p.H ? A::lo((uint32_t)rd[h]) : 0.f;
      Frag<F32> f;
      pack<A>(v, f);
      const int row = tid % TR;
      piece_write<F32, 2>(smem + (row / 32) * SUB, row % 32, 4 * (HD / 8) + tid / TR, f);
    }
  };
  int st = (int)blockIdx.x;
  fetch(min(st, ntot - 1));  // (in flight while the weights come in)
  // A share takes every SPLIT-th step, so that all have the same number from the fp16 gradients, whose third plane is zero, and begins with the
  // gate's: dz against 64 bits at 192 x 192 pairs in fp32 1.91e-7, with the gate's behind q, k and v, which are larger, 2.33e-7 (half of the
  // contraction in a row for each share 2.27e-7).  The last step is one share's (the others': the last one again, with zero weights).
  static_assert(3 * KH % SPLIT == 0 && KH % SPLIT == 0, "even shares of every section");
  constexpr int KG = KH / SPLIT;   // a share's steps of a section
  auto step_of = [=](int k) { return SPLIT == 1 ? k : k < KG ? (k + 3 * KG) * SPLIT + share : k < 4 * KG ? (k - KG) * SPLIT + share : KALL - 1; };
  Frag<F32> w[KW];
#pragma unroll
  for (int k = 0; k < KW; ++k) w[k] = frag_read<F32>(static_cast<const char*>(p.wt), ct * KALL + step_of(k), lane);
  if (SPLIT > 1 && share > 0) w[KW - 1] = frag_zero<F32>();
  if (st < ntot) put();
  __syncthreads();
  // the sums of a stage through LDS to the rows' threads, and the layer norm's backward
  auto finish = [&](const floatx16& acc, int st) {
    float* plane = dxs + ((size_t)share * TR + rs * 32 + l32) * XROW + ct * 32 + 4 * hh;
#pragma unroll
    for (int g = 0; g < 4; ++g) *reinterpret_cast<float4*>(plane + 8 * g) = make_float4(acc[4 * g], acc[4 * g + 1], acc[4 * g + 2], acc[4 * g + 3]);
    __syncthreads();
    // dz = rstd * (g - mean(g) - xhat * mean(g * xhat)), g = dx * gamma
#pragma unroll
    for (int n = 0; n < NZ; ++n) {
      const int row = min((tid + 512 * n) / (C / 8), TR - 1);
      float x[8], g[8], mean, rstd;
      unpack<A>(z[n], x);
      normalise<C>(x, p.eps, mean, rstd);
      if (c8 == 0) {
        const int b = st / nst, q = min((st - b * nst) * TR + row, LL - 1);
        p.stats[(int64_t)b * LL + q] = float2{mean, rstd};
      }
#pragma unroll
      for (int e = 0; e < 8; ++e) g[e] = 0.f;
#pragma unroll
      for (int s = 0; s < SPLIT; ++s) {
        const float* src = dxs + ((size_t)s * TR + row) * XROW + c8;
        const float4 a = *reinterpret_cast<const float4*>(src), b = *reinterpret_cast<const float4*>(src + 4);
        g[0] += a.x; g[1] += a.y; g[2] += a.z; g[3] += a.w;
        g[4] += b.x; g[5] += b.y; g[6] += b.z; g[7] += b.w;
      }
      float s1 = 0.f, s2 = 0.f;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        g[e] *= gam[e];
        s1 += g[e];
        s2 = __builtin_fmaf(g[e], x[e], s2);
      }
      s1 = row_sum<C / 8>(s1) * (1.0f / C);
      s2 = row_sum<C / 8>(s2) * (1.0f / C);
#pragma unroll
      for (int e = 0; e < 8; ++e) x[e] = rstd * (g[e] - s1 - x[e] * s2);
      Frag<F32> f;
      pack<A>(x, f);
      store8<F32>(p.dz, pair_off_of(p.dzs, st, n), f);
    }
  };
  [[maybe_unused]] bool bad = false;
  for (; st < ntot; st += (int)gridDim.x) {
    const int next = st + (int)gridDim.x;
#pragma unroll
    for (int n = 0; n < NZ; ++n) z[n] = load8<F32>(p.z, pair_off_of(p.zs, st, n));
    if constexpr (!F32) fetch(min(next, ntot - 1));
    floatx16 acc = zero16();
    if constexpr (F32) {
      // (the next step's operands are read during this one's products; the registers for that are the next stage's rows', which are
      // asked for behind the products)
      auto operand = [&](auto kc) {
        constexpr int k = decltype(kc)::value;
        return piece_frag<F32, (k >= KG) ? 2 : 3>(smem + rs * SUB, step_of(k), l32, hh);
      };
      Op<F32> x = operand(std::integral_constant<int, 0>{});
      static_for<0, KW>([&](auto kc) {
        constexpr int k = decltype(kc)::value;
        const Op<F32> cur = x;
        if constexpr (k + 1 < KW) x = operand(std::integral_constant<int, k + 1>{});
        acc = mma<A, 3, false, (k >= KG) ? 2 : 3>(to_op<true>(w[k]), cur, acc);
      });
      fetch(min(next, ntot - 1));
    } else {
#pragma unroll
      for (int k = 0; k < KW; ++k) acc = mma<A>(to_op<true>(w[k]), piece_frag<F32>(smem + rs * SUB, step_of(k), l32, hh), acc);
    }
    if constexpr (F32) bad = bad || not_finite(acc);
    finish(acc, st);
    if (next >= ntot) break;
    put();
    __syncthreads();
  }
  if constexpr (F32) {
    if (!__syncthreads_or(bad)) return;
#pragma clang loop unroll(disable)
    for (st = (int)blockIdx.x; st < ntot; st += (int)gridDim.x) {
#pragma unroll
      for (int n = 0; n < NZ; ++n) z[n] = load8<F32>(p.z, pair_off_of(p.zs, st, n));
      const int b = st / nst, q = min((st - b * nst) * TR + rs * 32 + l32, LL - 1);
      floatx16 acc = zero16();
#pragma clang loop unroll(disable)
      for (int ks = share; ks < KALL; ks += SPLIT) {
        const int s = ks / KH, e8 = (ks % KH) * 16 + hh * 8, h = e8 / p.D;
        const int64_t off = (((int64_t)b * p.H + h) * LL + q) * p.D + (e8 - h * p.D);
        float x[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
        if (s < 3) {
          unpack<A>(load8<false>(p.dqkv[s], off), x);
        } else if (s == 3) {
          unpack<A>(load8<true>(p.dgp, off), x);
        } else if (hh == 0) {
#pragma unroll
          for (int g = 0; g < 4; ++g)
            if (g < p.H) x[g] = load1<A, false>(p.db, ((int64_t)b * p.H + g) * LL + q);
        }
        acc = mma_f32(frag_read<true>(static_cast<const char*>(p.wt), ct * KALL + ks, lane).v, x, acc);
      }
      finish(acc, st);
      __syncthreads();
    }
  }
}

// ---- backward: weight gradients -----------------------------------------------------------------------
// Six products with the pair rows as contraction: section s = 0..3 is (d of projection s)^T xhat, with xhat
// the normalised row without gamma and beta (the reduction applies those: one product serves the weight, gamma
// and beta), section 4 is dout^T (gate * o), section 5 the bias projection's, which the workgroups of section 0 form beside
// theirs (by workgroups of its own, which loaded and normalised z for H columns, the launch took 80 us at 384 x 384 pairs in bf16 and 56
// at 192 x 192 in fp32; so 67 and 50).  A workgroup works off one chunk of
// rows of one section: stages of 64 rows (32 in fp32) are formed in registers, written to LDS as 32-column
// sub-tiles and read back transposed as MFMA operands; its waves own up to two 32 x 32 tiles of the result
// each.  The sums over the rows (bias gradients) are products with ones, in fp32 kept by the threads that load the rows; a row's mean
// and deviation come from blk_dx_kernel.  The sections of a chunk sit on one die, whose L2 serves z to four of them.
//
// Bound by memory: 300 MB in, z counted once, at 384 x 384 pairs in bf16 (4.5 TB/s).  A stage has 8 MFMAs per wave.  All
// addresses are a base plus the row, the next stage's loads are in flight during a stage, and two workgroups
// share a CU.  fp32: the three planes of a stage take the LDS of two, so a stage is read, then replaced between two
// barriers (with six sections 82 -> 55 us at 192 x 192 pairs; taken apart at every use instead, by up to four waves each, 69).  Sections in separate workgroups keep a partial sum at 64 KB (one workgroup for all six: 264 KB, 67 MB to
// write and read back over the chip, as much as the inputs at 384 x 384 pairs).
//
// One chunk's partial: the result tiles row-major [a][b], then (at C * HD) the row sums.
__host__ __device__ inline size_t wgrad_part_floats(int C, int HD) { return (size_t)C * HD + (C > HD ? C : HD); }
constexpr int kWgradSections = 6;   // of partial sums; the workgroups of section 0 form section 5, too
constexpr int wgrad_bias_bytes(int TR) { return 4 * (TR + 8) * 2; }  // dbias in a stage: a padded row per head

// Sub-tile of 32 columns in LDS: 16-bit rows of 64 bytes, swizzled as the attention's staged tiles; fp32: a plane of such
// rows after the other (PL of the three).
template <bool F32, int TR, int PL>
__device__ __forceinline__ void sub_write(char* tile, int row, int chunk, const Op<F32>& o) {
#pragma unroll
  for (int n = 0; n < (F32 ? PL : 1); ++n) *reinterpret_cast<u32x4*>(tile + n * (TR * 64) + 2 * swz_off<32>(row, chunk)) = o.p[n];
}
// Column l % 32 of the sub-tile, contraction rows rowbase + 8*(e/4) + 4*hh + e%4.
template <bool F32, int TR, int PL>
__device__ __forceinline__ Op<F32> sub_frag_t(const char* tile, int rowbase, const FragOffsets<32>& fo) {
  Op<F32> o;
#pragma unroll
  for (int n = 0; n < (F32 ? PL : 1); ++n)
    o.p[n] = __builtin_bit_cast(u32x4, lds_frag_t<32>(reinterpret_cast<const half_t*>(tile + n * (TR * 64)), rowbase, fo, 0));
  if constexpr (F32 && PL < 3) o.p[2] = u32x4{0, 0, 0, 0};
  return o;
}

enum WgradKind { kWgradQkv, kWgradGate, kWgradOut };

// BIAS: the bias heads' gradient, too, which are H more rows of operand A
template <class A, bool F32, int C, int HD, int KIND, bool BIAS = false>
__device__ __forceinline__ void wgrad_body(const BlockParams& p, int sec, int chunk, char* smem) {
  constexpr int NA = KIND == kWgradOut ? C / 32 : HD / 32;
  constexpr int NB = KIND == kWgradOut ? HD / 32 : C / 32;
  constexpr int NT = (NA * NB + 7) / 8;                 // result tiles per wave
  constexpr int TR = F32 ? 32 : 64;                     // rows per stage
  constexpr int PA = (TR * NA * 4 + 511) / 512;         // 8-element pieces per thread
  constexpr int PB = (TR * NB * 4 + 511) / 512;
  static_assert(4 * TR <= 512 && NA <= 4 && NB <= 4, "a thread has one dbias entry; a wave one tile more");
  constexpr int PLA = KIND == kWgradQkv ? 2 : 3;  // (fp32) planes of operand A: q, k, v's gradients are fp16
  constexpr int SUB = (F32 ? 3 : 1) * TR * 64;          // bytes of a sub-tile
  constexpr int BUFS = F32 ? 1 : 2;                     // stage buffers: two workgroups share a CU's LDS
  constexpr int DROW = TR + 8;                          // dbias: one row of TR entries per head
  constexpr int ABYTES = NA * SUB;
  constexpr int BUF = ABYTES + NB * SUB + (BIAS ? wgrad_bias_bytes(TR) : 0);
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), l32 = lane & 31, hh = lane >> 5;
  const int LL = (int)p.LL, nst = (LL + TR - 1) / TR;   // stages per batch entry
  const int ntot = p.B * nst, per = (ntot + p.nchunks - 1) / p.nchunks;
  const int first = chunk * per, last = min(ntot, first + per);
  FragOffsets<32> fo;
  fo.init(lane);

  const void* srca = KIND == kWgradQkv ? p.dqkv[sec] : KIND == kWgradGate ? p.dgp : p.dout;
  Frag<F32> ra[PA], rx[PB];
  Frag<false> ro[PB];
  float2 rs[PB];
  uint16_t rd = 0;
  // where this thread's pieces sit: row of the stage, and the offset of their first element inside row 0
  auto head_part = [&](int c8) { const int h = c8 / p.D; return ((int64_t)h * LL) * p.D + (c8 - h * p.D); };
  int64_t ao[PA], bo[PB];
#pragma unroll
  for (int n = 0; n < PA; ++n) {
    const int c8 = ((tid + 512 * n) % (NA * 4)) * 8;
    ao[n] = KIND == kWgradOut ? c8 : head_part(c8);
  }
#pragma unroll
  for (int n = 0; n < PB; ++n) {
    const int c8 = ((tid + 512 * n) % (NB * 4)) * 8;
    bo[n] = KIND == kWgradOut ? head_part(c8) : c8;
  }
  const float inv_l = 1.0f / (float)p.L;
  auto pair_row = [&](const int64_t (&s)[3], int b, int q) {
    const uint32_t i = div_by_length((uint32_t)q, (uint32_t)p.L, inv_l), j = (uint32_t)q - i * (uint32_t)p.L;
    return b * s[0] + (int64_t)i * s[1] + (int64_t)j * s[2];
  };
  auto fetch = [&](int st) {
    const int b = st / nst, p0 = (st - b * nst) * TR;
    const int64_t hb = (int64_t)b * p.H * LL * p.D;
#pragma unroll
    for (int n = 0; n < PA; ++n) {
      const int q = min(p0 + (tid + 512 * n) / (NA * 4), LL - 1);
      if constexpr (KIND == kWgradOut) ra[n] = load8<F32>(srca, pair_row(p.douts, b, q) + ao[n]);
      else if constexpr (KIND == kWgradGate) ra[n] = load8<F32>(srca, hb + (int64_t)q * p.D + ao[n]);
      else if constexpr (F32) unpack<A>(load8<false>(srca, hb + (int64_t)q * p.D + ao[n]), ra[n].v);
      else ra[n] = load8<false>(srca, hb + (int64_t)q * p.D + ao[n]);
    }
#pragma unroll
    for (int n = 0; n < PB; ++n) {
      const int q = min(p0 + (tid + 512 * n) / (NB * 4), LL - 1);
      if constexpr (KIND == kWgradOut) {
        rx[n] = load8<F32>(p.gate, hb + (int64_t)q * p.D + bo[n]);
        ro[n] = load8<false>(p.o, hb + (int64_t)q * p.D + bo[n]);
      } else {
        rx[n] = load8<F32>(p.z, pair_row(p.zs, b, q) + bo[n]);
        rs[n] = p.stats[(int64_t)b * LL + q];
      }
    }
    if constexpr (BIAS) {
      const int h = tid / TR, q = min(p0 + tid % TR, LL - 1);
      if (h < p.H) rd = static_cast<const uint16_t*>(p.db)[((int64_t)b * p.H + h) * LL + q];
    }
  };
  // forms operand B (gate * o, or the normalised row: the lanes of a row are neighbours) and writes both to LDS;
  // rows beyond the end are zero in both
  [[maybe_unused]] float csum[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};  // (fp32) of this thread's columns of operand A
  [[maybe_unused]] float dsum = 0.f;                                            // of this thread's dbias entry
  auto put = [&](char* buf, int st) {
    const int left = LL - (st % nst) * TR;
#pragma unroll
    for (int n = 0; n < PA; ++n) {
      const int pc = tid + 512 * n, row = pc / (NA * 4), c = pc % (NA * 4);
      if (TR * NA * 4 >= 512 || row < TR) {
        if (row >= left) ra[n] = frag_zero<F32>();
        sub_write<F32, TR, PLA>(buf + (c / 4) * SUB, row, c % 4, to_op(ra[n]));
        if constexpr (F32)
#pragma unroll
          for (int e = 0; e < 8; ++e) csum[e] += ra[n].v[e];
      }
    }
    if constexpr (BIAS) {
      const int h = tid / TR;
      if (h < p.H) {
        const uint16_t d = tid % TR < left ? rd : (uint16_t)0;  // (an infinite one times operand B's zeros would be NaN)
        reinterpret_cast<uint16_t*>(buf + ABYTES + NB * SUB)[h * DROW + tid % TR] = d;
        dsum += A::lo((uint32_t)d);
      }
    }
#pragma unroll
    for (int n = 0; n < PB; ++n) {
      const int pc = tid + 512 * n, row = pc / (NB * 4), c = pc % (NB * 4);
      float v[8];
      unpack<A>(rx[n], v);
      if constexpr (KIND == kWgradOut) {
        float w[8];
        unpack<A>(ro[n], w);
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] *= w[e];
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = (v[e] - rs[n].x) * rs[n].y;
      }
      Frag<F32> f;
      pack<A>(v, f);
      if (row >= left) f = frag_zero<F32>();
      if (TR * NB * 4 >= 512 || row < TR) sub_write<F32, TR, 3>(buf + ABYTES + (c / 4) * SUB, row, c % 4, to_op(f));
    }
  };
  // the bias heads as operand A: column l % 32 is head l % 32
  auto frag_d = [&](const char* buf, int k) {
    const char* s = buf + ABYTES + NB * SUB + ((size_t)(l32 < p.H ? l32 : 0) * DROW + k * 16 + 4 * hh) * 2;
    const u32x2 lo = *reinterpret_cast<const u32x2*>(s), hi = *reinterpret_cast<const u32x2*>(s + 16);
    Frag<false> d;
    d.w = u32x4{lo[0], lo[1], hi[0], hi[1]};
    if (l32 >= p.H) d = frag_zero<false>();
    if constexpr (F32) {
      Frag<true> f;
      unpack<A>(d, f.v);
      return to_op(f);
    } else {
      return to_op(d);
    }
  };

  auto head_tile = [&](const char* buf, int k, floatx16 c) {
    return mma<A, 2, false>(frag_d(buf, k), sub_frag_t<F32, TR, 3>(buf + ABYTES + (wave - 4) * SUB, k * 16, fo), c);
  };
  floatx16 acc[NT], more = zero16();
#pragma unroll
  for (int n = 0; n < NT; ++n) acc[n] = zero16();
  const int at = wave % NA;             // (NA divides 8: the same rows for both tiles of a wave)
  const bool own = wave < NA * NB;      // (fewer than eight tiles: the other waves only help staging)
  // one tile more: the row sums of operand A, as a product with ones (waves 0 .. NA - 1; fp32: by the threads that load the rows, since
  // three parts of an infinite entry would not sum to it), the bias heads' tiles (waves 4 .. 4 + NB - 1)
  const bool sums = !F32 && wave < NA, heads = BIAS && wave >= 4 && wave < 4 + NB;
  u32x4 ones;
#pragma unroll
  for (int e = 0; e < 4; ++e) ones[e] = A::is_bf16 ? 0x3F803F80u : 0x3C003C00u;
  if (first < last) {
    fetch(first);
    put(smem, first);
    if (first + 1 < last) fetch(first + 1);
    __syncthreads();
    for (int st = first; st < last; ++st) {
      const char* buf = smem + (BUFS == 2 ? (st - first) & 1 : 0) * BUF;
      if (own) {
#pragma unroll
        for (int k = 0; k < TR / 16; ++k) {
          const Op<F32> fa = sub_frag_t<F32, TR, PLA>(buf + at * SUB, k * 16, fo);
#pragma unroll
          for (int n = 0; n < NT; ++n)
            acc[n] = mma<A, PLA, PLA == 3>(fa, sub_frag_t<F32, TR, 3>(buf + ABYTES + (wave / NA + n * (8 / NA)) * SUB, k * 16, fo), acc[n]);
          if (sums) more = A::mfma(as_half8(fa.p[0]), as_half8(ones), more);
          if (NA * NB >= 8 && heads) more = head_tile(buf, k, more);
        }
        // (no unfinished product over the branches: the listings are checked line by line)
        if constexpr (BIAS) asm volatile("s_nop 15" : "+v"(more), "+v"(acc[NT - 1]));
      }
      if (NA * NB < 8 && heads) {
#pragma unroll
        for (int k = 0; k < TR / 16; ++k) more = head_tile(buf, k, more);
        asm volatile("s_nop 15" : "+v"(more));
      }
      if constexpr (BUFS == 1) __syncthreads();
      if (st + 1 < last) {
        put(smem + (BUFS == 2 ? (st + 1 - first) & 1 : 0) * BUF, st + 1);
        if (st + 2 < last) fetch(st + 2);
      }
      __syncthreads();
    }
  }
  if constexpr (F32) {
    bool again = not_finite(acc[0]);
#pragma unroll
    for (int n = 1; n < NT; ++n) again = again || not_finite(acc[n]);
    if (heads) again = again || not_finite(more);
    if ((own || heads) && again) {  // two rows at a time, one per lane half
      more = zero16();
#pragma unroll
      for (int n = 0; n < NT; ++n) acc[n] = zero16();
      const int col = at * 32 + l32;
#pragma clang loop unroll(disable)
      for (int r = first * TR; r < last * TR; r += 2) {
        const int st = r / TR, b = st / nst, row = (st - b * nst) * TR + r % TR + hh, q = min(row, LL - 1);
        const int64_t hb = (int64_t)b * p.H * LL * p.D + (int64_t)q * p.D;
        float x, y[NT];
        [[maybe_unused]] float xd = 0.f, yd = 0.f;
        if constexpr (KIND == kWgradOut) x = load1<A, true>(srca, pair_row(p.douts, b, q) + col);
        else x = load1<A, KIND == kWgradGate>(srca, hb + head_part(col));
        if constexpr (KIND == kWgradOut) {
#pragma unroll
          for (int n = 0; n < NT; ++n) {
            const int64_t off = hb + head_part((wave / NA + n * (8 / NA)) * 32 + l32);
            y[n] = load1<A, true>(p.gate, off) * load1<A, false>(p.o, off);
          }
        } else {
          const int64_t off = pair_row(p.zs, b, q) + l32;
          float z[NB], s = 0.f;
#pragma unroll
          for (int m = 0; m < NB; ++m) { z[m] = load1<A, true>(p.z, off + 32 * m); s += z[m]; }
#pragma unroll
          for (int m = 1; m < 32; m *= 2) s += __shfl_xor(s, m);
          const float mean = s * (1.0f / C);
          s = 0.f;
#pragma unroll
          for (int m = 0; m < NB; ++m) { z[m] -= mean; s = __builtin_fmaf(z[m], z[m], s); }
#pragma unroll
          for (int m = 1; m < 32; m *= 2) s += __shfl_xor(s, m);
          const float rstd = 1.0f / __builtin_sqrtf(s * (1.0f / C) + p.eps);
#pragma unroll
          for (int n = 0; n < NT; ++n) {
            y[n] = 0.f;
#pragma unroll
            for (int m = 0; m < NB; ++m) y[n] = wave / NA + n * (8 / NA) == m ? z[m] * rstd : y[n];
          }
          if constexpr (BIAS) {
            if (l32 < p.H && row < LL) xd = load1<A, false>(p.db, ((int64_t)b * p.H + l32) * LL + q);
#pragma unroll
            for (int m = 0; m < NB; ++m) yd = wave - 4 == m && row < LL ? z[m] * rstd : yd;
          }
        }
        if (row >= LL) x = 0.f;
#pragma unroll
        for (int n = 0; n < NT; ++n) acc[n] = __builtin_amdgcn_mfma_f32_32x32x2f32(x, row < LL ? y[n] : 0.f, acc[n], 0, 0, 0);
        if constexpr (BIAS) more = __builtin_amdgcn_mfma_f32_32x32x2f32(xd, yd, more, 0, 0, 0);
        asm volatile("s_nop 15" : "+v"(acc[0]), "+v"(acc[NT - 1]), "+v"(more));  // (the same)
      }
    }
  }
  // partial of this chunk
  float* out = p.part + ((size_t)sec * p.nchunks + chunk) * wgrad_part_floats(C, HD);
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const int a = at * 32 + 8 * (r / 4) + 4 * hh + r % 4;
    if (!own) continue;
#pragma unroll
    for (int n = 0; n < NT; ++n) out[(size_t)a * (NB * 32) + (wave / NA + n * (8 / NA)) * 32 + l32] = acc[n][r];
    if (sums && l32 == 0) out[(size_t)C * HD + a] = more[r];
  }
  float* ssum = reinterpret_cast<float*>(smem);  // (the last stage has been read: every wave is past its barrier)
  constexpr int PER = 512 / (NA * 4);
  if constexpr (F32) {
#pragma unroll
    for (int e = 0; e < 8; ++e) ssum[((tid % (NA * 4)) * 8 + e) * (PER + 1) + tid / (NA * 4)] = csum[e];
    __syncthreads();
    if (tid < NA * 32) {
      float s = 0.f;
      for (int k = 0; k < PER; ++k) s += ssum[tid * (PER + 1) + k];
      out[(size_t)C * HD + tid] = s;
    }
  }
  if constexpr (BIAS) {
    float* out5 = p.part + ((size_t)5 * p.nchunks + chunk) * wgrad_part_floats(C, HD);
    if (heads && hh == 0)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (r < p.H) out5[r * (NB * 32) + (wave - 4) * 32 + l32] = more[r];
    if constexpr (F32) __syncthreads();
    ssum[tid] = dsum;
    __syncthreads();
    if (tid < p.H) {
      float s = 0.f;
      for (int k = 0; k < TR; ++k) s += ssum[tid * TR + k];
      out5[(size_t)C * HD + tid] = s;
    }
  }
}

template <class A, bool F32, int C, int HD>
__global__ void __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(4))) blk_wgrad_kernel(BlockParams p) {
  extern __shared__ char smem[];
  const int slot = (int)blockIdx.x / kXcds;
  const int sec = slot % (kWgradSections - 1), chunk = (slot / (kWgradSections - 1)) * kXcds + (int)blockIdx.x % kXcds;
  if (sec == 0) wgrad_body<A, F32, C, HD, kWgradQkv, true>(p, sec, chunk, smem);
  else if (sec < 3) wgrad_body<A, F32, C, HD, kWgradQkv>(p, sec, chunk, smem);
  else if (sec == 3) wgrad_body<A, F32, C, HD, kWgradGate>(p, sec, chunk, smem);
  else wgrad_body<A, F32, C, HD, kWgradOut>(p, sec, chunk, smem);
}

// Sums the chunks in a fixed order: a workgroup takes half the columns of four rows of the projections' gradients (4*HD, then H of the
// bias projection) or of the output projection's (C), its threads four columns of a row and a group of chunks each.  (Whole rows
// were 161 workgroups at C = H*D = 128 and twelve chunks a thread, 10.7 us for 31 MB; this 322 and six, 9.2 us.)
// The rows' contributions to dgamma[c] = sum_n W[n][c] G[n][c] and dbeta[c] = sum_n W[n][c] * (sum over the
// pair rows of d[n]) go to p.red, one pair of rows of C floats per four rows.
__host__ __device__ inline int reduce_proj_groups(int HD, int H) { return (4 * HD + H + 3) / 4; }
template <class A, bool F32, int C, int HD>
__global__ void __launch_bounds__(1024) blk_reduce_kernel(BlockParams p) {
  __shared__ float4 part[1024];
  __shared__ float psum[1024];
  const int tid = threadIdx.x, ngp = reduce_proj_groups(HD, p.H);
  const int quad_rows = (int)blockIdx.x / 2, half = (int)blockIdx.x % 2;
  const bool proj = quad_rows < ngp;
  const int quads = (proj ? C : HD) / 8, groups = 256 / quads;
  const int row = tid / (quads * groups), grp = (tid / quads) % groups, c = (half * quads + tid % quads) * 4;
  const int n = (proj ? quad_rows : quad_rows - ngp) * 4 + row, nall = 4 * HD + p.H;
  const bool valid = !proj || n < nall;
  const int sec = !proj ? 4 : n < 4 * HD ? n / HD : 5, r = !proj ? n : n < 4 * HD ? n % HD : n - 4 * HD;
  const size_t pf = wgrad_part_floats(C, HD);
  float4 a = make_float4(0.f, 0.f, 0.f, 0.f);
  float sum = 0.f;
  if (valid) {
    const float* src = p.part + (size_t)sec * p.nchunks * pf;
#pragma unroll 8
    for (int k = grp; k < p.nchunks; k += groups) {
      const float4 v = *reinterpret_cast<const float4*>(src + (size_t)k * pf + (size_t)r * (quads * 8) + c);
      a.x += v.x; a.y += v.y; a.z += v.z; a.w += v.w;
      sum += src[(size_t)k * pf + (size_t)C * HD + r];
    }
  }
  part[tid] = a;
  psum[tid] = sum;
  __syncthreads();
  float dg[4] = {0.f, 0.f, 0.f, 0.f}, db[4] = {0.f, 0.f, 0.f, 0.f};
  if (grp == 0 && valid) {
    // (four sums side by side: twice as many groups in a row round once more often than half as many did)
    float g4[4][4], s4[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      s4[u] = 0.f;
#pragma unroll
      for (int e = 0; e < 4; ++e) g4[u][e] = 0.f;
    }
    for (int k = 0; k < groups; k += 4)
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const float4 v = part[tid + (k + u) * quads];
        g4[u][0] += v.x; g4[u][1] += v.y; g4[u][2] += v.z; g4[u][3] += v.w;
        s4[u] += psum[tid + (k + u) * quads];
      }
    float g[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) g[e] = (g4[0][e] + g4[1][e]) + (g4[2][e] + g4[3][e]);
    sum = (s4[0] + s4[1]) + (s4[2] + s4[3]);
    if (proj) {
      void* dst = sec < 4 ? p.dw[sec] : p.dwb;
      const void* w = sec < 4 ? p.w[sec] : p.wb;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float wv = load1<A, F32>(w, (int64_t)r * C + c + e);
        store1<A, F32>(dst, (int64_t)r * C + c + e, load1<A, F32>(p.gamma, c + e) * g[e] + load1<A, F32>(p.beta, c + e) * sum);
        dg[e] = wv * g[e];
        db[e] = wv * sum;
      }
      if (c == 0 && sec == 3 && p.dbg != nullptr) store1<A, F32>(p.dbg, r, sum);
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) store1<A, F32>(p.dwo, (int64_t)r * HD + c + e, g[e]);
      if (c == 0 && p.dbo != nullptr) store1<A, F32>(p.dbo, r, sum);
    }
  }
  if (!proj) return;
  // over the workgroup's four rows
  constexpr int CH = C / 2;
  __shared__ float4 sg[4 * (CH / 4)], sb[4 * (CH / 4)];
  if (grp == 0) {
    sg[row * quads + tid % quads] = make_float4(dg[0], dg[1], dg[2], dg[3]);
    sb[row * quads + tid % quads] = make_float4(db[0], db[1], db[2], db[3]);
  }
  __syncthreads();
  const float* f = reinterpret_cast<const float*>(tid < CH ? sg : sb);
  if (tid < 2 * CH) {
    const int col = tid % CH;
    p.red[((size_t)quad_rows * 2 + tid / CH) * C + half * CH + col] = f[col] + f[CH + col] + f[2 * CH + col] + f[3 * CH + col];
  }
}

// dgamma and dbeta from the workgroups' contributions: 16 columns per workgroup.
template <class A, bool F32>
__global__ void __launch_bounds__(1024) blk_norm_grad_kernel(BlockParams p, int C) {
  __shared__ float sm[1024];
  const int tid = threadIdx.x, col = (int)blockIdx.x * 16 + tid % 16, ngp = reduce_proj_groups(p.HD, p.H);
  float s = 0.f;  // (columns 0 .. C-1: dgamma, C .. 2C-1: dbeta)
  for (int n = tid / 16; n < ngp; n += 64) s += p.red[(size_t)n * 2 * C + col];
  sm[tid] = s;
  for (int w = 512; w >= 16; w /= 2) {
    __syncthreads();
    if (tid < w) sm[tid] += sm[tid + w];
  }
  if (tid < 16) store1<A, F32>(col < C ? p.dgamma : p.dbeta, col < C ? col : col - C, sm[tid]);
}

}  // namespace

// ---- host side ----------------------------------------------------------------------------------------
namespace {

constexpr int kCus = 256;

// (element type, fp32 block) instances
#define FTA_BLOCK_TYPES(X, ...) \
  if (dtype == kF16) X(F16, false, __VA_ARGS__) else if (dtype == kBF16) X(BF16, false, __VA_ARGS__) else X(F16, true, __VA_ARGS__)
#define FTA_BLOCK_C_HD(X)                                                                         \
  if (C == 64 && p.HD == 64) { FTA_BLOCK_TYPES(X, 64, 64) } else if (C == 64) { FTA_BLOCK_TYPES(X, 64, 128) } \
  else if (p.HD == 64) { FTA_BLOCK_TYPES(X, 128, 64) } else { FTA_BLOCK_TYPES(X, 128, 128) }

inline size_t frag_bytes(int dtype) { return dtype == 2 ? kFragBytes<true> : kFragBytes<false>; }
inline size_t op_bytes(int dtype) { return dtype == 2 ? kOpBytes<true> : kOpBytes<false>; }

// Column groups: a wave works off a row block's output tiles alone where there are enough row blocks for the
// eight waves of every CU, else neighbouring waves share them.
int column_groups(long blocks, int most) {
  int cg = 1;
  while (cg < most && blocks * cg < 8 * kCus) cg *= 2;
  return cg;
}
int workgroups(long items, int waves, int most) {
  const long n = (items + waves - 1) / waves;
  return (int)(n < most ? n : most);
}

}  // namespace

hipError_t launch_block_proj(BlockParams p, int C, int dtype, hipStream_t st) {
  // two stage buffers of 64 rows (fp32: 32) and the bias projection's weights
  const int rows = dtype == 2 ? 32 : 64;
  const size_t smem = (size_t)(2 * rows / 32 + 1) * (C / 16) * op_bytes(dtype) + (p.HD + 2 * rows) * sizeof(float);
  const int parts = dtype == 2 ? p.HD / 64 : 1;
  const dim3 grid((unsigned)(parts * workgroups((long)p.B * ((p.LL + rows - 1) / rows), 1, kCus / parts))), block(512);
#define FTA_BLOCK_CASE(AA, FF, CC, HH) return launch_kernel(blk_proj_kernel<AA, FF, CC, HH>, p, grid, block, smem, st);
  FTA_BLOCK_C_HD(FTA_BLOCK_CASE)
#undef FTA_BLOCK_CASE
}

hipError_t launch_block_out(BlockParams p, int C, int dtype, hipStream_t st) {
  const size_t smem = (size_t)(C / 32) * (p.HD / 16) * op_bytes(dtype) + C * sizeof(float);
  const long blocks = (long)p.B * p.nper;
  p.cg = column_groups(blocks, C / 32);
  const dim3 grid((unsigned)workgroups(blocks * p.cg, 8, dtype == 2 ? kCus : 2 * kCus)), block(512);
#define FTA_BLOCK_CASE(AA, FF, CC, HH) return launch_kernel(blk_out_kernel<AA, FF, CC, HH>, p, grid, block, smem, st);
  FTA_BLOCK_C_HD(FTA_BLOCK_CASE)
#undef FTA_BLOCK_CASE
}

hipError_t launch_block_dout(BlockParams p, int C, int dtype, hipStream_t st) {
  const size_t smem = (size_t)(p.HD / 32) * (C / 16) * op_bytes(dtype);
  const long blocks = (long)p.B * p.nper;
  p.cg = column_groups(blocks, p.HD / 32);
  p.nwg = workgroups(blocks * p.cg, 8, dtype == 2 ? kCus : 2 * kCus);
  const dim3 grid((unsigned)(p.nwg + 17)), block(512);  // (17: one fragment of the packed weights per wave at 4 x 33)
#define FTA_BLOCK_CASE(AA, FF, CC, HH) return launch_kernel(blk_dout_kernel<AA, FF, CC, HH>, p, grid, block, smem, st);
  FTA_BLOCK_C_HD(FTA_BLOCK_CASE)
#undef FTA_BLOCK_CASE
}

hipError_t launch_block_dx(BlockParams p, int C, int dtype, hipStream_t st) {
  const int rows = dtype == 2 ? 32 : 64, split = 8 / (rows / 32 * (C / 32));
  const size_t smem = (size_t)(rows / 32) * (4 * p.HD / 16 + 1) * op_bytes(dtype) + (size_t)split * rows * (C + 4) * sizeof(float);
  const dim3 grid((unsigned)workgroups((long)p.B * ((p.LL + rows - 1) / rows), 1, kCus)), block(512);
#define FTA_BLOCK_CASE(AA, FF, CC, HH) return launch_kernel(blk_dx_kernel<AA, FF, CC, HH>, p, grid, block, smem, st);
  FTA_BLOCK_C_HD(FTA_BLOCK_CASE)
#undef FTA_BLOCK_CASE
}

hipError_t launch_block_wgrad(BlockParams p, int C, int dtype, hipStream_t st) {
  // (the largest section: both operands C or HD columns wide, and a row of dbias per head)
  const int n = (p.HD + C) / 32;
  // (fp32: one stage of three planes)
  const size_t smem = dtype == 2 ? (size_t)n * 3 * 32 * 64 + wgrad_bias_bytes(32) : (size_t)2 * (n * 64 * 64 + wgrad_bias_bytes(64));
  const dim3 grid((unsigned)((kWgradSections - 1) * p.nchunks)), block(512);
  const dim3 rgrid((unsigned)(2 * (reduce_proj_groups(p.HD, p.H) + C / 4)));
#define FTA_BLOCK_CASE(AA, FF, CC, HH)                                                                       \
  {                                                                                                          \
    hipError_t e = launch_kernel(blk_wgrad_kernel<AA, FF, CC, HH>, p, grid, block, smem, st);                \
    if (e != hipSuccess) return e;                                                                           \
    hipLaunchKernelGGL((blk_reduce_kernel<AA, FF, CC, HH>), rgrid, dim3(1024), 0, st, p);                    \
    e = hipGetLastError();                                                                                   \
    if (e != hipSuccess) return e;                                                                           \
    hipLaunchKernelGGL((blk_norm_grad_kernel<AA, FF>), dim3((unsigned)(2 * CC / 16)), dim3(1024), 0, st, p, CC); \
    return hipGetLastError();                                                                                \
  }
  FTA_BLOCK_C_HD(FTA_BLOCK_CASE)
#undef FTA_BLOCK_CASE
}

// ---- C ABI ---------------------------------------------------------------------------------------------
namespace {

size_t align256(size_t n) { return (n + 255) / 256 * 256; }

// Byte offsets of the forward state and the backward workspace.
struct BlockLayout {
  size_t q, k, v, bias, o, gate, lse, state;
  size_t dog, dgp, dq, dk, dv, db, wt, stats, part, red, attn, attn_bytes, total;
  int nchunks;
};
bool block_supported(const fta_block& b) {
  return b.B >= 1 && b.L >= 1 && (b.C == 64 || b.C == 128) && (b.D == 32 || b.D == 64) && b.H >= 1 && b.H <= 32 &&
         (b.H * b.D == 64 || b.H * b.D == 128) && b.dtype >= 0 && b.dtype <= FTA_DTYPE_F32;
}
fta_options attn_options(const fta_block& b) {
  fta_options o{};
  o.dtype = b.dtype == FTA_DTYPE_BF16 ? FTA_DTYPE_BF16 : FTA_DTYPE_F16;
  o.dropout_p = b.dropout_p;
  o.seed = b.seed;
  o.precise = b.precise;
  return o;
}
BlockLayout block_layout(const fta_block& b) {
  BlockLayout l{};
  const size_t LL = (size_t)b.L * b.L, HD = (size_t)b.H * b.D, n = (size_t)b.B * LL * HD, m = (size_t)b.B * LL * b.H;
  const size_t es = b.dtype == FTA_DTYPE_F32 ? 4 : 2;
  size_t at = 0;
  auto take = [&](size_t bytes) { const size_t r = at; at += align256(bytes); return r; };
  l.q = take(2 * n); l.k = take(2 * n); l.v = take(2 * n); l.o = take(2 * n);
  l.bias = take(2 * m); l.gate = take(es * n); l.lse = take(4 * m);
  l.state = at;
  at = 0;
  l.dog = take(2 * n); l.dgp = take(es * n); l.dq = take(2 * n); l.dk = take(2 * n); l.dv = take(2 * n); l.db = take(2 * m);
  l.wt = take((size_t)(b.C / 32) * (4 * HD / 16 + 1) * frag_bytes(b.dtype));
  l.stats = take((size_t)b.B * LL * sizeof(float2));
  // Chunks of the weight-gradient kernel, a multiple of the dies: five sections of 96 are 480 workgroups, of which two
  // fit a CU (with six sections 56: 118 us at 384 x 384 pairs in bf16, 40: 110, 80: 91).  A chunk keeps at least four stages, so that its partial sums (64 KB at C = H*D = 128) are not
  // what the launch spends its time on.
  const size_t rows = b.dtype == FTA_DTYPE_F32 ? 32 : 64, stages = b.B * ((LL + rows - 1) / rows);
  l.nchunks = kXcds * (int)(stages < 64 ? 1 : stages > 32 * 12 ? 12 : stages / 32);
  l.part = take((size_t)kWgradSections * l.nchunks * wgrad_part_floats(b.C, (int)HD) * sizeof(float));
  l.red = take((size_t)reduce_proj_groups((int)HD, b.H) * 2 * b.C * sizeof(float));
  const fta_options opt = attn_options(b);
  l.attn_bytes = fta_bwd_workspace_bytes_ex(b.B, b.H, b.L, b.L, b.D, &opt);
  l.attn = take(l.attn_bytes);
  l.total = at;
  return l;
}
int check_stride(const void* ptr, const int64_t* s) {
  if (ptr == nullptr) return FTA_ERR_NULL_POINTER;
  if (reinterpret_cast<uintptr_t>(ptr) % 16 != 0) return FTA_ERR_MISALIGNED;
  for (int i = 0; i < 3; ++i)
    if (s[i] < 0 || s[i] % 8 != 0) return FTA_ERR_STRIDE;
  return FTA_OK;
}
int check_block(const fta_block* b) {
  if (b == nullptr) return FTA_ERR_NULL_POINTER;
  if (b->dtype < 0 || b->dtype > FTA_DTYPE_F32) return FTA_ERR_DTYPE;
  if (b->B < 1 || b->H < 1) return FTA_ERR_BATCH;
  if (b->D != 32 && b->D != 64) return FTA_ERR_HEAD_DIM;
  if (!block_supported(*b)) return FTA_ERR_BLOCK_SHAPE;
  const fta_options opt = attn_options(*b);
  if (!(opt.dropout_p >= 0.0f) || !(opt.dropout_p < 1.0f)) return FTA_ERR_DROPOUT;
  if (b->L < 1 || !fta_seq_len_supported_ex(b->L, b->D, &opt)) return FTA_ERR_SEQ_LEN;
  const int rc = check_stride(b->z, b->z_stride);
  if (rc != FTA_OK) return rc;
  for (const void* w : {b->norm_weight, b->norm_bias, b->wq, b->wk, b->wv, b->wb, b->wg, b->wo}) {
    if (w == nullptr) return FTA_ERR_NULL_POINTER;
    if (reinterpret_cast<uintptr_t>(w) % 16 != 0) return FTA_ERR_MISALIGNED;
  }
  return FTA_OK;
}
BlockParams block_params(const fta_block& b, const BlockLayout& l, char* state) {
  BlockParams p{};
  p.z = b.z;
  for (int i = 0; i < 3; ++i) p.zs[i] = b.z_stride[i];
  p.mask = b.mask;
  p.w[0] = b.wq; p.w[1] = b.wk; p.w[2] = b.wv; p.w[3] = b.wg;
  p.wb = b.wb; p.bg = b.bg; p.wo = b.wo; p.bo = b.bo;
  p.gamma = b.norm_weight; p.beta = b.norm_bias;
  p.qkv[0] = state + l.q; p.qkv[1] = state + l.k; p.qkv[2] = state + l.v;
  p.gate = state + l.gate; p.bias = state + l.bias; p.o = state + l.o;
  p.B = b.B; p.L = b.L; p.H = b.H; p.D = b.D; p.HD = b.H * b.D;
  p.LL = (int64_t)b.L * b.L;
  p.nper = (int)((p.LL + 31) / 32);
  p.cg = 1;
  p.eps = b.eps;
  return p;
}
fta_tensor5 head_tensor(const fta_block& b, const void* ptr) {
  const int64_t row = (int64_t)b.L * b.D;
  return fta_tensor5{const_cast<void*>(ptr), {row * b.L * b.H, row * b.L, row, b.D}};
}
fta_tensor4 bias_tensor(const fta_block& b, const void* ptr) {
  const int64_t LL = (int64_t)b.L * b.L;
  return fta_tensor4{const_cast<void*>(ptr), {LL * b.H, LL, b.L}};
}

}  // namespace
}  // namespace fta

extern "C" {

int fta_block_check(const fta_block* b) { return fta::check_block(b); }

size_t fta_block_state_bytes(const fta_block* b) {
  return (b == nullptr || !fta::block_supported(*b)) ? 0 : fta::block_layout(*b).state;
}

size_t fta_block_bwd_workspace_bytes(const fta_block* b) {
  return (b == nullptr || !fta::block_supported(*b)) ? 0 : fta::block_layout(*b).total;
}

int fta_block_fwd(const fta_block* b, void* out, const int64_t out_stride[3], void* state, void* stream) {
  int rc = fta::check_block(b);
  if (rc != FTA_OK || (rc = fta::check_stride(out, out_stride)) != FTA_OK) return rc;
  if (state == nullptr) return FTA_ERR_NULL_POINTER;
  if (reinterpret_cast<uintptr_t>(state) % 16 != 0) return FTA_ERR_MISALIGNED;
  if ((rc = fta::check_device()) != FTA_OK) return rc;
  const fta::BlockLayout l = fta::block_layout(*b);
  char* s = static_cast<char*>(state);
  fta::BlockParams p = fta::block_params(*b, l, s);
  p.out = out;
  for (int i = 0; i < 3; ++i) p.outs[i] = out_stride[i];
  hipStream_t st = static_cast<hipStream_t>(stream);
  hipError_t e = fta::launch_block_proj(p, b->C, b->dtype, st);
  if (e != hipSuccess) return static_cast<int>(e);
  const fta_options opt = fta::attn_options(*b);
  const fta_tensor5 q = fta::head_tensor(*b, s + l.q), k = fta::head_tensor(*b, s + l.k), v = fta::head_tensor(*b, s + l.v);
  const fta_tensor5 o = fta::head_tensor(*b, s + l.o);
  const fta_tensor4 bias = fta::bias_tensor(*b, s + l.bias);
  rc = fta_fwd_ex(&q, &k, &v, &bias, &o, reinterpret_cast<float*>(s + l.lse), b->B, b->H, b->L, b->L, b->D, b->sm_scale, &opt, stream);
  if (rc != FTA_OK) return rc;
  return static_cast<int>(fta::launch_block_out(p, b->C, b->dtype, st));
}

int fta_block_bwd(const fta_block* b, const void* state, const void* dout, const int64_t dout_stride[3],
                  const fta_block_grads* g, void* workspace, size_t workspace_bytes, void* stream) {
  int rc = fta::check_block(b);
  if (rc != FTA_OK || (rc = fta::check_stride(dout, dout_stride)) != FTA_OK) return rc;
  if (g == nullptr || state == nullptr || workspace == nullptr) return FTA_ERR_NULL_POINTER;
  if ((rc = fta::check_stride(g->z, g->z_stride)) != FTA_OK) return rc;
  for (const void* w : {g->norm_weight, g->norm_bias, g->wq, g->wk, g->wv, g->wb, g->wg, g->wo})
    if (w == nullptr) return FTA_ERR_NULL_POINTER;
  if (reinterpret_cast<uintptr_t>(state) % 16 != 0 || reinterpret_cast<uintptr_t>(workspace) % 16 != 0) return FTA_ERR_MISALIGNED;
  const fta::BlockLayout l = fta::block_layout(*b);
  if (workspace_bytes < l.total) return FTA_ERR_WORKSPACE;
  if ((rc = fta::check_device()) != FTA_OK) return rc;
  char* s = const_cast<char*>(static_cast<const char*>(state));
  char* w = static_cast<char*>(workspace);
  fta::BlockParams p = fta::block_params(*b, l, s);
  p.dout = dout;
  p.dz = g->z;
  for (int i = 0; i < 3; ++i) { p.douts[i] = dout_stride[i]; p.dzs[i] = g->z_stride[i]; }
  p.dog = w + l.dog; p.dgp = w + l.dgp;
  p.dqkv[0] = w + l.dq; p.dqkv[1] = w + l.dk; p.dqkv[2] = w + l.dv; p.db = w + l.db;
  p.wt = w + l.wt;
  p.stats = reinterpret_cast<float2*>(w + l.stats);
  p.part = reinterpret_cast<float*>(w + l.part);
  p.red = reinterpret_cast<float*>(w + l.red);
  p.dw[0] = g->wq; p.dw[1] = g->wk; p.dw[2] = g->wv; p.dw[3] = g->wg;
  p.dwb = g->wb; p.dbg = g->bg; p.dwo = g->wo; p.dbo = g->bo; p.dgamma = g->norm_weight; p.dbeta = g->norm_bias;
  p.nchunks = l.nchunks;
  hipStream_t st = static_cast<hipStream_t>(stream);
  hipError_t e = fta::launch_block_dout(p, b->C, b->dtype, st);
  if (e != hipSuccess) return static_cast<int>(e);
  const fta_options opt = fta::attn_options(*b);
  const fta_tensor5 q = fta::head_tensor(*b, s + l.q), k = fta::head_tensor(*b, s + l.k), v = fta::head_tensor(*b, s + l.v);
  const fta_tensor5 o = fta::head_tensor(*b, s + l.o), dog = fta::head_tensor(*b, w + l.dog);
  const fta_tensor5 dq = fta::head_tensor(*b, w + l.dq), dk = fta::head_tensor(*b, w + l.dk), dv = fta::head_tensor(*b, w + l.dv);
  const fta_tensor4 bias = fta::bias_tensor(*b, s + l.bias), db = fta::bias_tensor(*b, w + l.db);
  rc = fta_bwd_ex(&q, &k, &v, &bias, &o, reinterpret_cast<const float*>(s + l.lse), &dog, &dq, &dk, &dv, &db, w + l.attn, l.attn_bytes,
                  b->B, b->H, b->L, b->L, b->D, b->sm_scale, &opt, stream);
  if (rc != FTA_OK) return rc;
  e = fta::launch_block_dx(p, b->C, b->dtype, st);
  if (e != hipSuccess) return static_cast<int>(e);
  return static_cast<int>(fta::launch_block_wgrad(p, b->C, b->dtype, st));
}

}  // extern "C"
