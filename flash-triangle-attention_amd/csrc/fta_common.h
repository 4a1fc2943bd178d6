// Shared device helpers for the gfx950 triangle-attention kernels.
//
// Register layouts of v_mfma_f32_32x32x16_f16 (wave64), checked on hardware:
//   A (32 x 16): lane l holds row  l%32, k = 8*(l/32) .. +7   (8 halfs)
//   B (16 x 32): lane l holds col  l%32, k = 8*(l/32) .. +7   (8 halfs)
//   C/D (32x32): lane l holds col  l%32, register r holds row 8*(r/4) + 4*(l/32) + r%4
// The contraction index may be permuted freely as long as A and B use the same permutation.
// A C tile reused as a B operand (the P^T -> P^T*V^T trick) therefore uses, for the u-th
// 16-wide contraction step, registers 8u..8u+7, i.e. rows (2u + e/4)*8 + 4*(l/32) + e%4.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace fta {

typedef _Float16 half_t;
typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
typedef _Float16 half4_t __attribute__((ext_vector_type(4)));
typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef __fp16 fp16x4_b __attribute__((__vector_size__(4 * sizeof(__fp16))));
typedef __attribute__((address_space(3))) fp16x4_b lds_fp16x4_b;

constexpr float kLog2e = 1.4426950408889634f;
constexpr int kXcds = 8;  // MI355X: 8 accelerator dies, workgroups are dealt round-robin to them

__device__ __forceinline__ floatx16 mfma32(half8_t a, half8_t b, floatx16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ float exp2_fast(float x) { return __builtin_amdgcn_exp2f(x); }

// Row constants -lse and -delta that enter through the matrix core: one extra 16-wide contraction step adds the constant c to every
// element of an accumulator column or row, with c as a pair of 16-bit values on two contraction slots of one operand and
// their factors on the same slots of the other, zeros elsewhere.  -lse: split_2048(c), fp16 for every element type, against {2048, 1} on
// slots 0 and 1.  -delta has the range of the incoming gradient: T::delta_pair(c) against T::kDeltaOnes on slots 2 and 3, through
// T's MFMA.  (Either pair meets zeros of the other's step: a finite fp16 is finite read as bf16, a bf16 below 2^121 read as fp16.)
constexpr uint32_t kLseOnes = 0x3C006800u;
template <class T>
__device__ __forceinline__ half8_t aug_ones() {
  return __builtin_bit_cast(half8_t, u32x4{kLseOnes, T::kDeltaOnes, 0u, 0u});
}

// Two floats -> packed fp16 pair (round toward zero), as raw bits.
__device__ __forceinline__ uint32_t pack_rtz(float a, float b) {
  auto p = __builtin_amdgcn_cvt_pkrtz(a, b);
  return __builtin_bit_cast(uint32_t, p);
}

// Two floats -> packed fp16 pair (round to nearest even), as raw bits.
__device__ __forceinline__ uint32_t pack_rn(float a, float b) {
  half2_t p = {(half_t)a, (half_t)b};
  return __builtin_bit_cast(uint32_t, p);
}

__device__ __forceinline__ half2_t as_half2(uint32_t u) { return __builtin_bit_cast(half2_t, u); }

// The stationary bias of the kernels that add it through the matrix core: bias * log2(e) as fp16, kept
// FINITE.  A masked key (-inf, or anything whose product with log2(e) leaves the fp16 range, such as
// the usual -1e9 cast to fp16) would otherwise meet the zeros of the one-hot selector inside a
// contraction step (0 * inf = NaN for the other 15 keys of the step).  At the floor the exponent
// still underflows to exactly 0, as it does upstream (flash_tt_attn.py:78, :344-346, :418-420).
constexpr float kBiasFloorLog2 = -60000.0f;
__device__ __forceinline__ uint32_t bias_log2_half2(uint32_t u) {
  half2_t h = __builtin_bit_cast(half2_t, u);
  return pack_rn(__builtin_fmaxf((float)h[0] * kLog2e, kBiasFloorLog2), __builtin_fmaxf((float)h[1] * kLog2e, kBiasFloorLog2));
}

// The bias as it is added on the vector ALU (natural units), kept at or above kMaskedBias: -inf would be harmless there
// unless EVERY key a query has seen so far is masked (the running maximum is then -inf and the exponent becomes
// inf - inf).  At the floor a masked key still gets weight exp(-59904 - m) = 0 as soon as one unmasked key has been
// seen, and a leading run of masked keys is rescaled away like any other early partial sum.  A query whose keys are ALL at
// the floor attends by its scores alone (to their rounding beside the floor, 2^-8), as it would with a finite mask value:
// the floor is one value, exact in fp16 and in bf16, for the forward and for every backward kernel, because the backward
// forms its weights from the forward's logsumexp.  (bf16 had a floor of -2^30, beside which the rounding of the
// exponent alone is 2^6: the weights of such a query came out of the backward wrong by up to 2^64.)
constexpr float kMaskedBias = -59904.0f;
// The keys that a row's last tile has beyond the row (copies of the last real one) stand still lower, at kBeyond2 of the
// element type, a packed pair of -65280: beside masked keys, too, their weight is exactly 0.
__device__ __forceinline__ uint32_t finite_half2(uint32_t u) {
  half2_t h = __builtin_bit_cast(half2_t, u);
  const half2_t lowest = {(half_t)kMaskedBias, (half_t)kMaskedBias};
  h = __builtin_elementwise_max(h, lowest);
  return __builtin_bit_cast(uint32_t, h);
}

// -lse for the kernels that add bias * log2(e) through the matrix core.  A logsumexp below the floor of that bias belongs to
// a query that has no key above it: forward and backward then hold the masked keys at different values, -59904 log2(e)
// and -60000, and the difference goes into the constant, so that the weights are again those of the scores alone
// (without it the exponent is +26423 and the gradients inf and NaN).  Where all of a query's biases lie between
// the two floors, -59904 and -41588, the weights come out as 0.
constexpr float kMaskedShiftLog2 = (float)(-(double)kMaskedBias * 1.4426950408889634 + (double)kBiasFloorLog2);
__device__ __forceinline__ float folded_lse(float lse) { return lse < kBiasFloorLog2 ? -kMaskedShiftLog2 - lse : -lse; }

// Eight halfs times an fp32 factor, rounded to nearest: the mixed-precision FMA converts, multiplies
// and rounds in one instruction per element (the product is rounded once, to fp16).  The results
// usually feed an MFMA, which may not read a register in the two issue slots after a vector-ALU
// write to it; the compiler cannot see that these are vector-ALU writes, hence the trailing s_nop.
__device__ __forceinline__ half8_t scale_half8(half8_t x, float f) {
  const u32x4 w = __builtin_bit_cast(u32x4, x);
  uint32_t r0, r1, r2, r3;
  asm("v_fma_mixlo_f16 %0, %4, %8, 0 op_sel_hi:[1,0,0]\n\t"
      "v_fma_mixhi_f16 %0, %4, %8, 0 op_sel:[1,0,0] op_sel_hi:[1,0,0]\n\t"
      "v_fma_mixlo_f16 %1, %5, %8, 0 op_sel_hi:[1,0,0]\n\t"
      "v_fma_mixhi_f16 %1, %5, %8, 0 op_sel:[1,0,0] op_sel_hi:[1,0,0]\n\t"
      "v_fma_mixlo_f16 %2, %6, %8, 0 op_sel_hi:[1,0,0]\n\t"
      "v_fma_mixhi_f16 %2, %6, %8, 0 op_sel:[1,0,0] op_sel_hi:[1,0,0]\n\t"
      "v_fma_mixlo_f16 %3, %7, %8, 0 op_sel_hi:[1,0,0]\n\t"
      "v_fma_mixhi_f16 %3, %7, %8, 0 op_sel:[1,0,0] op_sel_hi:[1,0,0]\n\t"
      "s_nop 1"
      : "=&v"(r0), "=&v"(r1), "=&v"(r2), "=&v"(r3)
      : "v"(w[0]), "v"(w[1]), "v"(w[2]), "v"(w[3]), "v"(f));
  return __builtin_bit_cast(half8_t, u32x4{r0, r1, r2, r3});
}

// c = 2048*hi + lo with hi, lo fp16: about 22 significant bits over the range |c| < 1.3e8.
// Returned as the packed pair (hi in the low half); the matching MFMA operand holds {2048, 1}.
__device__ __forceinline__ uint32_t split_2048(float c) {
  const half_t hi = (half_t)(c * (1.0f / 2048.0f));
  const half_t lo = (half_t)__builtin_fmaf(-2048.0f, (float)hi, c);
  half2_t p = {hi, lo};
  return __builtin_bit_cast(uint32_t, p);
}

__device__ __forceinline__ half8_t as_half8(u32x4 u) { return __builtin_bit_cast(half8_t, u); }

// v_permlane32_swap exchanges the upper 32 lanes of its first register with the lower 32 lanes of
// its second one.  Fed the same value x twice it leaves {x.lower, x.lower} and {x.upper, x.upper}:
// every lane then sees both halves' values.  The second copy is made opaque to the optimiser,
// which otherwise folds the two (distinct) results of a swap with identical inputs into one.
__device__ __forceinline__ void both_halves(float x, float& lower, float& upper) {
  uint32_t u = __builtin_bit_cast(uint32_t, x);
  uint32_t w = u;
  asm volatile("" : "+v"(w));
  auto r = __builtin_amdgcn_permlane32_swap(u, w, false, false);
  lower = __builtin_bit_cast(float, (uint32_t)r[0]);
  upper = __builtin_bit_cast(float, (uint32_t)r[1]);
}
__device__ __forceinline__ float max_both_halves(float x) {
  float a, b;
  both_halves(x, a, b);
  return __builtin_fmaxf(a, b);
}
__device__ __forceinline__ float sum_both_halves(float x) {
  float a, b;
  both_halves(x, a, b);
  return a + b;
}

// ---- element types ---------------------------------------------------------------------------------
// The 16-bit element type of q, k, v, bias and the gradients.  Fragments travel as raw bits (half8_t,
// uint32_t pairs) everywhere; these traits hold what depends on the format: the MFMA, conversions,
// the packed row sum, and the bit patterns of the masked bias.
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));

struct F16 {
  static constexpr bool is_bf16 = false;
  static constexpr uint32_t kNegInf2 = 0xFC00FC00u;  // packed pair of -inf
  static constexpr uint32_t kBeyond2 = 0xFBF8FBF8u;  // packed pair of -65280
  static __device__ __forceinline__ floatx16 mfma(half8_t a, half8_t b, floatx16 c) { return mfma32(a, b, c); }
  static __device__ __forceinline__ float lo(uint32_t u) { return (float)as_half2(u)[0]; }
  static __device__ __forceinline__ float hi(uint32_t u) { return (float)as_half2(u)[1]; }
  static __device__ __forceinline__ float get(half8_t v, int e) { return (float)v[e]; }
  static __device__ __forceinline__ uint32_t pack(float a, float b) { return pack_rn(a, b); }        // round to nearest
  static __device__ __forceinline__ uint32_t pack_fast(float a, float b) { return pack_rtz(a, b); }  // operands of the next MFMA
  static __device__ __forceinline__ float sum2(uint32_t u, float acc) {  // acc + both halves
    const half2_t ones = {(half_t)1.0f, (half_t)1.0f};
    return __builtin_amdgcn_fdot2(as_half2(u), ones, acc, false);
  }
  static __device__ __forceinline__ uint32_t finite2(uint32_t u) { return finite_half2(u); }
  // -- what the hand-scheduled backward kernels need
  static __device__ __forceinline__ half8_t scale8(half8_t x, float f) { return scale_half8(x, f); }
  static __device__ __forceinline__ uint32_t bias_log2(uint32_t u) { return bias_log2_half2(u); }  // -> fp16 pair
  // The bias pair as it is (natural units: nothing is rounded), kept above the floor that stands for -inf.
  static __device__ __forceinline__ uint32_t bias_nat(uint32_t u) { return finite_half2(u); }
  // The product kept to 22 bits: hi = the rounded product, lo = what the rounding dropped, itself
  // rounded.  An MFMA over hi plus one over lo gives the scores the precision of an fp32 product
  // (the precise mode, where scores of several tens would feel the 11-bit rounding of hi alone).
  static __device__ __forceinline__ void scale8_hilo(half8_t x, float f, half8_t& hi8, half8_t& lo8) {
    const u32x4 w = __builtin_bit_cast(u32x4, x);
    u32x4 rh, rl;
    // (as assembly: lo has to be taken against the very hi that the matrix core gets.  From C++ the
    // compiler forms hi twice, once rounding the exact product for the subtraction and once rounding
    // the fp32 product for the operand, and the two differ wherever the product lies at a rounding
    // tie of fp16 -- every tenth element at a scale like 1.3 -- which leaves a whole unit of hi's
    // last place uncorrected there)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      uint32_t h, l;
      asm("v_fma_mixlo_f16 %0, %2, %3, 0 op_sel_hi:[1,0,0]\n\t"
          "v_fma_mixhi_f16 %0, %2, %3, 0 op_sel:[1,0,0] op_sel_hi:[1,0,0]\n\t"
          "v_fma_mixlo_f16 %1, %2, %3, -%0 op_sel_hi:[1,0,1]\n\t"
          "v_fma_mixhi_f16 %1, %2, %3, -%0 op_sel:[1,0,1] op_sel_hi:[1,0,1]"
          : "=&v"(h), "=&v"(l) : "v"(w[e]), "v"(f));
      rh[e] = h; rl[e] = l;
    }
    asm volatile("s_nop 1" : "+v"(rh), "+v"(rl));
    hi8 = __builtin_bit_cast(half8_t, rh);
    lo8 = __builtin_bit_cast(half8_t, rl);
  }
  static __device__ __forceinline__ float dot2(uint32_t a, uint32_t b, float acc) {
    return __builtin_amdgcn_fdot2(as_half2(a), as_half2(b), acc, false);
  }
  // 1 / (what the fp16 bit pattern of 1.0 is worth as an operand of this type's MFMA)
  static constexpr float kOneHotInv = 1.0f;
  // -delta as a pair for the matrix core, and the pair of its factors (see aug_ones)
  static __device__ __forceinline__ uint32_t delta_pair(float c) { return split_2048(c); }
  static constexpr uint32_t kDeltaOnes = kLseOnes;
  // Element-wise sum of two packed pairs, rounded once (what adding in fp32 and rounding gives too).
  static __device__ __forceinline__ uint32_t add2(uint32_t a, uint32_t b) {
    return __builtin_bit_cast(uint32_t, as_half2(a) + as_half2(b));
  }
};

struct BF16 {
  static constexpr bool is_bf16 = true;
  static constexpr uint32_t kNegInf2 = 0xFF80FF80u;
  static constexpr uint32_t kBeyond2 = 0xC77FC77Fu;
  static __device__ __forceinline__ floatx16 mfma(half8_t a, half8_t b, floatx16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
  }
  static __device__ __forceinline__ float lo(uint32_t u) { return __builtin_bit_cast(float, u << 16); }
  static __device__ __forceinline__ float hi(uint32_t u) { return __builtin_bit_cast(float, u & 0xFFFF0000u); }
  static __device__ __forceinline__ float get(half8_t v, int e) {
    const u32x4 w = __builtin_bit_cast(u32x4, v);
    return (e & 1) ? hi(w[e >> 1]) : lo(w[e >> 1]);
  }
  static __device__ __forceinline__ uint32_t pack(float a, float b) {
    bf16x2_t p = {(__bf16)a, (__bf16)b};  // v_cvt_pk_bf16_f32: round to nearest even
    return __builtin_bit_cast(uint32_t, p);
  }
  static __device__ __forceinline__ uint32_t pack_fast(float a, float b) { return pack(a, b); }
  static __device__ __forceinline__ float sum2(uint32_t u, float acc) {
    const bf16x2_t ones = {(__bf16)1.0f, (__bf16)1.0f};
    return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2_t, u), ones, acc, false);
  }
  static __device__ __forceinline__ uint32_t finite2(uint32_t u) {
    return pack(__builtin_fmaxf(lo(u), kMaskedBias), __builtin_fmaxf(hi(u), kMaskedBias));
  }
  // Eight bf16 times an fp32 factor, rounded to nearest even.  The results feed MFMAs written as
  // assembly: the closing statement makes the values complete there and puts the two idle issue slots
  // behind the last vector-ALU write that an MFMA operand needs.
  static __device__ __forceinline__ half8_t scale8(half8_t x, float f) {
    const u32x4 w = __builtin_bit_cast(u32x4, x);
    u32x4 r;
#pragma unroll
    for (int e = 0; e < 4; ++e) {  // (one statement per word: two temporaries at a time)
      uint32_t t0, t1, o;
      asm volatile("v_lshlrev_b32 %0, 16, %3\n\tv_and_b32 %1, 0xffff0000, %3\n\tv_mul_f32 %0, %0, %4\n\tv_mul_f32 %1, %1, %4\n\t"
                   "v_cvt_pk_bf16_f32 %2, %0, %1"
                   : "=&v"(t0), "=&v"(t1), "=&v"(o) : "v"(w[e]), "v"(f));
      r[e] = o;
    }
    asm volatile("s_nop 1" : "+v"(r));
    return __builtin_bit_cast(half8_t, r);
  }
  // The same product kept to 16 bits: hi = the rounded product, lo = what the rounding dropped, itself
  // rounded.  An MFMA over hi plus one over lo gives the scores the precision of the fp16 path; used
  // where the factor is large enough for the 8-bit rounding of hi alone to show in the gradients.
  static __device__ __forceinline__ void scale8_hilo(half8_t x, float f, half8_t& hi8, half8_t& lo8) {
    const u32x4 w = __builtin_bit_cast(u32x4, x);
    u32x4 rh, rl;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float t0 = lo(w[e]) * f, t1 = hi(w[e]) * f;
      rh[e] = pack(t0, t1);
      rl[e] = pack(t0 - lo(rh[e]), t1 - hi(rh[e]));
    }
    asm volatile("s_nop 1" : "+v"(rh), "+v"(rl));
    hi8 = __builtin_bit_cast(half8_t, rh);
    lo8 = __builtin_bit_cast(half8_t, rl);
  }
  // A pair of the user's bf16 bias values -> fp16 pair of bias * log2(e), kept finite on both sides
  // (the bias tile enters the scores through fp16 MFMAs also when the tensors are bf16: fp16 holds the
  // product with three more bits than bf16 would)
  static __device__ __forceinline__ uint32_t bias_log2(uint32_t u) {
    const float a = __builtin_fminf(__builtin_fmaxf(lo(u) * kLog2e, kBiasFloorLog2), -kBiasFloorLog2);
    const float b = __builtin_fminf(__builtin_fmaxf(hi(u) * kLog2e, kBiasFloorLog2), -kBiasFloorLog2);
    return pack_rn(a, b);
  }
  static __device__ __forceinline__ float dot2(uint32_t a, uint32_t b, float acc) {
    return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2_t, a), __builtin_bit_cast(bf16x2_t, b), acc, false);
  }
  // The one-hot selectors are shared with the fp16 MFMAs that add the bias: fp16 1.0 = 0x3C00, which a
  // bf16 MFMA reads as 2^-7 exactly.  Sums taken through such a selector are scaled back by 128.
  static constexpr float kOneHotInv = 128.0f;
  // -delta as hi + lo in bf16: 17 significant bits at every magnitude.  (As split_2048's fp16 pair a delta below 2^-8 kept fewer, one near
  // 6e-8 none, and one beyond 1.3e8 was infinite: with dO of 6e-8 dK was off by 5 %, at D = 64 dQ and dBias, too.  At unit dO the
  // gradients' errors against 64 bits are the same, means of 96 inputs within 2e-5 of each other; so are the times.)
  static __device__ __forceinline__ uint32_t delta_pair(float c) {
    const uint32_t h = pack(c, 0.0f);
    return pack(lo(h), c - lo(h));
  }
  static constexpr uint32_t kDeltaOnes = 0x3F803F80u;
  static __device__ __forceinline__ uint32_t add2(uint32_t a, uint32_t b) { return pack(lo(a) + lo(b), hi(a) + hi(b)); }
};

// The bias as the hand-scheduled forward kernels take it, whatever the element type: an fp16 pair at or above
// kMaskedBias.  (bf16 biases beyond 65504 are held there: the general kernels take them as they are.)
template <class T>
__device__ __forceinline__ uint32_t fwd1_bias_pair(uint32_t u) {
  if constexpr (T::is_bf16) {
    // (in place, with one temporary: 128 of these run with the register file full)
    uint32_t t;
    asm volatile(
        "v_lshlrev_b32 %1, 16, %0\n\t"
        "v_and_b32 %0, 0xffff0000, %0\n\t"
        "v_max_f32 %1, %2, %1\n\t"
        "v_max_f32 %0, %2, %0\n\t"
        "v_min_f32 %1, %3, %1\n\t"
        "v_min_f32 %0, %3, %0\n\t"
        "v_cvt_pk_f16_f32 %0, %1, %0"
        : "+v"(u), "=&v"(t)
        : "s"(kMaskedBias), "s"(65504.0f));
    return u;
  } else {
    return finite_half2(u);
  }
}

// ---- dropout ---------------------------------------------------------------------------------------
// Counter-based random bytes: a function of (seed, row, query, key) alone, so that the forward and
// both backward kernels -- which walk the scores in different orders and layouts -- see the same mask,
// and so does a host-side restatement (tests).  One call gives the 8 keep bytes of a block of
// 2 queries x 4 keys: word (j & 1) holds query j, byte (k & 3) of it key k.  The generator is
// Threefry-2x32 (Salmon et al., "Parallel random numbers: as easy as 1, 2, 3") cut to 8 rounds, with
// the counter (row, (j/2) << 16 | k/4) and the key (seed_lo, seed_hi): add, rotate, xor only.
struct u32pair { uint32_t x, y; };
__device__ __forceinline__ uint32_t rotl32(uint32_t v, int r) { return __builtin_amdgcn_alignbit(v, v, 32 - r); }
__device__ __forceinline__ u32pair threefry2x32_8(uint32_t c0, uint32_t c1, uint32_t k0, uint32_t k1) {
  const uint32_t k2 = k0 ^ k1 ^ 0x1BD11BDAu;
  uint32_t x = c0 + k0, y = c1 + k1;
#define FTA_TF_ROUND(R) x += y; y = rotl32(y, R) ^ x;
  FTA_TF_ROUND(13) FTA_TF_ROUND(15) FTA_TF_ROUND(26) FTA_TF_ROUND(6)
  x += k1; y += k2 + 1u;
  FTA_TF_ROUND(17) FTA_TF_ROUND(29) FTA_TF_ROUND(16) FTA_TF_ROUND(24)
  x += k2; y += k0 + 2u;
#undef FTA_TF_ROUND
  return u32pair{x, y};
}
// The four keep bytes of query j, keys 4*(k/4) .. +3 of row `row` (= (b*H + h)*L1 + i).
template <class DP>
__device__ __forceinline__ uint32_t keep_bits(const DP& d, uint32_t row, int j, int k) {
  const u32pair r = threefry2x32_8(row, ((uint32_t)(j >> 1) << 16) | (uint32_t)(k >> 2), d.seed_lo, d.seed_hi);
  return (j & 1) ? r.y : r.x;
}
// Both words of the block of queries 2*(j/2), 2*(j/2)+1 and keys 4*(k/4) .. +3.
template <class DP>
__device__ __forceinline__ u32pair keep_block(const DP& d, uint32_t row, int j, int k) {
  return threefry2x32_8(row, ((uint32_t)(j >> 1) << 16) | (uint32_t)(k >> 2), d.seed_lo, d.seed_hi);
}
template <class DP>
__device__ __forceinline__ bool keep_byte(const DP& d, uint32_t bits, int n) { return ((bits >> (8 * n)) & 0xFFu) >= d.thresh; }
// The keep bytes of four consecutive keys as masks of the packed pairs (keys 0, 1) and (2, 3): a kept weight's 16 bits
// all ones.  The four bytes are compared at once: bit 7 of d says whether the low seven bits reach the threshold's,
// and the bytes' own bit 7 decides together with it (or for thresholds below 128, and from there on); v_perm
// spreads the bits of bytes 1 and 3 of either operand (selectors 8 to 11).  Nine instructions for four weights, where a
// compare and a select per weight take eight and keep the pair from being converted by one instruction.
struct KeepMasks {
  uint32_t low, either;
  template <class DP>
  __device__ __forceinline__ explicit KeepMasks(const DP& d) : low((d.thresh & 0x7Fu) * 0x01010101u), either(d.thresh < 128u ? ~0u : 0u) {}
  __device__ __forceinline__ u32pair pairs(uint32_t bits) const {
    const uint32_t d = (bits | 0x80808080u) - low, x = bits ^ d;
    const uint32_t g = (x & either) | (~x & d);
    return u32pair{__builtin_amdgcn_perm(g << 8, g, 0x08080A0Au), __builtin_amdgcn_perm(g << 8, g, 0x09090B0Bu)};
  }
};
// Neighbouring lanes need the same blocks: a value from another lane of the own group of four
// (v_mov_b32 with a DPP quad permutation; lane i of a quad reads lane (SEL >> 2i) & 3).
template <int SEL>
__device__ __forceinline__ uint32_t quad_perm(uint32_t v) {
  return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, SEL, 0xF, 0xF, true);
}
// Four lanes with a word each, transposed as a 4 x 4 matrix of bytes: byte s of the result is byte q of lane s's word,
// q and s counted inside the group of four.  Two exchanges, with the neighbour and with the other pair.
__device__ __forceinline__ uint32_t quad_transpose_bytes(uint32_t v, int lane) {
  const uint32_t a = __builtin_amdgcn_perm(v, quad_perm<0xB1>(v), (lane & 1) ? 0x07030501u : 0x02060004u);
  return __builtin_amdgcn_perm(a, quad_perm<0x4E>(a), (lane & 2) ? 0x07060302u : 0x01000504u);
}
// Transposed score layout (the forward and the dQ kernel: a lane owns one query and, per tile, four
// groups of four keys: kfirst + 8g .. +3, g = 0..3).  The two lanes of a query pair (adjacent lanes:
// query and lane have the same parity) need the same four blocks, each its own word of them; each
// computes two blocks and hands the partner's words over: kb[g] = the keep bytes of group g.
template <class DP>
__device__ __forceinline__ void keep_bits4_shared(const DP& d, uint32_t row, int j, int kfirst, uint32_t (&kb)[4]) {
  const bool odd = (j & 1) != 0;
  uint32_t mine[2], got[2];
#pragma unroll
  for (int c = 0; c < 2; ++c) {
    const u32pair blk = keep_block(d, row, j, kfirst + 8 * (c + (odd ? 2 : 0)));  // even lane: groups 0, 1; odd lane: 2, 3
    mine[c] = odd ? blk.y : blk.x;
    got[c] = quad_perm<0xB1>(odd ? blk.x : blk.y);  // lanes 0 <-> 1, 2 <-> 3: the partner's block, this lane's word
  }
  kb[0] = odd ? got[0] : mine[0];
  kb[1] = odd ? got[1] : mine[1];
  kb[2] = odd ? mine[0] : got[0];
  kb[3] = odd ? mine[1] : got[1];
}

// ---- LDS tiles -----------------------------------------------------------------------------------
// A staged tile holds rows of D halfs, unpadded (row r starts at r*D), with the 16-byte chunks of
// a row XOR-swizzled: chunk c of row r sits in slot c ^ f(r), f(r) = (r>>2)&3 for D=32 and the three
// bits of (r>>1)&7 in reverse order for D=64.  With that, the 16 lanes of one LDS access phase that read
// the same chunk of 16 consecutive rows (MFMA operand reads) fall into 16 different 16-byte bank groups,
// and so do the 32 lanes of a transposing read, which take 8 bytes each from four consecutive rows
// (D=64: rows r and r+2 are 256 bytes = all 64 banks apart, so f must move them by four chunks: the
// plain (r>>1)&7 left them on the same banks, a two-way conflict on every such read).
template <int D>
__device__ __forceinline__ int swz_slot(int row, int chunk) {
  const int x = (row >> 1) & 7;
  return (D == 32) ? (chunk ^ ((row >> 2) & 3)) : (chunk ^ (((x & 1) << 2) | (x & 2) | (x >> 2)));
}
template <int D>
__device__ __forceinline__ int swz_off(int row, int chunk) {  // offset in halfs
  return row * D + (swz_slot<D>(row, chunk) << 3);
}

// The staged tiles are filled by asynchronous 16-byte-per-lane copies global -> LDS that do not pass
// through registers (global_load_lds_dwordx4: dma16s, dma16s_at below).  The LDS destination is
// wave-uniform: lane l writes lds_byte_addr + 16*l.  Completion is tracked by vmcnt; the compiler does
// not see these loads, so callers wait with wait_vmem_all() before the barrier that publishes the
// tile.  (A copy may not read M0 in the issue slot right after the scalar instruction that wrote it:
// one idle slot.)
__device__ __forceinline__ void wait_vmem_all() { __builtin_amdgcn_s_waitcnt(0x0F70); }  // vmcnt(0) only
// Waits until at most n vector-memory operations of this wave are outstanding (they retire in
// order, so everything but the n most recent ones has landed).  n is wave-uniform; s_waitcnt takes
// an immediate, hence the switch.  Values above 12 fall back to fewer outstanding (always safe).
__device__ __forceinline__ void wait_vmem_leq(int n) {
  switch (n) {
    case 0: __builtin_amdgcn_s_waitcnt(0x0F70); break;
    case 1: __builtin_amdgcn_s_waitcnt(0x0F71); break;
    case 2: __builtin_amdgcn_s_waitcnt(0x0F72); break;
    case 3: __builtin_amdgcn_s_waitcnt(0x0F73); break;
    case 4: __builtin_amdgcn_s_waitcnt(0x0F74); break;
    case 5: __builtin_amdgcn_s_waitcnt(0x0F75); break;
    case 6: __builtin_amdgcn_s_waitcnt(0x0F76); break;
    case 7: __builtin_amdgcn_s_waitcnt(0x0F77); break;
    case 8: __builtin_amdgcn_s_waitcnt(0x0F78); break;
    case 9: __builtin_amdgcn_s_waitcnt(0x0F79); break;
    case 10: __builtin_amdgcn_s_waitcnt(0x0F7A); break;
    case 11: __builtin_amdgcn_s_waitcnt(0x0F7B); break;
    default: __builtin_amdgcn_s_waitcnt(0x0F7C); break;
  }
}

// Cheaper form for hot loops: rounds n down to 12, 8, 4 or 0 (fewer outstanding is always safe).
__device__ __forceinline__ void wait_vmem_coarse(int n) {
  if (n >= 8) {
    if (n >= 12) __builtin_amdgcn_s_waitcnt(0x0F7C);
    else __builtin_amdgcn_s_waitcnt(0x0F78);
  } else {
    if (n >= 4) __builtin_amdgcn_s_waitcnt(0x0F74);
    else __builtin_amdgcn_s_waitcnt(0x0F70);
  }
}

__device__ __forceinline__ uint32_t lds_addr_of(const void* p) {
  return (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const char*)p;
}

// Issues the DMA copies of one tile: `rows` rows of D halfs, row `r` of the tile taken from
// gbase + grow(r)*gstride.  The 64*k-th..(64*k+63)-th chunks of the tile form one wave
// instruction; wave-instructions are dealt round-robin to the `nwaves` waves.
// Same copy with the global address split into a wave-uniform 64-bit base (SGPR pair) and a
// per-lane 32-bit byte offset: no vector ALU work at issue time.
__device__ __forceinline__ void dma16s(uint32_t voff, const void* sbase, uint32_t lds_byte_addr) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(voff), "s"(sbase), "s"(lds_byte_addr) : "memory", "m0");
}

// The same with the LDS address given as a scalar base plus a compile-time offset: the sum goes
// straight into M0 (one scalar instruction instead of two).
template <uint32_t IMM>
__device__ __forceinline__ void dma16s_at(uint32_t voff, const void* sbase, uint32_t lds_base) {
  if constexpr (IMM == 0)
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(voff), "s"(sbase), "s"(lds_base) : "memory", "m0");
  else
    asm volatile("s_add_i32 m0, %2, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(voff), "s"(sbase), "s"(lds_base), "n"(IMM) : "memory", "m0", "scc");
}

// Forces a pointer whose value is the same in every lane into scalar registers, for the copies and
// loads below that take their base address from a scalar register pair.  A vector-memory instruction
// may not read a scalar register within 5 issue slots of a vector-ALU instruction writing it (it
// would see the old value), and the compiler's hazard pass does not look inside asm blocks: the
// result therefore comes out of a scalar move, which may follow v_readfirstlane directly and after
// which a memory instruction may read at once.
__device__ __forceinline__ const void* uniform_ptr(const void* p) {
  const uint64_t v = (uint64_t)(uintptr_t)p;
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v);
  const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
  const uint64_t u = ((uint64_t)hi << 32) | lo;
  uint64_t r;
  asm("s_mov_b64 %0, %1" : "=s"(r) : "s"(u));
  return (const void*)(uintptr_t)r;
}

// Copy plan of one staged tile, computed once per thread.  A tile has `rows` rows of D halfs;
// tile row r maps to global row (r / T) * W + r % T of a window that the caller positions with a
// wave-uniform base pointer per stage (T rows per slab in the tile, W rows between slabs in
// memory).  The 64*k-th .. (64*k+63)-th 16-byte chunks of the tile form one wave instruction;
// wave-instructions are dealt round-robin to the waves, so wave w issues copies w, w + nwaves, ...
template <int MAXU>
struct DmaPlan {
  uint32_t goff[MAXU];  // per-lane byte offset from the stage's base pointer
  int n;                // copies this wave issues per tile (wave-uniform, <= MAXU)
  uint32_t lofs;        // LDS byte offset of this wave's first copy inside the tile
  uint32_t lstep;       // LDS byte distance between this wave's consecutive copies
};

template <int D, int MAXU>
__device__ __forceinline__ void dma_plan(DmaPlan<MAXU>& pl, int rows, int T, int W, int64_t gstride, int wave, int lane,
                                         int nwaves) {
  constexpr int CPR = D / 8;
  const int ninstr = rows * CPR / 64;
  pl.n = (ninstr > wave) ? (ninstr - wave + nwaves - 1) / nwaves : 0;
  pl.lofs = __builtin_amdgcn_readfirstlane((uint32_t)wave * 1024u);  // wave-uniform: keep it scalar
  pl.lstep = (uint32_t)nwaves * 1024u;
  pl.n = __builtin_amdgcn_readfirstlane(pl.n);
#pragma unroll
  for (int u = 0; u < MAXU; ++u) {
    const int p = (wave + u * nwaves) * 64 + lane;
    const int row = p / CPR, slot = p % CPR;
    const int chunk = swz_slot<D>(row, slot);  // XOR is its own inverse
    const int64_t grow = (int64_t)(row / T) * W + row % T;
    pl.goff[u] = (uint32_t)((grow * gstride + chunk * 8) * 2);
  }
}

// How many of the 1 KB copies that a tile of `rows` rows of D halfs takes fall to this wave.
__device__ __forceinline__ int dma_rows_count(int rows, int D, int wave, int nwaves) {
  const int ninstr = rows * (D / 8) / 64;
  return (ninstr > wave) ? (ninstr - wave + nwaves - 1) / nwaves : 0;
}

template <int MAXU>
__device__ __forceinline__ void dma_issue(const DmaPlan<MAXU>& pl, const void* sbase, uint32_t lds_tile_addr) {
#pragma unroll
  for (int u = 0; u < MAXU; ++u)
    if (u < pl.n) dma16s(pl.goff[u], sbase, lds_tile_addr + pl.lofs + (uint32_t)u * pl.lstep);
}

// The same tile copy for a tile whose last rows lie beyond the tensor's last row (L2 is not a multiple
// of the tile): tile row r is taken from global row min((r / T) * W + r % T + first, last_valid) of the
// window at `rowbase`, so nothing outside the tensor is read (the duplicated rows belong to keys or
// queries that are masked or never stored).  Offsets are computed on the fly; every wave issues the
// same copies, to the same LDS places, as dma_issue() does with a DmaPlan of the same geometry.
template <int D>
__device__ __forceinline__ void dma_tile_clamped(const void* rowbase, int64_t gstride, int rows, int T, int W, int first,
                                                 int last_valid, uint32_t lds_tile_addr, int wave, int lane, int nwaves) {
  constexpr int CPR = D / 8;
  const int ninstr = rows * CPR / 64;
  const void* sb = uniform_ptr(rowbase);
  for (int j = wave; j < ninstr; j += nwaves) {
    const int pidx = j * 64 + lane;
    const int row = pidx / CPR, slot = pidx % CPR;
    int g = (row / T) * W + row % T + first;
    g = g < last_valid ? g : last_valid;
    const uint32_t voff = (uint32_t)(((int64_t)g * gstride + swz_slot<D>(row, slot) * 8) * 2);
    dma16s(voff, sb, __builtin_amdgcn_readfirstlane(lds_tile_addr + (uint32_t)j * 1024u));
  }
}

// Four consecutive bias entries bias[j][k .. k+3] (k a multiple of 4) as two packed pairs; keys at or
// beyond L2 (the row's true length) read as any value (beyond_row()), queries beyond it read the last query's row.  One
// 8-byte load where the four entries exist and sit on an 8-byte boundary; entry by entry at the end of
// a row whose length is not a multiple of 4 and in rows that start on a 2-byte boundary (such a
// length, or a strided view).
__device__ __forceinline__ u32x2 load_bias4(const half_t* bias_bh, int64_t jstride, int j, int k, int L2) {
  const int jj = j < L2 ? j : L2 - 1;
  if (k >= L2) return u32x2{0u, 0u};
  const half_t* src = bias_bh + (int64_t)jj * jstride + k;
  if (k + 4 <= L2 && (reinterpret_cast<uintptr_t>(src) & 7u) == 0) return *reinterpret_cast<const u32x2*>(src);
  const uint16_t* s16 = reinterpret_cast<const uint16_t*>(src);
  uint32_t e[4];
#pragma unroll
  for (int n = 0; n < 4; ++n) e[n] = (k + n < L2) ? (uint32_t)s16[n] : 0u;
  return u32x2{e[0] | (e[1] << 16), e[2] | (e[3] << 16)};
}
// The pairs of keys k .. k+3 with those at or beyond L2 put to `beyond2` (see kMaskedBias).
__device__ __forceinline__ u32x2 beyond_row(u32x2 v, int k, int L2, uint32_t beyond2) {
  const int left = L2 - k;  // real ones
  return u32x2{left <= 0 ? beyond2 : left == 1 ? (v[0] & 0xFFFFu) | (beyond2 << 16) : v[0],
               left <= 2 ? beyond2 : left == 3 ? (v[1] & 0xFFFFu) | (beyond2 << 16) : v[1]};
}

// Eight consecutive bias entries from key k of a row, as whole-row loads want them: entries k .. k+7 of a row that holds
// them, any other piece (TAIL) as the row's last eight entries, which bias_piece_fix() shifts into place, with `beyond2` for
// the keys at or beyond L2.  Any 2-byte boundary.  (Rows of fewer than eight keys are read entry by entry.)
template <bool TAIL>
__device__ __forceinline__ u32x4 bias_piece_load(const half_t* row, int k, int L2, bool short_rows) {
  u32x4 v;
  if constexpr (!TAIL) {
    v = *reinterpret_cast<const u32x4*>(row + k);
  } else if (!short_rows || L2 >= 8) {
    __builtin_memcpy(&v, row + (k + 8 <= L2 ? k : L2 - 8), 16);
  } else {
    uint32_t e[8];
#pragma unroll
    for (int n = 0; n < 8; ++n) e[n] = k + n < L2 ? (uint32_t)reinterpret_cast<const uint16_t*>(row)[k + n] : 0u;
    v = u32x4{e[0] | (e[1] << 16), e[2] | (e[3] << 16), e[4] | (e[5] << 16), e[6] | (e[7] << 16)};
  }
  return v;
}
__device__ __forceinline__ u32x4 bias_piece_fix(u32x4 v, int k, int L2, uint32_t beyond2, bool short_rows) {
  if (short_rows && L2 < 8) {
#pragma unroll
    for (int n = 0; n < 4; ++n) v[n] = k + 2 * n >= L2 ? beyond2 : k + 2 * n + 1 >= L2 ? (v[n] & 0xFFFFu) | (beyond2 << 16) : v[n];
    return v;
  }
  const int sh = k + 8 <= L2 ? 0 : (k - (L2 - 8) < 8 ? k - (L2 - 8) : 8);  // entries to drop at the front
  if (sh & 4) v = u32x4{v[2], v[3], beyond2, beyond2};
  if (sh & 2) v = u32x4{v[1], v[2], v[3], beyond2};
  if (sh & 1)
    v = u32x4{__builtin_amdgcn_alignbit(v[1], v[0], 16), __builtin_amdgcn_alignbit(v[2], v[1], 16), __builtin_amdgcn_alignbit(v[3], v[2], 16),
              __builtin_amdgcn_alignbit(beyond2, v[3], 16)};
  if (sh & 8) v = u32x4{beyond2, beyond2, beyond2, beyond2};
  return v;
}

// The stationary bias of a wave: 32 queries from q0 against NC chunks of 32*CT keys (chunk c from key first_key(c)),
// passed through `conv` and handed to `sink(tile, group, pair)` in the S^T accumulator layout (keys
// 8*group + 4*hh + 0..3 of the tile's 32, of query l%32, as two packed pairs; tile c*CT + t).  Loaded that way, 8 bytes per lane, an instruction touches 32 rows and every
// 128-byte line is asked for by eight of them, more lines than the L1 holds between two: at 512 keys the set-up of a
// workgroup took 16 us.  Instead four or eight lanes load a row's keys as one piece of a line, all of them in flight at
// once, and the pieces change lanes through 2 or 4 KB (CT) of LDS that belong to the wave (no barrier: a wave's LDS operations are
// executed in order).
// TAIL: rows of L2 keys that may end inside the tile (keys beyond it come out as `beyond2`, queries beyond it as the last
// query's row), on any 2-byte boundary; SHORT: of fewer than eight keys, too.
template <int NC, int CT, bool TAIL, bool SHORT, class Key, class Conv, class Sink>
__device__ __forceinline__ void load_bias_tiles(const half_t* bias_bh, int64_t jstride, int q0, int L2, uint32_t beyond2, char* lds, int lane,
                                                Key&& first_key, Conv&& conv, Sink&& sink) {
  static_assert(CT == 1 || CT == 2, "chunks of 32 or 64 keys");
  constexpr int PR = 4 * CT, RI = 64 / PR, NI = 32 / RI;  // pieces per row, rows per instruction, instructions per chunk
  const int rowi = lane / PR, piece = lane % PR, l32 = lane & 31, hh = lane >> 5;
  auto slot = [](int row, int pc) { return row * (16 * PR) + ((pc ^ (CT == 2 ? row & 7 : (row >> 1) & 3)) << 4); };
  u32x4 raw[NC][NI];
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    const int j = q0 + RI * i + rowi;
    const half_t* row = bias_bh + (int64_t)(TAIL ? (j < L2 ? j : L2 - 1) : j) * jstride;
#pragma unroll
    for (int c = 0; c < NC; ++c) raw[c][i] = bias_piece_load<TAIL>(row, first_key(c) + 8 * piece, L2, SHORT);
  }
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    // (TAIL: converted before the pieces of the row's end are put in place, which `conv` would not leave as they are;
    // else on the way out of LDS)
    if constexpr (TAIL) {
#pragma unroll
      for (int i = 0; i < NI; ++i) raw[c][i] = u32x4{conv(raw[c][i][0]), conv(raw[c][i][1]), conv(raw[c][i][2]), conv(raw[c][i][3])};
      if (first_key(c) + 32 * CT > L2)  // the row ends in this chunk, or before it
#pragma unroll
        for (int i = 0; i < NI; ++i) raw[c][i] = bias_piece_fix(raw[c][i], first_key(c) + 8 * piece, L2, beyond2, SHORT);
    }
#pragma unroll
    for (int i = 0; i < NI; ++i) *reinterpret_cast<u32x4*>(lds + slot(RI * i + rowi, piece)) = raw[c][i];
#pragma unroll
    for (int t = 0; t < CT; ++t)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const u32x2 v = *reinterpret_cast<const u32x2*>(lds + slot(l32, 4 * t + g) + 8 * hh);
        if constexpr (TAIL) sink(c * CT + t, g, v);
        else sink(c * CT + t, g, u32x2{conv(v[0]), conv(v[1])});
      }
  }
}

// Per-lane LDS offsets (in halfs) of the MFMA operand reads inside a staged tile.  The swizzle
// term depends only on the lane as long as tiles start at a multiple of 32 rows (16 for the
// transposed reads), so it is folded into these offsets once; a read then costs one address
// register plus an immediate for the tile position.
template <int D>
struct FragOffsets {
  int a[D / 16];     // chunk 2*ks + hh of row l%32 of a 32-row tile (operand with contiguous contraction)
  int t[D / 32][2];  // transposed reads: column block dt, rows 4*hh + r (+8) of a 16-row block
  __device__ __forceinline__ void init(int lane) {
    const int l32 = lane & 31, hh = lane >> 5;
#pragma unroll
    for (int ks = 0; ks < D / 16; ++ks) a[ks] = swz_off<D>(l32, 2 * ks + hh);
    const int g16 = lane >> 4, s16 = lane & 15;
    const int r = s16 >> 2, c = s16 & 3;
#pragma unroll
    for (int dt = 0; dt < D / 32; ++dt) {
      const int chunk = 4 * dt + 2 * (g16 & 1) + (c >> 1);
      t[dt][0] = swz_off<D>(4 * hh + r, chunk) + 4 * (c & 1);
      t[dt][1] = swz_off<D>(4 * hh + r + 8, chunk) + 4 * (c & 1);
    }
  }
};

// MFMA A/B operand whose contraction index is contiguous in memory: 8 halfs (chunk 2*ks + hh) of
// row tile_row0 + l%32; tile_row0 must be a multiple of 32.
template <int D>
__device__ __forceinline__ half8_t lds_frag(const half_t* tile, int tile_row0, const FragOffsets<D>& fo, int ks) {
  return *reinterpret_cast<const half8_t*>(tile + tile_row0 * D + fo.a[ks]);
}

// Transposing LDS read (ds_read_b64_tr_b16).  Within each group of 16 lanes, lane s = 4*r + c
// passes the address of 4 consecutive halfs; lane i of the group receives element i%4 of the
// chunks given by lanes 4*0 + i/4, 4*1 + i/4, 4*2 + i/4, 4*3 + i/4.  With lane (r, c) pointing at
// M[row0 + r][col0 + 4c .. +3], lane i ends up with M[row0 + 0..3][col0 + i]: a column of 4.
__device__ __forceinline__ u32x2 lds_read_tr4(const half_t* p) {
  fp16x4_b v = __builtin_amdgcn_ds_read_tr16_b64_v4f16((lds_fp16x4_b*)(p));
  return __builtin_bit_cast(u32x2, v);
}

// MFMA A operand (32 rows x 16 contraction) taken as the TRANSPOSE of a staged tile
// M[contraction][column]: A[row = column 32*dt + l%32][slot e] = M[rowbase + (e/4)*8 + 4*hh + e%4][..],
// i.e. the contraction slots follow the accumulator-row order described at the top.  rowbase must
// be a multiple of 16.
template <int D>
__device__ __forceinline__ half8_t lds_frag_t(const half_t* tile, int rowbase, const FragOffsets<D>& fo, int dt) {
  u32x2 lo = lds_read_tr4(tile + rowbase * D + fo.t[dt][0]);
  u32x2 hi = lds_read_tr4(tile + rowbase * D + fo.t[dt][1]);
  u32x4 v = {lo[0], lo[1], hi[0], hi[1]};
  return as_half8(v);
}

// XCD-aware decode: hardware deals consecutive workgroup ids round-robin over the 8 dies, so
// id n lands on die n%8.  Re-number so that logically consecutive workgroups (which share K/V
// rows and the bias in that die's L2) sit on the same die, also where the count is no multiple of 8 (the first dies
// then have one more).
__device__ __forceinline__ int xcd_remap(int n, int total) {
  const int die = n % kXcds, each = total / kXcds, more = total % kXcds;
  return die * each + min(die, more) + n / kXcds;
}

// What a workgroup works on: `group` of queries (or keys) of one (b,h), a chunk of L1 rows.  Logically consecutive
// workgroups take the groups of a chunk (they read the same rows), then the chunks of a (b,h) (the same bias); where
// the heads of a row are interleaved in memory (`head_inner`: a projection's (.., H*D) layout) the heads come
// before the chunks, since a 128-byte line then holds two heads' rows and would else be fetched by two dies.
struct WorkId { int group, chunk, b, h; };
__device__ __forceinline__ WorkId work_id(int ngroups, int nchunks, int H, int head_inner) {
  int lid = xcd_remap(blockIdx.x, gridDim.x);
  WorkId w;
  w.group = lid % ngroups;
  lid /= ngroups;
  if (head_inner) {
    w.h = lid % H;
    lid /= H;
    w.chunk = lid % nchunks;
    w.b = lid / nchunks;
  } else {
    w.chunk = lid % nchunks;
    lid /= nchunks;
    w.h = lid % H;
    w.b = lid / H;
  }
  return w;
}

}  // namespace fta
