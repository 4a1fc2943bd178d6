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
// and everything that can be formed from a row in registers is: the normalised row never goes to memory (it
// is formed again where the backward needs it), nor do gate * o or the five input gradients before they
// are summed.  The row kernels (proj, out, dout, dx) let a wave own 32 pair rows: lane l holds row l % 32 as
// the B operands of its MFMAs (8 channels per 16-wide contraction step and lane half), so the layer-norm sums
// stay in a lane and its partner in the other half, and an accumulator tile (32 output channels x 32 rows) is
// written as two 16-byte pieces per lane.  The weights are the A operands: all of them in LDS in operand
// order, read with one conflict-free ds_read_b128 per contraction step, no barrier after they are loaded.
// Where they do not fit LDS (fp32: 264 KB) the proj kernel cuts them into column groups of workgroups and the
// dx kernel reads them from the cache in operand order.
//
// fp32 blocks run the fp32 matrix instructions (v_mfma_f32_32x32x2_f32): nothing is rounded to 16 bits
// that was not before (q, k, v, bias, o and their gradients).
//
// Measured, AlphaFold2's block (C 128, 4 heads of 32), bf16, against separate library calls: see the
// launch functions at the end of this file.
#include "fta_block.h"

#include "fta.h"

#include "fta_common.h"
#include "fta_kernels.h"

namespace fta {
namespace {

// ---- operand fragments: 8 consecutive contraction elements per lane -----------------------------------
template <bool F32> struct Frag;
template <> struct Frag<false> { u32x4 w; };
template <> struct Frag<true> { float v[8]; };
template <bool F32> struct Store { typedef uint16_t type; };
template <> struct Store<true> { typedef float type; };

template <class A>
__device__ __forceinline__ floatx16 mma(const Frag<false>& a, const Frag<false>& b, floatx16 c) {
  return A::mfma(as_half8(a.w), as_half8(b.w), c);
}
template <class A>
__device__ __forceinline__ floatx16 mma(const Frag<true>& a, const Frag<true>& b, floatx16 c) {
  // (element e of the two lane halves is one contraction pair: the same order for both operands)
#pragma unroll
  for (int e = 0; e < 8; ++e) c = __builtin_amdgcn_mfma_f32_32x32x2f32(a.v[e], b.v[e], c, 0, 0, 0);
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

__device__ __forceinline__ floatx16 zero16() {
  floatx16 v;
#pragma unroll
  for (int e = 0; e < 16; ++e) v[e] = 0.f;
  return v;
}

template <bool F32>
__device__ __forceinline__ float sigmoid(float x) {
  if constexpr (F32) return 1.0f / (1.0f + expf(-x));
  else return __builtin_amdgcn_rcpf(1.0f + exp2_fast(-kLog2e * x));
}

// 32 pair rows of one batch entry: which ones, and where this lane's row is.
struct RowBlock {
  int b;          // batch entry (wave-uniform)
  uint32_t p;     // this lane's row: i * L + j, the last one of the batch entry beyond the end
  bool valid;
  uint32_t i, j;
};
__device__ __forceinline__ RowBlock row_block(const BlockParams& p, int blk, int lane) {
  RowBlock r;
  r.b = blk / p.nper;
  const uint32_t p0 = (uint32_t)(blk - r.b * p.nper) * 32u + (uint32_t)(lane & 31);
  r.valid = p0 < (uint32_t)p.LL;
  r.p = r.valid ? p0 : (uint32_t)p.LL - 1u;
  r.i = r.p / (uint32_t)p.L;
  r.j = r.p - r.i * (uint32_t)p.L;
  return r;
}
__device__ __forceinline__ int64_t pair_off(const int64_t (&s)[3], const RowBlock& r) { return r.b * s[0] + r.i * s[1] + r.j * s[2]; }
// element of (b, h, i, j, d = 0) in a (B, H, L, L, D) tensor
__device__ __forceinline__ int64_t head_off(const BlockParams& p, const RowBlock& r, int h) {
  return (((int64_t)r.b * p.H + h) * p.LL + r.p) * p.D;
}

// Layer-norm statistics of this lane's row from its half of the row (C/16 fragments) and its partner's,
// in two passes over the registers, as mean and sum of squared deviations.
template <class A, bool F32, int KS>
__device__ __forceinline__ void row_stats(const Frag<F32> (&z)[KS], float eps, float& mean, float& rstd) {
  float s = 0.f;
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) {
    float x[8];
    unpack<A>(z[ks], x);
#pragma unroll
    for (int e = 0; e < 8; ++e) s += x[e];
  }
  mean = sum_both_halves(s) * (1.0f / (16 * KS));
  float v = 0.f;
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) {
    float x[8];
    unpack<A>(z[ks], x);
#pragma unroll
    for (int e = 0; e < 8; ++e) { const float d = x[e] - mean; v = __builtin_fmaf(d, d, v); }
  }
  v = sum_both_halves(v) * (1.0f / (16 * KS));
  rstd = 1.0f / __builtin_sqrtf(v + eps);
}

// ---- forward: layer norm and projections --------------------------------------------------------------
// Output tiles of 32 channels: 4*HD/32 of q, k, v, gate, then the heads of the bias (padded to 32).
template <class A, bool F32, int C>
__global__ void __launch_bounds__(512) blk_proj_kernel(BlockParams p) {
  constexpr int KS = C / 16;
  extern __shared__ char smem[];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, l32 = lane & 31, hh = lane >> 5;
  const int nw = blockDim.x >> 6;
  const int nt4 = 4 * p.HD / 32, ntiles = nt4 + (p.H + 31) / 32;
  const int per = (ntiles + gridDim.y - 1) / gridDim.y;  // tiles of this workgroup's column range
  const int t0 = blockIdx.y * per, t1 = min(ntiles, t0 + per);
  // weights -> LDS in operand order; layer-norm parameters and gate biases as fp32 behind them
  float* gam = reinterpret_cast<float*>(smem + (size_t)per * KS * kFragBytes<F32>);
  float* bet = gam + C;
  float* bgs = bet + C;
  for (int idx = wave; idx < (t1 - t0) * KS; idx += nw) {
    const int t = t0 + idx / KS, ks = idx % KS;
    const int n = t * 32 + l32;
    Frag<F32> f = frag_zero<F32>();
    if (t < nt4) {
      const int s = n / p.HD;
      f = load8<F32>(p.w[s], (int64_t)(n - s * p.HD) * C + ks * 16 + hh * 8);
    } else if (n - 32 * nt4 < p.H) {
      f = load8<F32>(p.wb, (int64_t)(n - 32 * nt4) * C + ks * 16 + hh * 8);
    }
    frag_write<F32>(smem, idx, lane, f);
  }
  for (int c = tid; c < C; c += blockDim.x) {
    gam[c] = load1<A, F32>(p.gamma, c);
    bet[c] = load1<A, F32>(p.beta, c);
  }
  for (int c = tid; c < p.HD; c += blockDim.x) bgs[c] = p.bg != nullptr ? load1<A, F32>(p.bg, c) : 0.f;
  __syncthreads();

  const int nitems = p.B * p.nper * p.cg, step = (int)gridDim.x * nw;
  int item = __builtin_amdgcn_readfirstlane((int)blockIdx.x * nw + wave);
  if (item >= nitems) return;
  Frag<F32> z[KS];
  RowBlock rb = row_block(p, item / p.cg, lane);
  auto fetch = [&]() {
    const int64_t zo = pair_off(p.zs, rb) + hh * 8;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) z[ks] = load8<F32>(p.z, zo + ks * 16);
  };
  fetch();
  for (; item < nitems; item += step) {
    const RowBlock cur = rb;
    const int g = item % p.cg;
    float mean, rstd;
    row_stats<A, F32, KS>(z, p.eps, mean, rstd);
    Frag<F32> x[KS];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      float v[8];
      unpack<A>(z[ks], v);
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const int c = ks * 16 + hh * 8 + e;
        v[e] = __builtin_fmaf((v[e] - mean) * rstd, gam[c], bet[c]);
      }
      pack<A>(v, x[ks]);
    }
    if (item + step < nitems) {  // the next row block's loads fly during this one's products
      rb = row_block(p, (item + step) / p.cg, lane);
      fetch();
    }
    for (int t = t0 + g; t < t1; t += p.cg) {
      floatx16 acc = zero16();
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) acc = mma<A>(frag_read<F32>(smem, (t - t0) * KS + ks, lane), x[ks], acc);
      if (t < nt4) {
        const int n = t * 32, s = n / p.HD, col = n - s * p.HD, h = col / p.D;
        const int64_t off = head_off(p, cur, h) + (col - h * p.D) + hh * 8;
        float y[2][8];
        rows8(acc, y);
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          if (s == 3) {
#pragma unroll
            for (int e = 0; e < 8; ++e) y[u][e] = sigmoid<F32>(y[u][e] + bgs[col + 16 * u + 8 * hh + e]);
            Frag<F32> f;
            pack<A>(y[u], f);
            if (cur.valid) store8<F32>(p.gate, off + 16 * u, f);
          } else {
            Frag<false> f;
            pack<A>(y[u], f);
            if (cur.valid) store8<false>(p.qkv[s], off + 16 * u, f);
          }
        }
      } else {
        float add = 0.f;  // 0 marks padded key positions, which no query may attend to
        if (p.mask != nullptr) add = (load1<A, F32>(p.mask, (int64_t)cur.b * p.L + cur.j) - 1.0f) * 30000.0f;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int h = (t - nt4) * 32 + 8 * (r / 4) + 4 * hh + r % 4;
          if (h < p.H && cur.valid) store1<A, false>(p.bias, ((int64_t)cur.b * p.H + h) * p.LL + cur.p, acc[r] + add);
        }
      }
    }
  }
}

// ---- forward: gating and output projection ------------------------------------------------------------
template <class A, bool F32, int C, int HD>
__global__ void __launch_bounds__(512) blk_out_kernel(BlockParams p) {
  constexpr int KS = HD / 16, NT = C / 32;
  extern __shared__ char smem[];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, l32 = lane & 31, hh = lane >> 5;
  const int nw = blockDim.x >> 6;
  float* bos = reinterpret_cast<float*>(smem + (size_t)NT * KS * kFragBytes<F32>);
  for (int idx = wave; idx < NT * KS; idx += nw)
    frag_write<F32>(smem, idx, lane, load8<F32>(p.wo, (int64_t)((idx / KS) * 32 + l32) * HD + (idx % KS) * 16 + hh * 8));
  for (int c = tid; c < C; c += blockDim.x) bos[c] = p.bo != nullptr ? load1<A, F32>(p.bo, c) : 0.f;
  __syncthreads();

  const int nitems = p.B * p.nper * p.cg, step = (int)gridDim.x * nw;
  int item = __builtin_amdgcn_readfirstlane((int)blockIdx.x * nw + wave);
  if (item >= nitems) return;
  Frag<F32> gt[KS];
  Frag<false> o[KS];
  RowBlock rb = row_block(p, item / p.cg, lane);
  auto fetch = [&]() {
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const int h = ks * 16 / p.D;
      const int64_t off = head_off(p, rb, h) + (ks * 16 - h * p.D) + hh * 8;
      gt[ks] = load8<F32>(p.gate, off);
      o[ks] = load8<false>(p.o, off);
    }
  };
  fetch();
  for (; item < nitems; item += step) {
    const RowBlock cur = rb;
    const int g = item % p.cg;
    Frag<F32> x[KS];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      float a[8], b[8];
      unpack<A>(gt[ks], a);
      unpack<A>(o[ks], b);
#pragma unroll
      for (int e = 0; e < 8; ++e) a[e] *= b[e];
      pack<A>(a, x[ks]);
    }
    if (item + step < nitems) {
      rb = row_block(p, (item + step) / p.cg, lane);
      fetch();
    }
    const int64_t oo = pair_off(p.outs, cur) + hh * 8;
    for (int t = g; t < NT; t += p.cg) {
      floatx16 acc = zero16();
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) acc = mma<A>(frag_read<F32>(smem, t * KS + ks, lane), x[ks], acc);
      float y[2][8];
      rows8(acc, y);
#pragma unroll
      for (int u = 0; u < 2; ++u) {
#pragma unroll
        for (int e = 0; e < 8; ++e) y[u][e] += bos[t * 32 + 16 * u + 8 * hh + e];
        Frag<F32> f;
        pack<A>(y[u], f);
        if (cur.valid) store8<F32>(p.out, oo + t * 32 + 16 * u, f);
      }
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
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, l32 = lane & 31, hh = lane >> 5;
  const int nw = blockDim.x >> 6;
  if ((int)blockIdx.x >= p.nwg) {
    const int ksall = 4 * HD / 16 + (p.H + 15) / 16;
    const int npack = (int)gridDim.x - p.nwg;
    for (int idx = ((int)blockIdx.x - p.nwg) * nw + wave; idx < (C / 32) * ksall; idx += npack * nw) {
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
  for (int idx = wave; idx < NT * KS; idx += nw) {
    float v[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = load1<A, F32>(p.wo, (int64_t)((idx % KS) * 16 + hh * 8 + e) * HD + (idx / KS) * 32 + l32);
    Frag<F32> f;
    pack<A>(v, f);
    frag_write<F32>(smem, idx, lane, f);
  }
  __syncthreads();

  const int nitems = p.B * p.nper * p.cg, step = p.nwg * nw;
  int item = __builtin_amdgcn_readfirstlane((int)blockIdx.x * nw + wave);
  if (item >= nitems) return;
  Frag<F32> x[KS];
  RowBlock rb = row_block(p, item / p.cg, lane);
  auto fetch = [&]() {
    const int64_t so = pair_off(p.douts, rb) + hh * 8;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) x[ks] = load8<F32>(p.dout, so + ks * 16);
  };
  fetch();
  for (; item < nitems; item += step) {
    const RowBlock cur = rb;
    const int g = item % p.cg;
    for (int t = g; t < NT; t += p.cg) {
      const int h = t * 32 / p.D;
      const int64_t off = head_off(p, cur, h) + (t * 32 - h * p.D) + hh * 8;
      Frag<F32> gt[2];
      Frag<false> o[2];
#pragma unroll
      for (int u = 0; u < 2; ++u) { gt[u] = load8<F32>(p.gate, off + 16 * u); o[u] = load8<false>(p.o, off + 16 * u); }
      floatx16 acc = zero16();
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) acc = mma<A>(frag_read<F32>(smem, t * KS + ks, lane), x[ks], acc);
      float y[2][8];
      rows8(acc, y);
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
        Frag<false> fo;
        Frag<F32> fd;
        pack<A>(y[u], fo);
        pack<A>(d, fd);
        if (cur.valid) {
          store8<false>(p.dog, off + 16 * u, fo);
          store8<F32>(p.dgp, off + 16 * u, fd);
        }
      }
    }
    if (item + step < nitems) {
      rb = row_block(p, (item + step) / p.cg, lane);
      fetch();
    }
  }
}

// ---- backward: input gradient and layer norm ----------------------------------------------------------
template <class A, bool F32, int C, int HD, bool WLDS>
__global__ void __launch_bounds__(512) blk_dx_kernel(BlockParams p) {
  constexpr int KS = C / 16, NT = C / 32, KH = HD / 16;
  extern __shared__ char smem[];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, hh = lane >> 5;
  const int nw = blockDim.x >> 6;
  const int kb = (p.H + 15) / 16, ksall = 4 * KH + kb;
  float* gam = reinterpret_cast<float*>(smem + (WLDS ? (size_t)NT * ksall * kFragBytes<F32> : 0));
  const char* wt = WLDS ? smem : static_cast<const char*>(p.wt);
  if (WLDS)
    for (int idx = tid; idx < NT * ksall * kFragBytes<F32> / 16; idx += blockDim.x)
      reinterpret_cast<u32x4*>(smem)[idx] = static_cast<const u32x4*>(p.wt)[idx];
  for (int c = tid; c < C; c += blockDim.x) gam[c] = load1<A, F32>(p.gamma, c);
  __syncthreads();

  const int nitems = p.B * p.nper, step = (int)gridDim.x * nw;
  for (int item = __builtin_amdgcn_readfirstlane((int)blockIdx.x * nw + wave); item < nitems; item += step) {
    const RowBlock cur = row_block(p, item, lane);
    Frag<F32> z[KS];
    const int64_t zo = pair_off(p.zs, cur) + hh * 8;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) z[ks] = load8<F32>(p.z, zo + ks * 16);
    floatx16 acc[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) acc[t] = zero16();
    auto step16 = [&](const Frag<F32>& d, int ks) {
#pragma unroll
      for (int t = 0; t < NT; ++t) acc[t] = mma<A>(frag_read<F32>(wt, t * ksall + ks, lane), d, acc[t]);
    };
    for (int s = 0; s < 3; ++s) {
      Frag<false> d[KH];
#pragma unroll
      for (int k = 0; k < KH; ++k) {
        const int h = k * 16 / p.D;
        d[k] = load8<false>(p.dqkv[s], head_off(p, cur, h) + (k * 16 - h * p.D) + hh * 8);
      }
#pragma unroll
      for (int k = 0; k < KH; ++k) {
        Frag<F32> f;
        if constexpr (F32) unpack<A>(d[k], f.v);
        else f = d[k];
        step16(f, s * KH + k);
      }
    }
    {
      Frag<F32> d[KH];
#pragma unroll
      for (int k = 0; k < KH; ++k) {
        const int h = k * 16 / p.D;
        d[k] = load8<F32>(p.dgp, head_off(p, cur, h) + (k * 16 - h * p.D) + hh * 8);
      }
#pragma unroll
      for (int k = 0; k < KH; ++k) step16(d[k], 3 * KH + k);
    }
    for (int k = 0; k < kb; ++k) {
      float v[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const int h = k * 16 + hh * 8 + e;
        v[e] = h < p.H ? load1<A, false>(p.db, ((int64_t)cur.b * p.H + h) * p.LL + cur.p) : 0.f;
      }
      Frag<F32> f;
      pack<A>(v, f);
      step16(f, 4 * KH + k);
    }
    float mean, rstd;
    row_stats<A, F32, KS>(z, p.eps, mean, rstd);
    // dz = rstd * (g - mean(g) - xhat * mean(g * xhat)), g = dx * gamma
    float s1 = 0.f, s2 = 0.f;
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      float y[2][8];
      rows8(acc[t], y);
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        float x[8];
        unpack<A>(z[2 * t + u], x);
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const float gx = y[u][e] * gam[t * 32 + 16 * u + 8 * hh + e];
          s1 += gx;
          s2 = __builtin_fmaf(gx, (x[e] - mean) * rstd, s2);
          acc[t][8 * u + e] = gx;  // (from here on in runs of eight channels)
        }
      }
    }
    s1 = sum_both_halves(s1) * (1.0f / C);
    s2 = sum_both_halves(s2) * (1.0f / C);
    const int64_t dzo = pair_off(p.dzs, cur) + hh * 8;
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        float x[8];
        unpack<A>(z[2 * t + u], x);
#pragma unroll
        for (int e = 0; e < 8; ++e) x[e] = rstd * (acc[t][8 * u + e] - s1 - (x[e] - mean) * rstd * s2);
        Frag<F32> f;
        pack<A>(x, f);
        if (cur.valid) store8<F32>(p.dz, dzo + t * 32 + 16 * u, f);
      }
  }
}

// ---- backward: weight gradients -----------------------------------------------------------------------
// Five products with the pair rows as contraction: section s = 0..3 is (d of projection s)^T xhat, with xhat
// the normalised row without gamma and beta (the reduction applies those: one product serves the weight, gamma
// and beta), section 4 is dout^T (gate * o).  Section 0 takes the bias projection along.  A workgroup works
// off one chunk of rows of one section: 32-row tiles (two per stage) are formed in registers, written to LDS as 32-column
// sub-tiles and read back transposed as MFMA operands; its waves own up to two 32 x 32 tiles of the result
// each.  The sums over the rows (bias gradients) come from one more product with a column of ones.
// One chunk's partial: NA*NB*1024 floats of the result tiles, row-major [a][b], then NA*32 row sums; for section 0
// also H*C and H floats of the bias projection.
__host__ __device__ inline size_t wgrad_part_floats(int C, int HD, int H) { return (size_t)C * HD + (C > HD ? C : HD) + (size_t)H * C + H; }

// Sub-tile of 32 columns in LDS: 16-bit rows of 64 bytes, swizzled as the attention's staged tiles; fp32 rows
// of 128 bytes as they are.
template <bool F32> constexpr int kSubRow = F32 ? 128 : 64;
template <bool F32>
__device__ __forceinline__ void sub_write(char* tile, int row, int chunk, const Frag<F32>& f) {
  if constexpr (F32) {
    float4* d = reinterpret_cast<float4*>(tile + row * 128 + chunk * 32);
    d[0] = make_float4(f.v[0], f.v[1], f.v[2], f.v[3]);
    d[1] = make_float4(f.v[4], f.v[5], f.v[6], f.v[7]);
  } else {
    *reinterpret_cast<u32x4*>(tile + 2 * swz_off<32>(row, chunk)) = f.w;
  }
}
// Column l % 32 of the sub-tile, contraction rows rowbase + 8*(e/4) + 4*hh + e%4.
template <bool F32>
__device__ __forceinline__ Frag<F32> sub_frag_t(const char* tile, int rowbase, const FragOffsets<32>& fo, int l32, int hh) {
  Frag<F32> f;
  if constexpr (F32) {
    const float* s = reinterpret_cast<const float*>(tile) + (rowbase + 4 * hh) * 32 + l32;
#pragma unroll
    for (int e = 0; e < 8; ++e) f.v[e] = s[(8 * (e / 4) + e % 4) * 32];
  } else {
    f.w = __builtin_bit_cast(u32x4, lds_frag_t<32>(reinterpret_cast<const half_t*>(tile), rowbase, fo, 0));
  }
  return f;
}

template <class A, bool F32, int C, int HD>
__global__ void __launch_bounds__(512) blk_wgrad_kernel(BlockParams p) {
  constexpr int W = (C > HD) ? C : HD;      // columns a stage buffer holds
  constexpr int TR = F32 ? 32 : 64;         // rows per stage
  constexpr int NP = (TR * W / 8 + 511) / 512;  // 8-element pieces per thread and operand
  constexpr int SUB = TR * kSubRow<F32>;    // bytes of a sub-tile
  constexpr int BUF = 2 * (W / 32) * SUB;   // both operands
  extern __shared__ char smem[];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, l32 = lane & 31, hh = lane >> 5;
  const int sec = (int)blockIdx.x % 5, chunk = (int)blockIdx.x / 5;
  const int na = (sec == 4 ? C : HD) / 32, nb = (sec == 4 ? HD : C) / 32;
  const int nst = (int)((p.LL + TR - 1) / TR);               // stages per batch entry
  const int ntot = p.B * nst, per = (ntot + p.nchunks - 1) / p.nchunks;
  const int first = chunk * per, last = min(ntot, first + per);
  FragOffsets<32> fo;
  fo.init(lane);

  Frag<F32> ra[NP], rx[NP];
  Frag<false> ro[NP];
  bool rv[NP];
  const int ca = na * 4, cb = nb * 4;  // 8-element pieces per row of the two operands
  // this thread's pieces of stage st: operand A (the gradient rows) and what operand B is formed from
  auto fetch = [&](int st) {
    const int b = st / nst;
    const uint32_t p0 = (uint32_t)(st - b * nst) * TR;
#pragma unroll
    for (int n = 0; n < NP; ++n) {
      const int pc = tid + 512 * n;
      {
        const uint32_t row = pc / ca, c8 = (pc % ca) * 8;
        if (row < (uint32_t)TR) {
          uint32_t q = p0 + row;
          q = q < (uint32_t)p.LL ? q : (uint32_t)p.LL - 1u;
          if (sec == 4) {
            const uint32_t i = q / (uint32_t)p.L, j = q - i * (uint32_t)p.L;
            ra[n] = load8<F32>(p.dout, b * p.douts[0] + i * p.douts[1] + j * p.douts[2] + c8);
          } else {
            const int h = c8 / p.D;
            const int64_t off = (((int64_t)b * p.H + h) * p.LL + q) * p.D + (c8 - h * p.D);
            if (sec == 3) {
              ra[n] = load8<F32>(p.dgp, off);
            } else {
              const Frag<false> d = load8<false>(p.dqkv[sec], off);
              if constexpr (F32) unpack<A>(d, ra[n].v);
              else ra[n] = d;
            }
          }
        }
      }
      {
        const uint32_t row = pc / cb, c8 = (pc % cb) * 8;
        rv[n] = false;
        if (row < (uint32_t)TR) {
          uint32_t q = p0 + row;
          rv[n] = q < (uint32_t)p.LL;
          q = rv[n] ? q : (uint32_t)p.LL - 1u;
          if (sec == 4) {
            const int h = c8 / p.D;
            const int64_t off = (((int64_t)b * p.H + h) * p.LL + q) * p.D + (c8 - h * p.D);
            rx[n] = load8<F32>(p.gate, off);
            ro[n] = load8<false>(p.o, off);
          } else {
            const uint32_t i = q / (uint32_t)p.L, j = q - i * (uint32_t)p.L;
            rx[n] = load8<F32>(p.z, b * p.zs[0] + i * p.zs[1] + j * p.zs[2] + c8);
          }
        }
      }
    }
  };
  // forms operand B (gate * o, or the normalised row: the lanes of a row are neighbours) and writes both to LDS;
  // rows beyond the end are zero in operand B
  auto put = [&](char* buf) {
#pragma unroll
    for (int n = 0; n < NP; ++n) {
      const int pc = tid + 512 * n;
      {
        const int row = pc / ca, c = pc % ca;
        if (row < TR) sub_write<F32>(buf + (c / 4) * SUB, row, c % 4, ra[n]);
      }
      const int row = pc / cb, c = pc % cb;
      float v[8];
      unpack<A>(rx[n], v);
      if (sec == 4) {
        float w[8];
        unpack<A>(ro[n], w);
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] *= w[e];
      } else {
        float s = 0.f;
#pragma unroll
        for (int e = 0; e < 8; ++e) s += v[e];
#pragma unroll
        for (int m = 1; m < C / 8; m *= 2) s += __shfl_xor(s, m, 64);
        const float mean = s * (1.0f / C);
        s = 0.f;
#pragma unroll
        for (int e = 0; e < 8; ++e) { v[e] -= mean; s = __builtin_fmaf(v[e], v[e], s); }
#pragma unroll
        for (int m = 1; m < C / 8; m *= 2) s += __shfl_xor(s, m, 64);
        const float rstd = 1.0f / __builtin_sqrtf(s * (1.0f / C) + p.eps);
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] *= rstd;
      }
      if (row < TR) {
        Frag<F32> f;
        pack<A>(v, f);
        if (!rv[n]) f = frag_zero<F32>();
        sub_write<F32>(buf + (W / 32 + c / 4) * SUB, row, c % 4, f);
      }
    }
  };

  floatx16 acc[2], sums = zero16(), accb = zero16(), sumb = zero16();
  acc[0] = zero16();
  acc[1] = zero16();
  const int at = wave % na;                                        // (na is 2 or 4: the same rows for both tiles of a wave)
  const int bt[2] = {wave / na, wave / na + 8 / na};
  const bool own[2] = {bt[0] < nb, bt[1] < nb};
  const bool own_sum = wave < na;
  const bool own_bias = (sec == 0) && wave >= 4 && wave - 4 < nb;  // bias projection: columns of sub-tile wave - 4
  Frag<F32> ones;
  {
    float v[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = 1.0f;
    pack<A>(v, ones);
  }
  // (double buffered: stage st is multiplied while the next one's loads are in flight)
  if (first < last) {
    fetch(first);
    put(smem);
    if (first + 1 < last) fetch(first + 1);
    __syncthreads();
    for (int st = first; st < last; ++st) {
      const char* buf = smem + ((st - first) & 1) * BUF;
      Frag<F32> dbf[TR / 16];
      if (own_bias) {
        const int b = st / nst;
        const uint32_t p0 = (uint32_t)(st - b * nst) * TR;
#pragma unroll
        for (int k = 0; k < TR / 16; ++k) {
          float v[8];
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            const uint32_t q = p0 + k * 16 + 8 * (e / 4) + 4 * hh + e % 4;
            v[e] = (l32 < p.H && q < (uint32_t)p.LL) ? load1<A, false>(p.db, ((int64_t)b * p.H + l32) * p.LL + q) : 0.f;
          }
          pack<A>(v, dbf[k]);
        }
      }
#pragma unroll
      for (int k = 0; k < TR / 16; ++k) {
        const Frag<F32> fa = sub_frag_t<F32>(buf + at * SUB, k * 16, fo, l32, hh);
#pragma unroll
        for (int n = 0; n < 2; ++n)
          if (own[n]) acc[n] = mma<A>(fa, sub_frag_t<F32>(buf + (W / 32 + bt[n]) * SUB, k * 16, fo, l32, hh), acc[n]);
        if (own_sum) {
          // (rows beyond the end repeat the last one here: the ones are zero there)
          Frag<F32> o1 = ones;
          const int b = st / nst;
          const uint32_t left = (uint32_t)p.LL - (uint32_t)(st - b * nst) * TR;
          if (left < (uint32_t)TR) {
            float v[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] = (uint32_t)(k * 16 + 8 * (e / 4) + 4 * hh + e % 4) < left ? 1.0f : 0.0f;
            pack<A>(v, o1);
          }
          sums = mma<A>(fa, o1, sums);
        }
        if (own_bias) {
          accb = mma<A>(dbf[k], sub_frag_t<F32>(buf + (W / 32 + wave - 4) * SUB, k * 16, fo, l32, hh), accb);
          if (wave == 4) sumb = mma<A>(dbf[k], ones, sumb);
        }
      }
      if (st + 1 < last) {
        put(smem + ((st + 1 - first) & 1) * BUF);
        if (st + 2 < last) fetch(st + 2);
      }
      __syncthreads();
    }
  }
  // partial of this chunk
  float* out = p.part + ((size_t)sec * p.nchunks + chunk) * wgrad_part_floats(C, HD, p.H);
  const int ncol = nb * 32;
#pragma unroll
  for (int n = 0; n < 2; ++n)
    if (own[n])
#pragma unroll
      for (int r = 0; r < 16; ++r) out[(size_t)(at * 32 + 8 * (r / 4) + 4 * hh + r % 4) * ncol + bt[n] * 32 + l32] = acc[n][r];
  float* osum = out + (size_t)C * HD;
  if (own_sum && l32 == 0)
#pragma unroll
    for (int r = 0; r < 16; ++r) osum[at * 32 + 8 * (r / 4) + 4 * hh + r % 4] = sums[r];
  if (own_bias) {
    float* ob = osum + W;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int h = 8 * (r / 4) + 4 * hh + r % 4;
      if (h < p.H) {
        ob[(size_t)h * C + (wave - 4) * 32 + l32] = accb[r];
        if (wave == 4 && l32 == 0) ob[(size_t)p.H * C + h] = sumb[r];
      }
    }
  }
}

// Sums the chunks in order, four columns per thread: rows [0, 4*HD) the projections, then H of the bias
// projection, then C of the output projection.
template <class A, bool F32>
__global__ void __launch_bounds__(256) blk_reduce_kernel(BlockParams p, int C) {
  const int HD = p.HD, H = p.H, W = C > HD ? C : HD;
  const size_t pf = wgrad_part_floats(C, HD, H);
  const int cq = C / 4, nproj = (4 * HD + H) * cq, nout = C * (HD / 4);
  const int t = (int)(blockIdx.x * 256 + threadIdx.x);
  if (t >= nproj + nout) return;
  const float* src;
  const float* ssum;
  int n, c;
  if (t < nproj) {
    n = t / cq;
    c = (t % cq) * 4;
    const int s = n < 4 * HD ? n / HD : 0;
    src = p.part + (size_t)s * p.nchunks * pf;
    if (n < 4 * HD) { ssum = src + (size_t)C * HD + n % HD; src += (size_t)(n % HD) * C + c; }
    else { src += (size_t)C * HD + W; ssum = src + (size_t)H * C + (n - 4 * HD); src += (size_t)(n - 4 * HD) * C + c; }
  } else {
    const int u = t - nproj;
    n = u / (HD / 4);
    c = (u % (HD / 4)) * 4;
    src = p.part + (size_t)4 * p.nchunks * pf;
    ssum = src + (size_t)C * HD + n;
    src += (size_t)n * HD + c;
  }
  float a[4] = {0.f, 0.f, 0.f, 0.f}, sum = 0.f;
  for (int k = 0; k < p.nchunks; ++k) {
    const float* s = src + (size_t)k * pf;
#pragma unroll
    for (int e = 0; e < 4; ++e) a[e] += s[e];
    sum += ssum[(size_t)k * pf];
  }
  if (t < nproj) {
    float* g = p.red + (size_t)n * C + c;
#pragma unroll
    for (int e = 0; e < 4; ++e) g[e] = a[e];
    if (c == 0) p.red[(size_t)(4 * HD + H) * C + n] = sum;
    void* dst = n < 4 * HD ? p.dw[n / HD] : p.dwb;
    const int64_t off = (int64_t)(n < 4 * HD ? n % HD : n - 4 * HD) * C + c;
#pragma unroll
    for (int e = 0; e < 4; ++e)
      store1<A, F32>(dst, off + e, load1<A, F32>(p.gamma, c + e) * a[e] + load1<A, F32>(p.beta, c + e) * sum);
    if (c == 0 && n >= 3 * HD && n < 4 * HD && p.dbg != nullptr) store1<A, F32>(p.dbg, n - 3 * HD, sum);
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e) store1<A, F32>(p.dwo, (int64_t)n * HD + c + e, a[e]);
    if (c == 0 && p.dbo != nullptr) store1<A, F32>(p.dbo, n, sum);
  }
}

// dgamma[c] = sum_n W[n][c] G[n][c], dbeta[c] = sum_n W[n][c] * (sum over the rows of d[n]): 16 columns per workgroup.
template <class A, bool F32>
__global__ void __launch_bounds__(512) blk_norm_grad_kernel(BlockParams p, int C) {
  __shared__ float sg[512], sb[512];
  const int tid = threadIdx.x, c = (int)blockIdx.x * 16 + tid % 16, nall = 4 * p.HD + p.H;
  float g = 0.f, b = 0.f;
  for (int n = tid / 16; n < nall; n += 32) {
    const float w = n < 4 * p.HD ? load1<A, F32>(p.w[n / p.HD], (int64_t)(n % p.HD) * C + c)
                                 : load1<A, F32>(p.wb, (int64_t)(n - 4 * p.HD) * C + c);
    g = __builtin_fmaf(w, p.red[(size_t)n * C + c], g);
    b = __builtin_fmaf(w, p.red[(size_t)nall * C + n], b);
  }
  sg[tid] = g;
  sb[tid] = b;
  for (int s = 256; s >= 16; s /= 2) {
    __syncthreads();
    if (tid < s) { sg[tid] += sg[tid + s]; sb[tid] += sb[tid + s]; }
  }
  if (tid < 16) {
    store1<A, F32>(p.dgamma, c, sg[tid]);
    store1<A, F32>(p.dbeta, c, sb[tid]);
  }
}

}  // namespace

// ---- host side ----------------------------------------------------------------------------------------
namespace {

constexpr int kCus = 256;

// (element type, fp32 block) instances
#define FTA_BLOCK_TYPES(X, ...) \
  if (dtype == kF16) X(F16, false, __VA_ARGS__) else if (dtype == kBF16) X(BF16, false, __VA_ARGS__) else X(F16, true, __VA_ARGS__)
#define FTA_BLOCK_C(X) \
  if (C == 64) { FTA_BLOCK_TYPES(X, 64) } else { FTA_BLOCK_TYPES(X, 128) }
#define FTA_BLOCK_C_HD(X)                                                                         \
  if (C == 64 && p.HD == 64) { FTA_BLOCK_TYPES(X, 64, 64) } else if (C == 64) { FTA_BLOCK_TYPES(X, 64, 128) } \
  else if (p.HD == 64) { FTA_BLOCK_TYPES(X, 128, 64) } else { FTA_BLOCK_TYPES(X, 128, 128) }

inline size_t frag_bytes(int dtype) { return dtype == 2 ? kFragBytes<true> : kFragBytes<false>; }

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
  const long blocks = (long)p.B * p.nper;
  const int ntiles = 4 * p.HD / 32 + (p.H + 31) / 32, KS = C / 16;
  const size_t extra = (size_t)(2 * C + p.HD) * sizeof(float);
  int gy = 1;
  while ((size_t)((ntiles + gy - 1) / gy) * KS * frag_bytes(dtype) + extra > 160 * 1024) ++gy;
  const size_t smem = (size_t)((ntiles + gy - 1) / gy) * KS * frag_bytes(dtype) + extra;
  p.cg = column_groups(blocks * gy, 8);
  const dim3 grid((unsigned)workgroups(blocks * p.cg, 8, kCus / gy), (unsigned)gy), block(512);
#define FTA_BLOCK_CASE(AA, FF, CC) return launch_kernel(blk_proj_kernel<AA, FF, CC>, p, grid, block, smem, st);
  FTA_BLOCK_C(FTA_BLOCK_CASE)
#undef FTA_BLOCK_CASE
}

hipError_t launch_block_out(BlockParams p, int C, int dtype, hipStream_t st) {
  const size_t smem = (size_t)(C / 32) * (p.HD / 16) * frag_bytes(dtype) + C * sizeof(float);
  const long blocks = (long)p.B * p.nper;
  p.cg = column_groups(blocks, C / 32);
  const dim3 grid((unsigned)workgroups(blocks * p.cg, 8, 2 * kCus)), block(512);
#define FTA_BLOCK_CASE(AA, FF, CC, HH) return launch_kernel(blk_out_kernel<AA, FF, CC, HH>, p, grid, block, smem, st);
  FTA_BLOCK_C_HD(FTA_BLOCK_CASE)
#undef FTA_BLOCK_CASE
}

hipError_t launch_block_dout(BlockParams p, int C, int dtype, hipStream_t st) {
  const size_t smem = (size_t)(p.HD / 32) * (C / 16) * frag_bytes(dtype);
  const long blocks = (long)p.B * p.nper;
  p.cg = column_groups(blocks, p.HD / 32);
  p.nwg = workgroups(blocks * p.cg, 8, 2 * kCus);
  const dim3 grid((unsigned)(p.nwg + 17)), block(512);  // (17: one fragment of the packed weights per wave at 4 x 33)
#define FTA_BLOCK_CASE(AA, FF, CC, HH) return launch_kernel(blk_dout_kernel<AA, FF, CC, HH>, p, grid, block, smem, st);
  FTA_BLOCK_C_HD(FTA_BLOCK_CASE)
#undef FTA_BLOCK_CASE
}

hipError_t launch_block_dx(BlockParams p, int C, int dtype, hipStream_t st) {
  const long blocks = (long)p.B * p.nper;
  const size_t wbytes = (size_t)(C / 32) * (4 * p.HD / 16 + (p.H + 15) / 16) * frag_bytes(dtype);
  // Weights in LDS where they fit and a workgroup has a row block for each of its eight waves; few row blocks
  // run as many small workgroups that read the weights from the cache.
  const bool wlds = wbytes + C * sizeof(float) <= 160 * 1024 && blocks >= 4 * kCus;
  int nw = 8;
  while (nw > 1 && blocks < (long)nw * kCus) nw /= 2;
  const dim3 grid((unsigned)workgroups(blocks, nw, wlds ? kCus : 2 * kCus * 8 / nw)), block((unsigned)(64 * nw));
  const size_t smem = (wlds ? wbytes : 0) + C * sizeof(float);
#define FTA_BLOCK_CASE(AA, FF, CC, HH)                                                                      \
  {                                                                                                         \
    if constexpr (!FF)                                                                                      \
      if (wlds) return launch_kernel(blk_dx_kernel<AA, FF, CC, HH, true>, p, grid, block, smem, st);        \
    return launch_kernel(blk_dx_kernel<AA, FF, CC, HH, false>, p, grid, block, smem, st);                   \
  }
  FTA_BLOCK_C_HD(FTA_BLOCK_CASE)
#undef FTA_BLOCK_CASE
}

hipError_t launch_block_wgrad(BlockParams p, int C, int dtype, hipStream_t st) {
  const int W = C > p.HD ? C : p.HD;
  const size_t smem = (size_t)2 * 2 * (W / 32) * (dtype == 2 ? 32 * 128 : 64 * 64);
  const dim3 grid((unsigned)(5 * p.nchunks)), block(512);
#define FTA_BLOCK_CASE(AA, FF, CC, HH)                                                          \
  {                                                                                             \
    hipError_t e = launch_kernel(blk_wgrad_kernel<AA, FF, CC, HH>, p, grid, block, smem, st);   \
    if (e != hipSuccess) return e;                                                              \
  }
  FTA_BLOCK_C_HD(FTA_BLOCK_CASE)
#undef FTA_BLOCK_CASE
  const int nred = (4 * p.HD + p.H) * (C / 4) + C * (p.HD / 4);
#define FTA_BLOCK_CASE(AA, FF, UNUSED)                                                                                    \
  {                                                                                                                       \
    hipLaunchKernelGGL((blk_reduce_kernel<AA, FF>), dim3((unsigned)((nred + 255) / 256)), dim3(256), 0, st, p, C);        \
    hipError_t e = hipGetLastError();                                                                                     \
    if (e != hipSuccess) return e;                                                                                        \
    hipLaunchKernelGGL((blk_norm_grad_kernel<AA, FF>), dim3((unsigned)(C / 16)), dim3(512), 0, st, p, C);                 \
    return hipGetLastError();                                                                                             \
  }
  FTA_BLOCK_TYPES(FTA_BLOCK_CASE, 0)
#undef FTA_BLOCK_CASE
}

// ---- C ABI ---------------------------------------------------------------------------------------------
namespace {

size_t align256(size_t n) { return (n + 255) / 256 * 256; }

// Byte offsets of the forward state and the backward workspace.
struct BlockLayout {
  size_t q, k, v, bias, o, gate, lse, state;
  size_t dog, dgp, dq, dk, dv, db, wt, part, red, attn, attn_bytes, total;
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
  l.wt = take((size_t)(b.C / 32) * (4 * HD / 16 + (b.H + 15) / 16) * frag_bytes(b.dtype));
  // Chunks of the weight-gradient kernel: 51 x 5 sections fill the chip once; a chunk keeps at least four stages,
  // so that its partial sums (64 KB at C = H*D = 128) are not what the launch spends its time on.
  const size_t rows = b.dtype == FTA_DTYPE_F32 ? 32 : 64, stages = b.B * ((LL + rows - 1) / rows);
  l.nchunks = (int)(stages / 4 < 1 ? 1 : stages / 4 > 51 ? 51 : stages / 4);
  l.part = take((size_t)5 * l.nchunks * wgrad_part_floats(b.C, (int)HD, b.H) * sizeof(float));
  l.red = take((4 * HD + b.H) * (b.C + 1) * sizeof(float));
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
