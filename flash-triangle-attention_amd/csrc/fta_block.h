// Kernel parameters of the AlphaFold2 block around the attention (fta_block.hip).
#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

namespace fta {

// All element strides are of the NODE's view of the pair tensors: index (b, i, j) is row i, key j of the
// attention, so that the ending node only swaps two strides.  q, k, v, gate, o and their gradients are
// laid out (B, H, L, L, D) contiguously, bias and dbias (B, H, L, L).
struct BlockParams {
  const void* z; void* out; const void* dout; void* dz;
  int64_t zs[3], outs[3], douts[3], dzs[3];
  const void* mask;                       // (B, L) of the block's type, or null
  const void* w[4];                       // q, k, v, gate projections, (H*D, C)
  const void* wb; const void* bg;         // (H, C), (H*D)
  const void* wo; const void* bo;         // (C, H*D), (C)
  const void* gamma; const void* beta;    // (C)
  void* qkv[3]; void* gate; void* bias;   // forward state (qkv, bias: the attention's 16-bit type; gate: the block's type)
  const void* o;
  void* dog; void* dgp;                   // dO (16-bit type), gradient of the gate before the sigmoid (block's type)
  const void* dqkv[3]; const void* db;    // attention gradients
  void* wt;                               // packed transposed projection weights, in MFMA operand order
  float2* stats;                          // the layer norm's {mean, reciprocal deviation} of every pair row
  float* part;                            // weight-gradient partial sums, one block of wgrad_part_floats() per section and chunk
  float* red;                             // contributions to the layer norm's gradients, (groups, 2, C)
  void* dw[4]; void* dwb; void* dbg; void* dwo; void* dbo; void* dgamma; void* dbeta;
  int B, L, H, D, HD;
  int64_t LL;                             // L * L
  int nper;                               // 32-row blocks per batch entry: ceil(LL / 32)
  int cg;                                 // column groups a row block's output tiles are dealt to
  int nwg;                                // workgroups of the work proper (the ones behind them pack weights)
  int nchunks;                            // chunks of the weight-gradient kernel
  float eps;
};

}  // namespace fta
