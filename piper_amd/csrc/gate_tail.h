// The last step of the gate's weight and bias gradients: partial sums that the blocks of an earlier launch left in the
// workspace are added up, in a fixed order.  A few microseconds of work behind a launch of its own, so it is written as
// extra blocks (of 256 threads) that another kernel can carry: the norm's backward where there is one.
#pragma once
#include "pk_common.h"

constexpr int kColsumBlocks = 64;

struct GateTail {
  const float* part;      // split-K partial results of d_w_gate [splits][n], or nullptr
  float* d_w;
  int64_t n;              // a multiple of 4
  int32_t splits, accumulate;
  int32_t w_blocks;       // blocks for them (1,024 elements each), then one for 256 experts each:
  const float* col_part;  // partial column sums of d_logits [col_blocks][E], or nullptr
  float* d_bias;
  int32_t E, col_blocks, bias_blocks;
  int blocks() const { return w_blocks + bias_blocks; }
};

namespace {

// column sums: all loads first (one round trip), then the sum in block order
__device__ __forceinline__ void colsum_final(int block, const float* __restrict__ part, int nblocks, int E, float* __restrict__ d_bias,
                                             int accumulate) {
  const int e = block * 256 + threadIdx.x;
  if (e >= E) return;
  float v[kColsumBlocks];
#pragma unroll
  for (int b = 0; b < kColsumBlocks; ++b) v[b] = b < nblocks ? part[(int64_t)b * E + e] : 0.f;
  float s = 0.f;
#pragma unroll
  for (int b = 0; b < kColsumBlocks; ++b) s += v[b];
  d_bias[e] = accumulate ? d_bias[e] + s : s;
}
__device__ __forceinline__ void gate_tail(const GateTail& t, int block) {
  if (block >= t.w_blocks) {
    colsum_final(block - t.w_blocks, t.col_part, t.col_blocks, t.E, t.d_bias, t.accumulate);
    return;
  }
  const int64_t i = ((int64_t)block * 256 + threadIdx.x) * 4;
  if (i >= t.n) return;
  floatx4_t s = {0.f, 0.f, 0.f, 0.f};
  if (t.accumulate) s = *reinterpret_cast<const floatx4_t*>(t.d_w + i);
  for (int z0 = 0; z0 < t.splits; z0 += 8) {
    floatx4_t v[8];
#pragma unroll
    for (int z = 0; z < 8; ++z) v[z] = *reinterpret_cast<const floatx4_t*>(t.part + (int64_t)min(z0 + z, t.splits - 1) * t.n + i);
#pragma unroll
    for (int z = 0; z < 8; ++z)
      if (z0 + z < t.splits) s += v[z];
  }
  *reinterpret_cast<floatx4_t*>(t.d_w + i) = s;
}
__global__ __launch_bounds__(256) void gate_tail_kernel(const GateTail t) { gate_tail(t, blockIdx.x); }

inline int launch_gate_tail(const GateTail& t, hipStream_t s) {
  if (t.blocks() == 0) return PK_OK;
  PK_LAUNCH_NOCHECK(pk_timing::K_GATE_LOGITS_BWD, s, gate_tail_kernel, dim3((unsigned)t.blocks()), dim3(256), 0, s, t);
  PK_RETURN_IF_LAUNCH_FAILED();
  return PK_OK;
}

}  // namespace

// pk_rmsnorm_bwd whose kernel also does the work of `tail` (permute.hip)
int pk_rmsnorm_bwd_with_tail(const void* d_y, const void* x, int dtype, const void* weight, const float* rstd, const void* d_x_addend,
                             void* d_x, void* d_weight, int accumulate, int64_t T, int64_t H, void* workspace, int64_t workspace_bytes,
                             const GateTail& tail, hipStream_t s);
