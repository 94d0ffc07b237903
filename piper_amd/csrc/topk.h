// Softmax and top-k of a token's logits by one wave, and the wave-wide reductions it is made of.
#pragma once
#include "pk_common.h"

namespace {

// Order-preserving map float -> uint32 (larger float -> larger uint).  -0.0 is folded into
// +0.0 and every NaN into the positive quiet NaN so that ties and NaNs behave like
// torch.sort(descending=True, stable=True).
__device__ __forceinline__ uint32_t orderable(float v) {
  v = v + 0.0f;
  uint32_t u = __float_as_uint(v);
  if (v != v) u = 0x7fc00000u;
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
__device__ __forceinline__ float from_orderable(uint32_t o) {
  const uint32_t u = (o & 0x80000000u) ? (o ^ 0x80000000u) : ~o;
  return __uint_as_float(u);
}

// Wave-wide reductions on the vector ALU: lanes are combined within rows of 16 and then across rows with
// data-parallel-primitive operands, and lane 63 ends with the result, read back into a scalar.  Six
// dependent instructions, where a butterfly of LDS-permute shuffles waits for the LDS six times (twelve
// for a 64-bit value): top-8 of 128 spent most of its time in them.
template <int CTRL, int ROWS>
__device__ __forceinline__ uint32_t dpp_or_zero(uint32_t v) {
  return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, ROWS, 0xf, false);
}
#define PK_DPP_STEPS(OP)                    \
  OP(0x111, 0xf) /* row_shr 1 */            \
  OP(0x112, 0xf) /* row_shr 2 */            \
  OP(0x114, 0xf) /* row_shr 4 */            \
  OP(0x118, 0xf) /* row_shr 8 */            \
  OP(0x142, 0xa) /* row_bcast 15 */         \
  OP(0x143, 0xc) /* row_bcast 31 */
__device__ __forceinline__ uint32_t wave_max_u32(uint32_t v) {      // identity 0
#define PK_STEP(C, R) { const uint32_t o = dpp_or_zero<C, R>(v); v = o > v ? o : v; }
  PK_DPP_STEPS(PK_STEP)
#undef PK_STEP
  return (uint32_t)__builtin_amdgcn_readlane((int)v, 63);
}
__device__ __forceinline__ float wave_sum_f32(float f) {
#define PK_STEP(C, R) f += __uint_as_float(dpp_or_zero<C, R>(__float_as_uint(f)));
  PK_DPP_STEPS(PK_STEP)
#undef PK_STEP
  return __uint_as_float((uint32_t)__builtin_amdgcn_readlane((int)__float_as_uint(f), 63));
}
#undef PK_DPP_STEPS

// Top-k of NT tokens by one wave (two at a time hide each other's latency).  Lane l owns experts l, l+64, ... (EPL of
// them): `val` their logits (0 past the last expert).  Lanes below K get the score and the expert of the k-th choice.
template <int EPL, int NT>
__device__ __forceinline__ void topk_of(const float (&val)[NT][EPL], int lane, int E, int K, int route_norm, float route_scale,
                                        float (&out_s)[NT], int (&out_e)[NT]) {
  uint32_t key[NT][EPL];
  float vmax[NT], my_v[NT];
  int my_e[NT];
#pragma unroll
  for (int n = 0; n < NT; ++n) {
    vmax[n] = my_v[n] = 0.f;
    my_e[n] = 0;
#pragma unroll
    for (int j = 0; j < EPL; ++j)
      key[n][j] = lane + 64 * j < E ? orderable(val[n][j]) : 0u;  // 0 never wins: no value maps to it (the smallest, -inf, maps to 0x007fffff)
  }
  for (int k = 0; k < K; ++k) {
    uint32_t best[NT];
#pragma unroll
    for (int n = 0; n < NT; ++n) {
      best[n] = 0u;
#pragma unroll
      for (int j = 0; j < EPL; ++j) best[n] = key[n][j] > best[n] ? key[n][j] : best[n];
    }
#pragma unroll
    for (int n = 0; n < NT; ++n) best[n] = wave_max_u32(best[n]);
#pragma unroll
    for (int n = 0; n < NT; ++n) {
      // the lowest expert id among those that hold the maximum: ids are lane + 64 j
      int e_win = 0;
      bool found = false;
#pragma unroll
      for (int j = 0; j < EPL; ++j) {
        const unsigned long long at = __ballot(key[n][j] == best[n]);
        if (!found && at != 0ull) {
          found = true;
          const int l = (int)__ffsll((long long)at) - 1;
          e_win = l + 64 * j;
          if (lane == l) key[n][j] = 0u;
        }
      }
      const float v_win = from_orderable(best[n]);
      if (k == 0) vmax[n] = v_win;
      if (lane == k) { my_v[n] = v_win; my_e[n] = e_win; }
    }
  }
#pragma unroll
  for (int n = 0; n < NT; ++n) {
    float part = 0.f;
#pragma unroll
    for (int j = 0; j < EPL; ++j)
      if (lane + 64 * j < E) part += expf(val[n][j] - vmax[n]);
    const float denom = wave_sum_f32(part);
    float s = (lane < K) ? expf(my_v[n] - vmax[n]) / denom : 0.f;
    if (route_norm) {
      const float S = wave_sum_f32(s);
      s = s / (S + 1e-20f);
    }
    out_s[n] = s * route_scale;
    out_e[n] = my_e[n];
  }
}

}  // namespace
