// Ragged work units on the device: expert e of a grouped GEMM owns ceil(rows_e / BM) row tiles times
// n_tiles column tiles; which unit belongs to which expert follows from the row offsets alone, so no
// tile list is built and the host never waits for the routing.
#pragma once
#include "pk_common.h"

namespace pk_units {

// Division of a non-negative int32 by a divisor fixed per launch without the ~25 instructions of
// the general integer division: multiply-high by 2^(32-s) for d = 2^s, otherwise by
// floor(2^(31+s)/d)+1 followed by a shift by s-1 with s = ceil(log2 d) (exact for 0 <= n < 2^31).
struct FastDiv {
  uint32_t mul;    // 0: divisor is 1
  int32_t shift;
  int64_t d;       // the divisor itself (host side checks)
};
inline FastDiv make_fastdiv(int64_t d) {
  FastDiv f = {0u, 0, d < 1 ? 1 : d};
  if (d <= 1) return f;
  int s = 0;
  while (((int64_t)1 << s) < d) ++s;
  if (((int64_t)1 << s) == d) { f.mul = 1u << (32 - s); return f; }   // mulhi by 2^(32-s) is the shift by s
  f.mul = (uint32_t)((((uint64_t)1 << (31 + s)) / (uint64_t)d) + 1u);
  f.shift = s - 1;
  return f;
}
// No branch on the divisor's kind (it would sit between the MFMAs of the loops that divide per lane):
// the product is always formed and a mask picks n itself for a divisor of 1.
__device__ __forceinline__ int fastdiv(int n, const FastDiv f) {
  const uint32_t u = (uint32_t)n;
  const uint32_t q = __umulhi(u, f.mul) >> f.shift;
  const uint32_t keep = f.mul == 0u ? 0xffffffffu : 0u;
  return (int)((u & keep) | (q & ~keep));
}

// Read-only tables (row offsets, row maps) addressed wave-uniformly: going through the constant
// address space makes these scalar loads (lgkmcnt), which leaves vmcnt to the LDS ring.
typedef const __attribute__((address_space(4))) int32_t* const_i32_ptr;
__device__ __forceinline__ const_i32_ptr as_const(const int32_t* p) { return (const_i32_ptr)(uintptr_t)p; }

// Per-lane slice of the prefix sum of work units over experts: lane l covers experts
// [l*epl, (l+1)*epl).  Built once per wave with ordinary loads; locating a unit afterwards
// takes a ballot plus a short scalar walk, so it can run in the middle of the k-loop without
// touching the vector-memory counter that tracks the LDS ring.
struct UnitIndex {
  int excl, incl, total, epl;
};
template <int BM>
__device__ __forceinline__ UnitIndex build_unit_index(const int32_t* __restrict__ starts, int E, int n_tiles) {
  const int lane = threadIdx.x & 63;
  UnitIndex ui;
  ui.epl = (E + 63) >> 6;
  const int e_lo = lane * ui.epl, e_hi = min(E, e_lo + ui.epl);
  int mine = 0;
  for (int e = e_lo; e < e_hi; ++e) mine += ((starts[e + 1] - starts[e] + BM - 1) / BM) * n_tiles;
  int incl = mine;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const int v = __shfl_up(incl, off, PK_WAVE);
    if (lane >= off) incl += v;
  }
  ui.incl = incl;
  ui.excl = incl - mine;
  ui.total = __builtin_amdgcn_readlane(incl, 63);
  return ui;
}
// unit < ui.total.  Units of expert e are laid out [n-tile][m-tile], so neighbouring units share
// the weight tile.  Everything returned is wave-uniform.
template <int BM>
__device__ __forceinline__ void locate_unit(const UnitIndex& ui, const_i32_ptr starts, int E, int n_tiles,
                                            int unit, int& e_out, int& mt_out, int& nt_out) {
  const unsigned long long bal = __ballot(unit >= ui.excl && unit < ui.incl);
  const int src = __builtin_amdgcn_readfirstlane(__ffsll((long long)bal) - 1);
  int u = unit - __builtin_amdgcn_readlane(ui.excl, src);
  int e = src * ui.epl;
  const int e_hi = min(E, e + ui.epl);
  int tiles = 1;
  for (; e < e_hi; ++e) {
    tiles = (starts[e + 1] - starts[e] + BM - 1) / BM;
    const int units = tiles * n_tiles;
    if (u < units) break;
    u -= units;
  }
  tiles = tiles > 0 ? tiles : 1;
  e_out = e;
  nt_out = u / tiles;
  mt_out = u - nt_out * tiles;
}

}  // namespace pk_units
