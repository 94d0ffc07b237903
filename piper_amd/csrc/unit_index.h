// Ragged work units on the device: expert e of a grouped GEMM owns ceil(rows_e / BM) row tiles times
// n_tiles column tiles; which unit belongs to which expert follows from the row offsets alone, so no
// tile list is built and the host never waits for the routing.
#pragma once
#include "pk_common.h"

namespace pk_units {

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
