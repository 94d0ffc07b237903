// Forward products of the experts when an expert has only a few rows (decode, short prefills): every
// weight is used for a handful of tokens, so the kernel is a stream of the weights and its one concern
// is to keep enough of them in flight.
//
//   DUAL : h = silu(x . w1^T) * (x . w3^T)   (g and u written where asked for)
//   else : y = h . w2^T
//
// A unit is 16 * MT rows of one expert times NW weight tiles of 16 output columns (DUAL: NW / 2 gate and
// as many up tiles).  The four waves of a workgroup split the reduction in steps of 64 elements and add
// their sums through LDS.  Weights go from memory straight into the registers of
// v_mfma_f32_16x16x32_bf16 (each is needed by one wave only, LDS would be a detour).  The next step is
// requested before the current one is multiplied, and four workgroups share a CU: 128 kB of weights in
// flight per CU, and the dependent loads at a workgroup's start (row offsets, row map) hide behind the
// others.  Measured on the way (1.2 GB of weights, 64 tokens of the 128-expert region): four steps ahead
// with two workgroups per CU 306 us, two with four 252, one with four and a contiguous share of the
// reduction per wave 225; nontemporal loads +12 %.  Rows of x come out of the L2.
// Against the 128-row persistent tiles, whose units are 1 MB of weights and leave most of the chip idle
// at one token and a ragged last round at more: figures at skinny_rows in grouped_gemm.hip.
#pragma once
#include "pk_common.h"
#include "unit_index.h"

namespace pk_skinny {

constexpr int THREADS = 256, WAVES = 4, STEP = 64;

struct Params {
  const bf16_t* A;           // [rows, lda]
  int64_t lda;
  const int32_t* row_map;    // optional: A row = row_map[sorted row] / map_div
  int32_t map_div;
  const bf16_t* B0;          // [E][N][ldb]; DUAL: gate
  const bf16_t* B1;          // DUAL: up
  int64_t ldb, strideB;
  const int32_t* starts;
  int32_t E, K, N, n_tiles;
  bf16_t* O0;                // y;  DUAL: g or nullptr
  bf16_t* O1;                //     DUAL: u or nullptr
  bf16_t* O2;                //     DUAL: h
  int64_t ldc;
};

template <int MT, int NW, bool DUAL>
__global__ __launch_bounds__(THREADS, 4) void kernel(const Params p) {
  constexpr int BM = 16 * MT, NT = DUAL ? NW / 2 : NW, BN = 16 * NT;
  __shared__ float red[WAVES][MT * NW][256];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15, g = lane >> 4;
  const pk_units::UnitIndex ui = pk_units::build_unit_index<BM>(p.starts, p.E, p.n_tiles);
  const int unit = blockIdx.x;
  if (unit >= ui.total) return;
  int e, mt, nt;
  pk_units::locate_unit<BM>(ui, pk_units::as_const(p.starts), p.E, p.n_tiles, unit, e, mt, nt);
  const int row0 = p.starts[e] + mt * BM;
  const int rows = min(BM, p.starts[e + 1] - row0);
  const int n0 = nt * BN;

  const bf16_t* wp[NW];
  bool w_ok[NW];
#pragma unroll
  for (int t = 0; t < NW; ++t) {
    const int col = n0 + (DUAL ? t >> 1 : t) * 16 + r;
    w_ok[t] = col < p.N;
    wp[t] = (DUAL && (t & 1) ? p.B1 : p.B0) + (int64_t)e * p.strideB + (int64_t)(w_ok[t] ? col : 0) * p.ldb + 8 * g;
  }
  const bf16_t* xp[MT];
  bool x_ok[MT];
#pragma unroll
  for (int m = 0; m < MT; ++m) {
    x_ok[m] = 16 * m + r < rows;
    int64_t src = row0 + (x_ok[m] ? 16 * m + r : 0);
    if (p.row_map) src = p.row_map[src] / p.map_div;
    xp[m] = p.A + src * p.lda + 8 * g;
  }

  struct Regs {
    u32x4_t w[NW][2], x[MT][2];
  };
  const int steps = (p.K + STEP - 1) / STEP;
  const int first = wave * steps / WAVES, mine = (wave + 1) * steps / WAVES - first;   // a contiguous share of the steps
  const u32x4_t zero = {0u, 0u, 0u, 0u};
  auto request = [&](Regs& q, int i) {      // the i-th step of this wave's share
    const int k0 = (first + i) * STEP;
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      const bool in = k0 + 32 * half + 8 * g < p.K;
#pragma unroll
      for (int t = 0; t < NW; ++t) q.w[t][half] = in && w_ok[t] ? *reinterpret_cast<const u32x4_t*>(wp[t] + k0 + 32 * half) : zero;
    }
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      const bool in = k0 + 32 * half + 8 * g < p.K;
#pragma unroll
      for (int m = 0; m < MT; ++m) q.x[m][half] = in && x_ok[m] ? *reinterpret_cast<const u32x4_t*>(xp[m] + k0 + 32 * half) : zero;
    }
  };
  floatx4_t acc[MT][NW];
#pragma unroll
  for (int m = 0; m < MT; ++m)
#pragma unroll
    for (int t = 0; t < NW; ++t) acc[m][t] = floatx4_t{0.f, 0.f, 0.f, 0.f};
  auto multiply = [&](const Regs& q) {
#pragma unroll
    for (int half = 0; half < 2; ++half)
#pragma unroll
      for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int t = 0; t < NW; ++t)
          acc[m][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, q.w[t][half]),
                                                              __builtin_bit_cast(bf16x8_t, q.x[m][half]), acc[m][t], 0, 0, 0);
  };
  Regs a, b;
  if (mine > 0) request(a, 0);
  for (int i = 0; i < mine; i += 2) {
    __builtin_amdgcn_sched_barrier(0);
    if (i + 1 < mine) request(b, i + 1);
    __builtin_amdgcn_sched_barrier(0);
    multiply(a);
    if (i + 1 >= mine) break;
    __builtin_amdgcn_sched_barrier(0);
    if (i + 2 < mine) request(a, i + 2);
    __builtin_amdgcn_sched_barrier(0);
    multiply(b);
  }

  // acc[m][t][v] of lane (g, r): output column 16 t + 4 g + v, row 16 m + r.  Stored as [row][column]
#pragma unroll
  for (int m = 0; m < MT; ++m)
#pragma unroll
    for (int t = 0; t < NW; ++t)
      *reinterpret_cast<floatx4_t*>(&red[wave][m * NW + t][r * 16 + 4 * g]) = acc[m][t];
  __syncthreads();
  const int row = tid >> 4, c = tid & 15;
#pragma unroll
  for (int m = 0; m < MT; ++m) {
    if (16 * m + row >= rows) continue;
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const int n = n0 + 16 * t + c;
      if (n >= p.N) continue;
      const int64_t o = (int64_t)(row0 + 16 * m + row) * p.ldc + n;
      auto total = [&](int which) {
        float s = 0.f;
#pragma unroll
        for (int w = 0; w < WAVES; ++w) s += red[w][m * NW + which][tid];
        return s;
      };
      if constexpr (DUAL) {
        const bf16_t gv = (bf16_t)total(2 * t), uv = (bf16_t)total(2 * t + 1);
        if (p.O0) p.O0[o] = gv;
        if (p.O1) p.O1[o] = uv;
        const float gf = (float)gv;
        p.O2[o] = (bf16_t)((gf / (1.f + __expf(-gf))) * (float)uv);
      } else {
        p.O0[o] = (bf16_t)total(t);
      }
    }
  }
}

template <int MT, int NW, bool DUAL>
inline int launch(Params p, int64_t A_rows, int kernel_id, hipStream_t s) {
  constexpr int BN = 16 * (DUAL ? NW / 2 : NW);
  p.n_tiles = (int32_t)pk_ceil_div(p.N, BN);
  // an expert with rows has at most one partly filled row tile
  const int64_t units = (A_rows / (16 * MT) + (A_rows < p.E ? A_rows : p.E)) * p.n_tiles;
  if (units > 0x7fffff00ll) return PK_ERR_SHAPE;
  PK_LAUNCH_NOCHECK(kernel_id, s, (kernel<MT, NW, DUAL>), dim3((unsigned)units), dim3(THREADS), 0, s, p);
  PK_RETURN_IF_LAUNCH_FAILED();
  return PK_OK;
}

// rows: expected rows of an expert that has any.  Units of 16 rows up to 8 of them (a second tile would
// mostly multiply nothing: -4 % at one row), of 32 rows beyond (an expert's weights are read once per
// unit: -20 % at 16 rows, even at 10).
template <bool DUAL>
inline int launch_for_rows(const Params& p, int64_t A_rows, int64_t rows, int kernel_id, hipStream_t s) {
  if (rows <= 8) return launch<1, 2, DUAL>(p, A_rows, kernel_id, s);
  return launch<2, 2, DUAL>(p, A_rows, kernel_id, s);
}

}  // namespace pk_skinny
