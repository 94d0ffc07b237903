// Grouped GEMMs on the matrix cores for what the 256-wide bf16 kernels of grouped_gemm.hip do not
// take: fp32 operands (v_mfma_f32_32x32x2_f32: exact fp32 products and sums) and bf16 widths that are
// no multiple of 128.  Every row only has to be a whole number of 16-byte pieces (4 fp32 or 8 bf16
// elements); row, column and reduction remainders are fetched as zeros and masked on store.
//
//   ragged M: C[rows_e, N] = sum_seg A_seg[rows_e, K] . B_seg[e]     (forward, input gradient)
//   ragged K: C[e][M, N] (+)= A[rows_e, M]^T . B[rows_e, N]           (weight gradient)
//
// One workgroup of four waves (2 x 2) per output tile of 64 x 64 or 128 x 128.  A k-tile is 128 bytes
// of the reduction index of every operand row (32 fp32 or 64 bf16); the pieces of tile k+1 are fetched
// into registers while tile k is multiplied out of LDS and then stored to the other LDS buffer: one
// barrier per k-tile.  The operands pass through registers rather than straight into LDS because the
// masking then costs one select per piece and nothing has to be counted by hand; at fp32, where a
// k-tile of a 64 x 64 wave tile is 64 MFMAs of 64 cycles, the round trip to memory is covered entirely,
// and with bf16 two (128 x 128) or five (64 x 64) workgroups share a CU.
// Against one 64 x 64 FMA tile per workgroup (simt_gemm.h, which keeps the widths that are no multiple
// of 16 bytes): see the figures at tile_gemm_ok in grouped_gemm.hip.
#pragma once
#include "pk_common.h"
#include "unit_index.h"

namespace pk_tile {

constexpr int THREADS = 256;
constexpr int NXCD = 8;

typedef short shortx4_t __attribute__((ext_vector_type(4)));
typedef short shortx8_t __attribute__((ext_vector_type(8)));

template <typename T> constexpr int kBK = 128 / (int)sizeof(T);      // reduction depth of a k-tile
template <typename T> constexpr int kPiece = 16 / (int)sizeof(T);    // elements of a 16-byte piece

// ---- LDS tiles, in 16-byte pieces, XOR-swizzled against bank conflicts (both are X * 128 bytes):
// KC: [X rows of the M or N index][8 pieces along k];  piece c of row r sits at c ^ ((r >> 1) & 7)
// MN: [BK k][X columns of the M or N index];            piece c of k-row k sits at c ^ swz(k)
template <typename T, int X>
struct Mn {
  static constexpr int CPR = X * (int)sizeof(T) / 16;
  __device__ static __forceinline__ int swz(int k) {
    // the transposing read of bf16 takes four k-rows at once: spread them over the banks
    if (sizeof(T) == 4) return 0;
    return CPR >= 16 ? (k & 3) << 2 : (k & 1) << 2;
  }
};
__device__ __forceinline__ int kc_swz(int r) { return (r >> 1) & 7; }

// The reduction elements of one step (two pieces of every row: 16 bf16 or 8 fp32) for 32 rows of the
// M or N index, as MFMA operands.  Lane l stands for row l % 32 and the step's piece l / 32; the four
// fp32 values of a piece feed four MFMAs in turn, which pairs k and k+4 instead of k and k+1: the
// same products, since both operands are dealt alike.
template <typename T> struct Frag;
template <> struct Frag<bf16_t> { bf16x8_t v; };
template <> struct Frag<float> { floatx4_t v; };

template <typename T>
__device__ __forceinline__ Frag<T> frag_kc(const char* tile, int row0, int step, int lane) {
  const int r = row0 + (lane & 31), c = 2 * step + (lane >> 5);
  Frag<T> f;
  f.v = *reinterpret_cast<const decltype(f.v)*>(tile + r * 128 + ((c ^ kc_swz(r)) << 4));
  return f;
}
template <typename T, int X>
__device__ __forceinline__ Frag<T> frag_mn(const char* tile, int col0, int step, int lane) {
  Frag<T> f;
  if constexpr (sizeof(T) == 4) {
    const char* p = tile + ((8 * step + 4 * (lane >> 5)) * X + col0 + (lane & 31)) * 4;
#pragma unroll
    for (int j = 0; j < 4; ++j) f.v[j] = *reinterpret_cast<const float*>(p + j * X * 4);
  } else {
    // within 16 lanes, lane i points at 4 consecutive columns of k-row i / 4 and receives 4 consecutive
    // k of column i
    const int i = lane & 15;
    const int k = 16 * step + 8 * (lane >> 5) + (i >> 2);
    const int col = col0 + 16 * ((lane >> 4) & 1) + 4 * (i & 3);
    const char* p0 = tile + k * (X * 2) + (((col >> 3) ^ Mn<T, X>::swz(k)) << 4) + (col & 7) * 2;
    const char* p1 = tile + (k + 4) * (X * 2) + (((col >> 3) ^ Mn<T, X>::swz(k + 4)) << 4) + (col & 7) * 2;
    const shortx4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) shortx4_t*)(p0));
    const shortx4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) shortx4_t*)(p1));
    f.v = __builtin_bit_cast(bf16x8_t, (shortx8_t)__builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
  }
  return f;
}
// acc += b . a, operands swapped so that a lane holds 4 consecutive columns of one output row:
//   acc[v] = C[row = lane % 32][col = 8 * (v / 4) + 4 * (lane / 32) + v % 4]
__device__ __forceinline__ void mma(floatx16_t& acc, const Frag<bf16_t>& a, const Frag<bf16_t>& b) {
  acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(b.v, a.v, acc, 0, 0, 0);
}
__device__ __forceinline__ void mma(floatx16_t& acc, const Frag<float>& a, const Frag<float>& b) {
#pragma unroll
  for (int j = 0; j < 4; ++j) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(b.v[j], a.v[j], acc, 0, 0, 0);
}

template <typename T>
__device__ __forceinline__ void store4(T* p, const float (&f)[4]);
template <>
__device__ __forceinline__ void store4<float>(float* p, const float (&f)[4]) {
  *reinterpret_cast<floatx4_t*>(p) = floatx4_t{f[0], f[1], f[2], f[3]};
}
template <>
__device__ __forceinline__ void store4<bf16_t>(bf16_t* p, const float (&f)[4]) {
  bf16x4_t v;
#pragma unroll
  for (int i = 0; i < 4; ++i) v[i] = (bf16_t)f[i];
  *reinterpret_cast<bf16x4_t*>(p) = v;
}
template <typename T>
__device__ __forceinline__ void load4(const T* p, float (&f)[4]);
template <>
__device__ __forceinline__ void load4<float>(const float* p, float (&f)[4]) {
  const floatx4_t v = *reinterpret_cast<const floatx4_t*>(p);
#pragma unroll
  for (int i = 0; i < 4; ++i) f[i] = v[i];
}
template <>
__device__ __forceinline__ void load4<bf16_t>(const bf16_t* p, float (&f)[4]) {
  const bf16x4_t v = *reinterpret_cast<const bf16x4_t*>(p);
#pragma unroll
  for (int i = 0; i < 4; ++i) f[i] = (float)v[i];
}

// ---------------------------------------------------------------------------------- ragged M
struct RaggedM {
  const void* A0;           // A of k-segment 0, row-major [rows, lda]
  const void* A1;           // k-segment 1 (nseg == 2)
  int64_t lda;
  const int32_t* row_map;   // optional gather: A row = row_map[sorted row] / map_div
  int32_t map_div;
  const void* B0;           // weights of k-segment 0 (DUAL: gate)
  const void* B1;           // weights of k-segment 1 (DUAL: up)
  int64_t ldb, strideB;     // row stride, elements between experts
  const int32_t* starts;
  int32_t E, K, nseg, N;
  int32_t n_tiles;
  void* O0;                 // C;  DUAL: g (optional)
  void* O1;                 //     DUAL: u (optional)
  void* O2;                 //     DUAL: h = silu(g) * u
  int64_t ldc;
};

// Tile b of a launch.  Blocks b, b + 8, ... run on one XCD: four neighbouring tiles (which share
// weights or rows) stay on it, the next four go to the next XCD.
__device__ __forceinline__ int unit_of_block(int b) {
  const int x = b % NXCD, q = b / NXCD;
  return ((q >> 2) * NXCD + x) * 4 + (q & 3);
}

// DUAL: two weight matrices (gate and up) against the same A rows, SiLU(g) * u in the epilogue.
template <typename T, int TM, int TN, bool B_KC, bool DUAL>
__global__ __launch_bounds__(THREADS) void ragged_m_kernel(const RaggedM p) {
  constexpr int BM = 64 * TM, BN = 64 * TN, BK = kBK<T>, PIECE = kPiece<T>;
  constexpr int NB = DUAL ? 2 : 1;
  constexpr int LA = BM * 8 / THREADS, LB = BN * 8 / THREADS;
  constexpr int A_BYTES = BM * 128, B_BYTES = BN * 128, STAGE = A_BYTES + NB * B_BYTES;
  static_assert(!DUAL || B_KC, "gate and up weights are K-contiguous");
  __shared__ __attribute__((aligned(16))) char smem[2 * STAGE];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave >> 1, wn = wave & 1;
  const pk_units::UnitIndex ui = pk_units::build_unit_index<BM>(p.starts, p.E, p.n_tiles);
  const int unit = unit_of_block(blockIdx.x);
  if (unit >= ui.total) return;
  int e, mt, nt;
  pk_units::locate_unit<BM>(ui, pk_units::as_const(p.starts), p.E, p.n_tiles, unit, e, mt, nt);
  const int row0 = p.starts[e] + mt * BM;
  const int rows = min(BM, p.starts[e + 1] - row0);
  const int n0 = nt * BN;

  // the thread's A rows (fixed over the reduction) and B rows or columns
  const T* a_ptr[LA];
  const T* b_ptr[LB];
  int b_k[LB];                       // MN weights: k-row of the piece inside a k-tile
  const int a_kofs = (tid & 7) * PIECE;
  bool a_ok[LA], b_ok[LB];
#pragma unroll
  for (int i = 0; i < LA; ++i) {
    const int r = (tid + i * THREADS) >> 3;
    a_ok[i] = r < rows;
    int64_t src = row0 + (a_ok[i] ? r : 0);
    if (p.row_map) src = p.row_map[src] / p.map_div;
    a_ptr[i] = reinterpret_cast<const T*>(p.A0) + src * p.lda + a_kofs;
  }
  const T* const B = reinterpret_cast<const T*>(p.B0) + (int64_t)e * p.strideB;
#pragma unroll
  for (int i = 0; i < LB; ++i) {
    const int s = tid + i * THREADS;
    if (B_KC) {
      const int n = n0 + (s >> 3);
      b_ok[i] = n < p.N;
      b_k[i] = a_kofs;
      b_ptr[i] = B + (int64_t)(b_ok[i] ? n : 0) * p.ldb + a_kofs;
    } else {
      b_k[i] = s / Mn<T, BN>::CPR;
      const int n = n0 + (s % Mn<T, BN>::CPR) * PIECE;
      b_ok[i] = n < p.N;
      b_ptr[i] = B + (int64_t)b_k[i] * p.ldb + (b_ok[i] ? n : 0);
    }
  }
  const int64_t seg_a = reinterpret_cast<const T*>(p.A1) - reinterpret_cast<const T*>(p.A0);
  const int64_t seg_b = reinterpret_cast<const T*>(p.B1) - reinterpret_cast<const T*>(p.B0);
  const int kt_per_seg = (p.K + BK - 1) / BK, nkt = kt_per_seg * p.nseg;

  u32x4_t ra[LA], rb[NB][LB];
  auto fetch = [&](int kt) {
    const bool second = kt >= kt_per_seg;
    const int k0 = (second ? kt - kt_per_seg : kt) * BK;
    const u32x4_t zero = {0u, 0u, 0u, 0u};
#pragma unroll
    for (int i = 0; i < LA; ++i) {
      ra[i] = zero;
      if (a_ok[i] && k0 + a_kofs < p.K) ra[i] = *reinterpret_cast<const u32x4_t*>(a_ptr[i] + k0 + (second ? seg_a : 0));
    }
#pragma unroll
    for (int q = 0; q < NB; ++q)
#pragma unroll
      for (int i = 0; i < LB; ++i) {
        rb[q][i] = zero;
        const int64_t k_at = B_KC ? (int64_t)k0 : (int64_t)k0 * p.ldb;
        if (b_ok[i] && k0 + b_k[i] < p.K)
          rb[q][i] = *reinterpret_cast<const u32x4_t*>(b_ptr[i] + k_at + (DUAL ? (q ? seg_b : 0) : (second ? seg_b : 0)));
      }
  };
  auto deposit = [&](char* st) {
#pragma unroll
    for (int i = 0; i < LA; ++i) {
      const int s = tid + i * THREADS, r = s >> 3, c = s & 7;
      *reinterpret_cast<u32x4_t*>(st + r * 128 + ((c ^ kc_swz(r)) << 4)) = ra[i];
    }
#pragma unroll
    for (int q = 0; q < NB; ++q)
#pragma unroll
      for (int i = 0; i < LB; ++i) {
        const int s = tid + i * THREADS;
        char* const t = st + A_BYTES + q * B_BYTES;
        if (B_KC) {
          const int r = s >> 3, c = s & 7;
          *reinterpret_cast<u32x4_t*>(t + r * 128 + ((c ^ kc_swz(r)) << 4)) = rb[q][i];
        } else {
          using M = Mn<T, BN>;
          const int k = s / M::CPR, c = s % M::CPR;
          *reinterpret_cast<u32x4_t*>(t + k * (M::CPR * 16) + ((c ^ M::swz(k)) << 4)) = rb[q][i];
        }
      }
  };

  floatx16_t acc[NB][TM][TN];
#pragma unroll
  for (int q = 0; q < NB; ++q)
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[q][i][j][v] = 0.f;

  const bool wave_has_rows = wm * 32 * TM < rows;
  fetch(0);
  deposit(smem);
  __syncthreads();
  for (int kt = 0; kt < nkt; ++kt) {
    const char* const st = smem + (kt & 1) * STAGE;
    const bool more = kt + 1 < nkt;
    if (more) fetch(kt + 1);
    if (wave_has_rows) {
#pragma unroll
      for (int step = 0; step < 4; ++step) {
        Frag<T> a[TM], b[NB][TN];
#pragma unroll
        for (int i = 0; i < TM; ++i) a[i] = frag_kc<T>(st, (wm * TM + i) * 32, step, lane);
#pragma unroll
        for (int q = 0; q < NB; ++q)
#pragma unroll
          for (int j = 0; j < TN; ++j) {
            const char* const t = st + A_BYTES + q * B_BYTES;
            if constexpr (B_KC) b[q][j] = frag_kc<T>(t, (wn * TN + j) * 32, step, lane);
            else b[q][j] = frag_mn<T, BN>(t, (wn * TN + j) * 32, step, lane);
          }
#pragma unroll
        for (int q = 0; q < NB; ++q)
#pragma unroll
          for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) mma(acc[q][i][j], a[i], b[q][j]);
      }
    }
    if (more) {
      deposit(smem + ((kt + 1) & 1) * STAGE);
      __syncthreads();
    }
  }

#pragma unroll
  for (int i = 0; i < TM; ++i) {
    const int r = (wm * TM + i) * 32 + (lane & 31);
    if (r >= rows) continue;
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int n = n0 + (wn * TN + j) * 32 + 8 * q + 4 * (lane >> 5);
        if (n >= p.N) continue;
        const int64_t o = (int64_t)(row0 + r) * p.ldc + n;
        float f[4];
#pragma unroll
        for (int t = 0; t < 4; ++t) f[t] = acc[0][i][j][4 * q + t];
        if constexpr (DUAL) {
          float u[4], h[4];
#pragma unroll
          for (int t = 0; t < 4; ++t) {
            f[t] = pk_to_float<T>(pk_from_float<T>(f[t]));     // g and u are tensors of T
            u[t] = pk_to_float<T>(pk_from_float<T>(acc[NB - 1][i][j][4 * q + t]));
            h[t] = (f[t] / (1.f + expf(-f[t]))) * u[t];
          }
          if (p.O0) store4<T>(reinterpret_cast<T*>(p.O0) + o, f);
          if (p.O1) store4<T>(reinterpret_cast<T*>(p.O1) + o, u);
          store4<T>(reinterpret_cast<T*>(p.O2) + o, h);
        } else {
          store4<T>(reinterpret_cast<T*>(p.O0) + o, f);
        }
      }
  }
}

template <typename T, bool B_KC, bool DUAL>
inline int launch_ragged_m(RaggedM p, int64_t A_rows, int cus, int kernel_id, hipStream_t s) {
  // 128 x 128 tiles once they give every CU work for two rounds; below that the chip is filled by
  // four times as many 64 x 64 tiles
  const int64_t big = (A_rows / 128 + (p.E + 1) / 2) * pk_ceil_div(p.N, 128);
  const bool large = big >= 2 * (int64_t)cus;
  const int64_t bm = large ? 128 : 64;
  p.n_tiles = (int32_t)pk_ceil_div(p.N, bm);
  const int64_t units = (pk_ceil_div(A_rows, bm) + p.E) * p.n_tiles;
  if (units > 0x7fffff00ll) return PK_ERR_SHAPE;
  const dim3 grid((unsigned)(pk_ceil_div(units, 4 * NXCD) * 4 * NXCD)), block(THREADS);
  if (large) PK_LAUNCH_NOCHECK(kernel_id, s, (ragged_m_kernel<T, 2, 2, B_KC, DUAL>), grid, block, 0, s, p);
  else PK_LAUNCH_NOCHECK(kernel_id, s, (ragged_m_kernel<T, 1, 1, B_KC, DUAL>), grid, block, 0, s, p);
  PK_RETURN_IF_LAUNCH_FAILED();
  return PK_OK;
}

// ---------------------------------------------------------------------------------- ragged K
struct RaggedKProblem {
  const void* A; int64_t lda; const int32_t* a_map;
  const void* B; int64_t ldb; const int32_t* b_map;
  void* C;                  // [E][M][N]
  int32_t M, N;
};
struct RaggedK {
  RaggedKProblem prob[3];
  int32_t first[4];         // first tile of problem q within an expert's tiles; first[nprob] = all of them
  int32_t nprob;
  const int32_t* starts;
  int32_t E, map_div, accumulate;
};

template <typename T, int TM, int TN>
__global__ __launch_bounds__(THREADS) void ragged_k_kernel(const RaggedK p) {
  constexpr int BM = 64 * TM, BN = 64 * TN, BK = kBK<T>, PIECE = kPiece<T>;
  constexpr int LA = BM * 8 / THREADS, LB = BN * 8 / THREADS;
  constexpr int A_BYTES = BM * 128, STAGE = A_BYTES + BN * 128;
  using MA = Mn<T, BM>;
  using MB = Mn<T, BN>;
  __shared__ __attribute__((aligned(16))) char smem[2 * STAGE];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave >> 1, wn = wave & 1;
  const int per_expert = p.first[p.nprob];
  const int unit = unit_of_block(blockIdx.x);
  if (unit >= p.E * per_expert) return;
  const int e = unit / per_expert;
  int t = unit - e * per_expert, which = 0;
  while (which + 1 < p.nprob && t >= p.first[which + 1]) ++which;
  t -= p.first[which];
  const RaggedKProblem& q = p.prob[which];
  const int n_tiles = (q.N + BN - 1) / BN;
  const int m0 = t / n_tiles * BM, n0 = t % n_tiles * BN;
  const int row0 = p.starts[e], rows = p.starts[e + 1] - row0;
  const int nkt = (rows + BK - 1) / BK;

  int a_k[LA], b_k[LB], a_col[LA], b_col[LB];
#pragma unroll
  for (int i = 0; i < LA; ++i) {
    const int s = tid + i * THREADS;
    a_k[i] = s / MA::CPR;
    a_col[i] = m0 + (s % MA::CPR) * PIECE;
  }
#pragma unroll
  for (int i = 0; i < LB; ++i) {
    const int s = tid + i * THREADS;
    b_k[i] = s / MB::CPR;
    b_col[i] = n0 + (s % MB::CPR) * PIECE;
  }
  // operand rows of a k-tile (-1: past the expert's rows or the operand's columns), looked up one
  // tile before its pieces are fetched
  int a_row[LA], b_row[LB];
  auto lookup = [&](int kt) {
#pragma unroll
    for (int i = 0; i < LA; ++i) {
      const int k = kt * BK + a_k[i];
      a_row[i] = -1;
      if (k < rows && a_col[i] < q.M) a_row[i] = q.a_map ? q.a_map[row0 + k] / p.map_div : row0 + k;
    }
#pragma unroll
    for (int i = 0; i < LB; ++i) {
      const int k = kt * BK + b_k[i];
      b_row[i] = -1;
      if (k < rows && b_col[i] < q.N) b_row[i] = q.b_map ? q.b_map[row0 + k] / p.map_div : row0 + k;
    }
  };
  u32x4_t ra[LA], rb[LB];
  auto fetch = [&]() {
    const u32x4_t zero = {0u, 0u, 0u, 0u};
#pragma unroll
    for (int i = 0; i < LA; ++i) {
      ra[i] = zero;
      if (a_row[i] >= 0) ra[i] = *reinterpret_cast<const u32x4_t*>(reinterpret_cast<const T*>(q.A) + (int64_t)a_row[i] * q.lda + a_col[i]);
    }
#pragma unroll
    for (int i = 0; i < LB; ++i) {
      rb[i] = zero;
      if (b_row[i] >= 0) rb[i] = *reinterpret_cast<const u32x4_t*>(reinterpret_cast<const T*>(q.B) + (int64_t)b_row[i] * q.ldb + b_col[i]);
    }
  };
  auto deposit = [&](char* st) {
#pragma unroll
    for (int i = 0; i < LA; ++i) {
      const int s = tid + i * THREADS, c = s % MA::CPR;
      *reinterpret_cast<u32x4_t*>(st + a_k[i] * (MA::CPR * 16) + ((c ^ MA::swz(a_k[i])) << 4)) = ra[i];
    }
#pragma unroll
    for (int i = 0; i < LB; ++i) {
      const int s = tid + i * THREADS, c = s % MB::CPR;
      *reinterpret_cast<u32x4_t*>(st + A_BYTES + b_k[i] * (MB::CPR * 16) + ((c ^ MB::swz(b_k[i])) << 4)) = rb[i];
    }
  };

  floatx16_t acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;

  if (nkt > 0) {
    lookup(0);
    fetch();
    lookup(1);
    deposit(smem);
    __syncthreads();
    for (int kt = 0; kt < nkt; ++kt) {
      const char* const st = smem + (kt & 1) * STAGE;
      const bool more = kt + 1 < nkt;
      if (more) {
        fetch();
        lookup(kt + 2);
      }
#pragma unroll
      for (int step = 0; step < 4; ++step) {
        Frag<T> a[TM], b[TN];
#pragma unroll
        for (int i = 0; i < TM; ++i) a[i] = frag_mn<T, BM>(st, (wm * TM + i) * 32, step, lane);
#pragma unroll
        for (int j = 0; j < TN; ++j) b[j] = frag_mn<T, BN>(st + A_BYTES, (wn * TN + j) * 32, step, lane);
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int j = 0; j < TN; ++j) mma(acc[i][j], a[i], b[j]);
      }
      if (more) {
        deposit(smem + ((kt + 1) & 1) * STAGE);
        __syncthreads();
      }
    }
  } else if (p.accumulate) {
    return;                       // an expert without rows adds nothing
  }

  T* const C = reinterpret_cast<T*>(q.C) + (int64_t)e * q.M * q.N;
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    const int m = m0 + (wm * TM + i) * 32 + (lane & 31);
    if (m >= q.M) continue;
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int n = n0 + (wn * TN + j) * 32 + 8 * v + 4 * (lane >> 5);
        if (n >= q.N) continue;
        T* const c = C + (int64_t)m * q.N + n;
        float f[4];
#pragma unroll
        for (int x = 0; x < 4; ++x) f[x] = acc[i][j][4 * v + x];
        if (p.accumulate) {
          float old[4];
          load4<T>(c, old);
#pragma unroll
          for (int x = 0; x < 4; ++x) f[x] += old[x];
        }
        store4<T>(c, f);
      }
  }
}

template <typename T>
inline int launch_ragged_k(RaggedK p, int cus, int kernel_id, hipStream_t s) {
  auto plan = [&](int bm) {
    int64_t tiles = 0;
    for (int q = 0; q < p.nprob; ++q) {
      p.first[q] = (int32_t)tiles;
      tiles += pk_ceil_div(p.prob[q].M, bm) * pk_ceil_div(p.prob[q].N, bm);
    }
    p.first[p.nprob] = (int32_t)tiles;
    return tiles * p.E;
  };
  int64_t units = plan(128);
  const bool large = units >= 2 * (int64_t)cus;      // as for the ragged-M tiles
  if (!large) units = plan(64);
  if (units > 0x7fffff00ll) return PK_ERR_SHAPE;
  if (units == 0) return PK_OK;
  const dim3 grid((unsigned)(pk_ceil_div(units, 4 * NXCD) * 4 * NXCD)), block(THREADS);
  if (large) PK_LAUNCH_NOCHECK(kernel_id, s, (ragged_k_kernel<T, 2, 2>), grid, block, 0, s, p);
  else PK_LAUNCH_NOCHECK(kernel_id, s, (ragged_k_kernel<T, 1, 1>), grid, block, 0, s, p);
  PK_RETURN_IF_LAUNCH_FAILED();
  return PK_OK;
}

}  // namespace pk_tile
