// Grouped GEMMs on the matrix cores for what the 256-wide bf16 kernels of grouped_gemm.hip do not
// take or are too coarse for: fp32 operands (v_mfma_f32_32x32x2_f32: exact fp32 products and sums), bf16
// widths that are no multiple of 128 (256 for weight gradients), and products with few tiles.  Every row
// only has to be a whole number of 16-byte pieces (4 fp32 or 8 bf16 elements); rows and columns past the ends are read from a
// tile's first ones and never stored, reduction remainders are cleared on their way into LDS.
//
//   ragged M: C[rows_e, N] = sum_seg A_seg[rows_e, K] . B_seg[e]     (forward, input gradient)
//   ragged K: C[e][M, N] (+)= A[rows_e, M]^T . B[rows_e, N]           (weight gradient)
//
// One workgroup per output tile: four waves (2 x 2) for tiles of 64 x 64 or 128 x 128, two (2 x 1) for the
// 64 x 32 tiles that fp32 ragged-M products take where 64 x 64 ones leave CUs idle.  A k-tile is 128 bytes
// of the reduction index of every operand row (32 fp32 or 64 bf16); two k-tiles are in flight in
// registers while another is multiplied out of LDS; two LDS buffers, one barrier per
// k-tile.  The operands pass through registers rather than straight into LDS because the masking then
// costs one select per piece and nothing has to be counted by hand.  Where the tiles are too few for
// the chip, several groups of waves share a tile's reduction.
//
// What the k-loops wait for.  No load stands behind a branch (addresses are clamped, the last k-tile is masked on its way into
// LDS), the loop has one way out, and the k-tiles behind it have code of their own: then the compiler knows how
// many loads are younger than the ones it needs.  With the loads behind masks it waited for all of them (vmcnt(0)) in every
// second or third k-tile, so that nothing was in flight across it; three workgroups on a CU hid most of that in the ragged-M
// products, but not in the weight gradients, whose reductions are short.  Measured, caches cold, us, before -> now:
//   weight gradients, bf16: 24 experts 1000 x 360, 172 rows 44.1 -> 32.5; 32 experts 1024 x 512, 128 rows 56.6 -> 42.8 (64-wide
//   tiles 70.0 -> 52); fp32: 16 experts 512 x 256, 250 rows 53.8 -> 42.4; 32 experts 1024 x 512, 128 rows 182 -> 154
//   down 32 experts 512 -> 1024, 128 rows 17.4 -> 15.0; d_x 24 experts 1000 x 360, 172 rows 26.6 -> 24.7; gate/up 128 experts
//   2048 x 768, 32 rows 184 -> 170, 24 experts 1000 x 360 27.3 -> 26.0, fp32 32 experts 1024 x 512 119 -> 113
// Three k-tiles in flight, or the fragments of all four steps at once, cost a workgroup per CU (188 registers instead of
// 144 in gate/up): 24 experts 1000 x 360, down 14.5 -> 16.0, 32 experts 1024 x 512, weight gradients in 64-wide tiles 52 -> 62.
// What is left in a k-tile of the 64 x 64 kernels: without their loads 0.6 us, without their LDS reads 0.7, together 0.85.
// Against one 64 x 64 FMA tile per workgroup (simt_gemm.h, which keeps the widths that are no multiple
// of 16 bytes): see the figures at tile_gemm_ok in grouped_gemm.hip.
#pragma once
#include "pk_common.h"
#include "launch_rules.h"
#include "unit_index.h"
#include <type_traits>

namespace pk_tile {

constexpr int NXCD = pk_rules::NXCD, CUS = 256;

typedef short shortx4_t __attribute__((ext_vector_type(4)));
typedef short shortx8_t __attribute__((ext_vector_type(8)));

template <typename T> constexpr int kBK = 128 / (int)sizeof(T);      // reduction depth of a k-tile
template <typename T> constexpr int kPiece = 16 / (int)sizeof(T);    // elements of a 16-byte piece
constexpr int DEPTH = 2;      // k-tiles in flight in registers
constexpr int AHEAD = 2;      // steps of a k-tile whose fragments are in registers or on their way there

// ---- LDS tiles, in 16-byte pieces, XOR-swizzled against bank conflicts (both are X * 128 bytes):
// KC: [X rows of the M or N index][8 pieces along k];  piece c of row r sits at c ^ ((r >> 1) & 7)
// MN: [BK k][X columns of the M or N index];            piece c of k-row k sits at c ^ swz(k)
template <typename T, int X>
struct Mn {
  static constexpr int CPR = X * (int)sizeof(T) / 16;
  __device__ static __forceinline__ int swz(int k) {
    // the transposing read of bf16 takes four k-rows at once: spread them over the banks
    if (sizeof(T) == 4) return 0;
    return CPR >= 16 ? (k & 3) << 2 : CPR >= 8 ? (k & 1) << 2 : 0;
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
// (fp32: the four MFMAs of a piece go round the tiles, so that neighbours do not share an accumulator)
template <int TM, int TN>
__device__ __forceinline__ void mma_tiles(floatx16_t (&acc)[TM][TN], const Frag<bf16_t> (&a)[TM], const Frag<bf16_t> (&b)[TN]) {
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(b[j].v, a[i].v, acc[i][j], 0, 0, 0);
}
template <int TM, int TN>
__device__ __forceinline__ void mma_tiles(floatx16_t (&acc)[TM][TN], const Frag<float> (&a)[TM], const Frag<float> (&b)[TN]) {
#pragma unroll
  for (int q = 0; q < 4; ++q)
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(b[j].v[q], a[i].v[q], acc[i][j], 0, 0, 0);
}

// a 16-byte piece of a row, as floats
template <typename T>
__device__ __forceinline__ void load_piece(const T* p, float (&f)[kPiece<T>]) {
  if constexpr (sizeof(T) == 4) {
    const floatx4_t v = *reinterpret_cast<const floatx4_t*>(p);
#pragma unroll
    for (int i = 0; i < 4; ++i) f[i] = v[i];
  } else {
    const bf16x8_t v = *reinterpret_cast<const bf16x8_t*>(p);
#pragma unroll
    for (int i = 0; i < 8; ++i) f[i] = (float)v[i];
  }
}
template <typename T>
__device__ __forceinline__ void store_piece(T* p, const float (&f)[kPiece<T>]) {
  if constexpr (sizeof(T) == 4) {
    *reinterpret_cast<floatx4_t*>(p) = floatx4_t{f[0], f[1], f[2], f[3]};
  } else {
    bf16x8_t v;
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = (bf16_t)f[i];
    *reinterpret_cast<bf16x8_t*>(p) = v;
  }
}

// The way of a product from the accumulators to memory: the waves put 32 rows each into LDS as fp32 [rows][X],
// then every thread of the workgroup takes 16-byte pieces of T of it, neighbours along a row.  Straight from
// the accumulators a store covers 16 bytes in each of 32 rows, and every 128-byte line is opened eight times
// (weight gradients of 512 tokens, 1536 x 384, 64 experts 101 -> 76 us, d_h of 4,096 tokens, 512 x 256, 16 experts 33 -> 27).
// 16-byte units of a row are XOR-ed with the row against bank conflicts.
template <int X>
__device__ __forceinline__ void stage_acc(float* lds, int row, int col, const float* four) {
  *reinterpret_cast<floatx4_t*>(lds + row * X + (((col >> 2) ^ (row & (X / 4 - 1))) << 2)) = floatx4_t{four[0], four[1], four[2], four[3]};
}
template <int X, int N>
__device__ __forceinline__ void staged(const float* lds, int row, int col, float (&f)[N]) {
#pragma unroll
  for (int h = 0; h < N / 4; ++h) {
    const floatx4_t v = *reinterpret_cast<const floatx4_t*>(lds + row * X + ((((col >> 2) + h) ^ (row & (X / 4 - 1))) << 2));
#pragma unroll
    for (int i = 0; i < 4; ++i) f[4 * h + i] = v[i];
  }
}

// f(std::integral_constant<int, 0>{}), ..., f(std::integral_constant<int, N - 1>{})
template <int N, int I = 0, typename F>
__device__ __forceinline__ void static_for(F&& f) {
  if constexpr (I < N) {
    f(std::integral_constant<int, I>{});
    static_for<N, I + 1>(f);
  }
}

// The k-loop of a tile: fetch(set) requests the k-tile of that number into the register set of that number, step(set, kt, more)
// multiplies k-tile kt out of it and, with `more`, requests k-tile kt + DEPTH into it.  Exactly the k-tiles that are there are
// requested: an expert with one or two of them is bound by the memory's answer to these.  The loop has nothing to skip and one way
// out, and whatever leads to a step has requested the same number of tiles behind its own: the compiler's counts depend on both.
// us, one loop that always requests DEPTH tiles more -> this, each launch behind a fill of 640 MB: weight gradients 24 experts 1000 x 360, 8 rows 28.4 ->
// 26.1 (rows not gathered 26.5 -> 25.0), 32 rows 28.8 -> 27.1, 172 rows 42.2 -> 40.2; 32 experts 1000 x 512, uneven rows not gathered,
// 8 38.7 -> 34.6, 64 49.1 -> 47.0; fp32 32 experts 1024 x 512, 16 rows 73.7 -> 70.2; 24 experts 1000 x 360, 96 rows 88.1 -> 84.7.  bf16 in
// 64 x 64 tiles: d_x 24 experts 1000 x 360, 8 rows 19.8 -> 18.9, 96 rows 26.6 -> 25.6; gate/up 172 rows 37.6 -> 35.8; d_h 32 experts
// 1000 x 512, 24 uneven rows 24.4 -> 23.4.  The launch bounds keep the waves on a SIMD: without them the 128 x 128 weight gradients
// have one (36 us at the first of these sizes).
template <typename Fetch, typename Step>
__device__ __forceinline__ void run_k_tiles(int n, Fetch&& fetch, Step&& step) {
  static_assert(DEPTH == 2, "the rounds below");
  constexpr std::integral_constant<int, 0> s0{};
  constexpr std::integral_constant<int, 1> s1{};
  if (n > 1) {
    fetch(s0);
    __builtin_amdgcn_sched_barrier(0);         // in this order
    fetch(s1);
    __builtin_amdgcn_sched_barrier(0);
    int kt = 0;
    for (; kt + 3 < n; kt += 2) {
      step(s0, kt, true);
      step(s1, kt + 1, true);
    }
    if (kt + 3 == n) {
      step(s0, kt, true);
      step(s1, kt + 1, false);
      step(s0, kt + 2, false);
    } else {
      step(s0, kt, false);
      step(s1, kt + 1, false);
    }
  } else if (n == 1) {
    fetch(s0);
    step(s0, 0, false);
  }
}

// acc of group 0 += acc of the other groups, in group order (every thread of the workgroup calls it).
template <int KS, int TILES, int THREADS>
__device__ __forceinline__ void add_groups(floatx16_t* acc, float* lds, int group, int tid) {
  __syncthreads();                         // the last k-tiles have been read
  if (group > 0) {
#pragma unroll
    for (int t = 0; t < TILES; ++t)
#pragma unroll
      for (int v = 0; v < 16; ++v) lds[(((group - 1) * TILES + t) * 16 + v) * THREADS + tid] = acc[t][v];
  }
  __syncthreads();
  if (group == 0) {
#pragma unroll
    for (int g = 1; g < KS; ++g)
#pragma unroll
      for (int t = 0; t < TILES; ++t)
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[t][v] += lds[(((g - 1) * TILES + t) * 16 + v) * THREADS + tid];
  }
}
// Groups of four waves per output tile: few tiles leave most CUs idle and a long reduction on the
// others, so it is split inside the workgroup (up to four ways, at least four k-tiles each).
inline int reduction_groups(int64_t tiles, int64_t k_tiles, int cus) {
  int ks = 1;
  while (ks < 4 && tiles * ks * 2 <= 2 * (int64_t)cus && k_tiles >= ks * 2 * 2) ks *= 2;
  return ks;
}

// ---------------------------------------------------------------------------------- ragged M
struct RaggedM {
  const void* A0;           // A of k-segment 0, row-major [rows, lda]
  const void* A1;           // k-segment 1 (nseg == 2)
  int64_t lda;
  const int32_t* row_map;   // optional gather: A row = row_map[sorted row] / map_div
  pk_units::FastDiv map_div;
  const void* B0;           // weights of k-segment 0 (DUAL: gate)
  const void* B1;           // weights of k-segment 1 (DUAL: up)
  int64_t ldb, strideB;     // row stride, elements between experts
  const int32_t* starts;
  int32_t E, K, nseg, N;
  int32_t n_tiles;
  void* O0;                 // C;  GATE_UP: g (optional);  BWD, BWD_SCALED: d_g
  void* O1;                 //     GATE_UP: u (optional);  BWD, BWD_SCALED: d_u
  void* O2;                 //     GATE_UP: h = silu(g) * u;  BWD_SCALED: score * h
  int64_t ldc;
  const void* Gin;          // BWD, BWD_SCALED: g and u of the forward [rows, ldc]
  const void* Uin;
  int32_t hw_sigmoid;       // GATE_UP, bf16: hardware exponential and reciprocal, as the persistent kernels form h
  const float* scores;      // BWD_SCALED: score of every routed slot (row_map names the slot of a sorted row)
  float* ds_part;           // BWD_SCALED: [column tiles][total_rows]: the score gradient in parts
  int64_t total_rows;
};

// Tile b of a launch.  Blocks b, b + 8, ... run on one XCD: CHUNK neighbouring tiles (which share
// weights or rows) stay on it, the next ones go to the next XCD (16 against 4: -3 to -12 % where the
// operands do not fit the L2 of an XCD; 32 leaves XCDs without work at small sizes).
constexpr int CHUNK = 16;
__device__ __forceinline__ int unit_of_block(int b) {
  const int x = b % NXCD, q = b / NXCD;
  return ((q / CHUNK) * NXCD + x) * CHUNK + (q % CHUNK);
}

// What happens to the product.
// GATE_UP: two weight matrices (gate and up) against the same A rows, SiLU(g) * u.
// BWD: the product is d_h; d_g = d_h * u * silu'(g), d_u = d_h * silu(g).
// BWD_SCALED: the A rows are rows of d_out (gathered), the product is d_h before the routed row's score:
// d_g and d_u from score * d_h, score * h for the weight gradient, and the row sums of d_h * h over a
// tile's columns, whose total is the score's gradient.  d_h never leaves the workgroup.
enum Epilogue { PLAIN = 0, GATE_UP = 1, BWD = 2, BWD_SCALED = 3 };
// SPARSE (fp32): at least half of a tile's rows are not there, about.  They are left out of the loads, which then stand behind
// branches: the compiler still knows of the weights' loads behind them.  Read from the tile's first row instead, as everywhere else,
// they take up the path to the registers and a long fp32 reduction with few rows is 5 to 17 % slower (us, all rows read -> this: 24
// experts 1000 x 360, 8 rows: gate/up 49.0 -> 45.4, d_h 26.2 -> 25.1, d_x 34.2 -> 33.3; 32 experts 1024 x 512, 16 rows, d_x 59.8 -> 53.7; 64 experts
// 896 x 384, 16 rows, gate/up 83.7 -> 81.3, d_x 81.3 -> 78.2).  With more rows the branches cost as much (24 experts 1000 x 360, 48 rows,
// gate/up 51.4 -> 54.7; 128 experts 512 x 128, 48 uneven rows, d_x 41.9 -> 48.6), with fewer than twelve k-tiles there is little to
// gain (128 experts 512 x 128, 32 rows, down 20.0 -> 21.1), and with more tiles than fit the CUs at once nothing (figures at
// absent_rows_left_out); the 32 x 32 tiles gain in d_h alone (24 experts 1000 x 360, 8 rows 26.0 -> 25.1; 16 experts 408 x 472, 16 rows,
// d_x 19.8 -> 20.6).
// Gate and up of more tiles than CUs wait for all of a round's k-tiles before they ask for the next ones, which masked loads did by
// themselves: where some CUs have two tiles and others one, requests that run ahead make these wait (us, without -> this, r rows an
// expert: 24 experts 2048 x 384, r 8, 83 -> 75, masked 71; 1024 x 384 46.5 -> 44, 42; 1000 x 360 45.3 -> 43.5, 42; 40 experts 1024 x 256, r 8,
// 43.8 -> 42.2; 64 experts 1536 x 384, r 24, 133.8 -> 129.8; 128 experts 512 x 256, uneven r 24, 75.3 -> 73.2).  With a tile for every CU
// at most it costs as much (24 experts 1000 x 256, r 8, 30.2 -> 32.1; 12 experts 1000 x 360 29.0 -> 30.2), and 64 x 64 tiles in two groups
// lose (32 experts 1024 x 512, uneven r 24, 89.4 -> 96.8).
template <typename T, int WM, int WN, int TM, int TN, int KS, bool B_KC, int EPI, bool SPARSE>
__global__ __launch_bounds__(64 * WM * WN * KS, (sizeof(T) == 4 && !SPARSE) || WM * WN < 4 || KS > 1 || TM * TN > 1 ? 1 : EPI == GATE_UP ? 3 : 4)
void ragged_m_kernel(const RaggedM p) {
  constexpr int THREADS = 64 * WM * WN;       // of a group: WM x WN waves of TM x TN MFMA tiles
  constexpr int BM = 32 * WM * TM, BN = 32 * WN * TN, BK = kBK<T>, PIECE = kPiece<T>;
  constexpr bool DUAL = EPI == GATE_UP;
  constexpr int NB = DUAL ? 2 : 1;
  // run_k_tiles in bf16 with 64 x 64 tiles; the longer code costs the others registers, and with them a workgroup on a CU or spills
  constexpr bool EXACT = sizeof(T) == 2 && TM * TN == 1;
  constexpr int LA = BM * 8 / THREADS, LB = BN * 8 / THREADS;
  constexpr int A_BYTES = BM * 128, B_BYTES = BN * 128, STAGE = A_BYTES + NB * B_BYTES;
  static_assert(!DUAL || B_KC, "gate and up weights are K-contiguous");
  static_assert((KS - 1) * NB * BM * BN * 4 <= KS * 2 * STAGE, "the partial sums reuse the k-tiles' LDS");
  __shared__ __attribute__((aligned(16))) char smem_[KS * 2 * STAGE];

  // KS groups of four waves take every KS-th k-tile each, in LDS of their own
  const int group = __builtin_amdgcn_readfirstlane((int)threadIdx.x / THREADS);
  const int tid = threadIdx.x % THREADS, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / WN, wn = wave % WN;
  char* const smem = smem_ + group * 2 * STAGE;
  const pk_units::UnitIndex ui = pk_units::build_unit_index<BM>(p.starts, p.E, p.n_tiles);
  const int unit = unit_of_block(blockIdx.x);
  if (unit >= ui.total) return;
  int e, mt, nt;
  pk_units::locate_unit<BM>(ui, pk_units::as_const(p.starts), p.E, p.n_tiles, unit, e, mt, nt);
  const int row0 = p.starts[e] + mt * BM;
  const int rows = min(BM, p.starts[e + 1] - row0);
  const int n0 = nt * BN;

  // The thread's A rows (fixed over the reduction) and B rows or columns.  Rows past the expert's end and columns
  // past N read the tile's first ones instead: what comes of them is stored nowhere.  Only the reduction index
  // is masked, on the way into LDS, so that no load stands behind a branch: the compiler then counts the loads in
  // flight, where a branch around one makes it wait for all of them.
  const T* a_ptr[LA];
  const T* b_ptr[LB];
  int b_k[LB];                       // MN weights: k-row of the piece inside a k-tile
  const int a_kofs = (tid & 7) * PIECE;
#pragma unroll
  for (int i = 0; i < LA; ++i) {
    const int r = (tid + i * THREADS) >> 3;
    int64_t src = row0 + (r < rows ? r : 0);
    if (p.row_map) src = pk_units::fastdiv(p.row_map[src], p.map_div);
    a_ptr[i] = reinterpret_cast<const T*>(p.A0) + src * p.lda + a_kofs;
  }
  const T* const B = reinterpret_cast<const T*>(p.B0) + (int64_t)e * p.strideB;
#pragma unroll
  for (int i = 0; i < LB; ++i) {
    const int s = tid + i * THREADS;
    if (B_KC) {
      const int n = n0 + (s >> 3);
      b_k[i] = a_kofs;
      b_ptr[i] = B + (int64_t)(n < p.N ? n : n0) * p.ldb + a_kofs;
    } else {
      b_k[i] = s / Mn<T, BN>::CPR;
      const int n = n0 + (s % Mn<T, BN>::CPR) * PIECE;
      b_ptr[i] = B + (int64_t)b_k[i] * p.ldb + (n < p.N ? n : n0);
    }
  }
  const int64_t seg_a = reinterpret_cast<const T*>(p.A1) - reinterpret_cast<const T*>(p.A0);
  const int64_t seg_b = reinterpret_cast<const T*>(p.B1) - reinterpret_cast<const T*>(p.B0);
  const int kt_per_seg = (p.K + BK - 1) / BK, nkt = kt_per_seg * p.nseg;

  // k-tile kt into register set d: what lies past K, or past the last tile, is read from the start of the
  // reduction and masked by deposit()
  u32x4_t ra_[DEPTH][LA], rb_[DEPTH][NB][LB];
  if constexpr (SPARSE) {
#pragma unroll
    for (int d = 0; d < DEPTH; ++d)
#pragma unroll
      for (int i = 0; i < LA; ++i) ra_[d][i] = u32x4_t{0u, 0u, 0u, 0u};
  }
  auto fetch = [&](auto d_c, int kt) {
    auto& ra = ra_[decltype(d_c)::value];
    auto& rb = rb_[decltype(d_c)::value];
    kt = kt < nkt ? kt : 0;
    const bool second = kt >= kt_per_seg;
    const int k0 = (second ? kt - kt_per_seg : kt) * BK;
    const int64_t sa = second ? seg_a : 0, sb = second ? seg_b : 0;
    const int ka = k0 + a_kofs < p.K ? k0 : -a_kofs;
#pragma unroll
    for (int i = 0; i < LA; ++i)
      if (!SPARSE || ((tid + i * THREADS) >> 3) < rows) ra[i] = *reinterpret_cast<const u32x4_t*>(a_ptr[i] + (sa + ka));
#pragma unroll
    for (int q = 0; q < NB; ++q)
#pragma unroll
      for (int i = 0; i < LB; ++i) {
        const int64_t kb = B_KC ? (int64_t)ka : (int64_t)(k0 + b_k[i] < p.K ? k0 : -b_k[i]) * p.ldb;
        rb[q][i] = *reinterpret_cast<const u32x4_t*>(b_ptr[i] + (DUAL ? (q ? seg_b : 0) : sb) + kb);
      }
  };
  auto deposit = [&](auto d_c, int kt, char* st) {
    auto& ra = ra_[decltype(d_c)::value];
    auto& rb = rb_[decltype(d_c)::value];
    // reduction elements left from this tile on (both operands are masked: zero times infinity is not zero)
    const int left = kt >= nkt ? 0 : p.K - (kt >= kt_per_seg ? kt - kt_per_seg : kt) * BK;
    if (left < BK) {
      const u32x4_t zero = {0u, 0u, 0u, 0u};
#pragma unroll
      for (int i = 0; i < LA; ++i) ra[i] = a_kofs < left ? ra[i] : zero;
#pragma unroll
      for (int q = 0; q < NB; ++q)
#pragma unroll
        for (int i = 0; i < LB; ++i) rb[q][i] = b_k[i] < left ? rb[q][i] : zero;
    }
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
  const int mine = (nkt + KS - 1) / KS;      // k-tiles of a group (past the last one: zeros)
  // DEPTH of the group's k-tiles are in flight, each in a register set of its own
  auto step = [&](auto d_c, int kt, bool more) {
    char* const st = smem + (EXACT ? decltype(d_c)::value : kt & 1) * STAGE;
    deposit(d_c, kt * KS + group, st);
    __syncthreads();
    if (more) fetch(d_c, (kt + DEPTH) * KS + group);
    if (wave_has_rows) {
      Frag<T> a[AHEAD][TM], b[AHEAD][NB][TN];
      auto read = [&](int step) {
#pragma unroll
        for (int i = 0; i < TM; ++i) a[step % AHEAD][i] = frag_kc<T>(st, (wm * TM + i) * 32, step, lane);
#pragma unroll
        for (int q = 0; q < NB; ++q)
#pragma unroll
          for (int j = 0; j < TN; ++j) {
            const char* const t = st + A_BYTES + q * B_BYTES;
            if constexpr (B_KC) b[step % AHEAD][q][j] = frag_kc<T>(t, (wn * TN + j) * 32, step, lane);
            else b[step % AHEAD][q][j] = frag_mn<T, BN>(t, (wn * TN + j) * 32, step, lane);
          }
      };
#pragma unroll
      for (int step = 0; step < AHEAD - 1; ++step) read(step);
#pragma unroll
      for (int step = 0; step < 4; ++step) {
        if (step + AHEAD - 1 < 4) read(step + AHEAD - 1);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int q = 0; q < NB; ++q) mma_tiles<TM, TN>(acc[q], a[step % AHEAD], b[step % AHEAD][q]);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  };
  if constexpr (EXACT) {
    run_k_tiles(mine, [&](auto d) { fetch(d, d * KS + group); }, step);
  } else if (mine > 0) {
    static_for<DEPTH>([&](auto d) {
      fetch(d, d * KS + group);
      __builtin_amdgcn_sched_barrier(0);       // in this order: the counts of loads in flight depend on it
    });
    int kt = 0;
    const bool in_step = SPARSE && EPI == GATE_UP && (KS == 1 || WM * WN < 4) && ui.total > CUS;
    for (; kt + DEPTH <= mine; kt += DEPTH) {  // nothing to skip and one way out, for the counts' sake too
      if (in_step) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      static_for<DEPTH>([&](auto d) { step(d, kt + d, true); });
    }
    static_for<DEPTH - 1>([&](auto d) { if (kt + d < mine) step(d, kt + d, false); });
  }
  if constexpr (KS > 1) {
    add_groups<KS, NB * TM * TN, THREADS>(reinterpret_cast<floatx16_t*>(&acc), reinterpret_cast<float*>(smem_), group, tid);
  }

  constexpr int CHUNK_ROWS = 32 * WM, ROW_PIECES = BN / PIECE, ALL = THREADS * KS;
  static_assert(NB * CHUNK_ROWS * BN * 4 <= KS * 2 * STAGE, "the staged rows reuse the k-tiles' LDS");
  static_assert(CHUNK_ROWS * ROW_PIECES % 64 == 0 && 64 % ROW_PIECES == 0, "whole waves, a row in one wave");
  float* const lds = reinterpret_cast<float*>(smem_);
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    __syncthreads();                         // the LDS has been read for the last time
    if (group == 0) {
#pragma unroll
      for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
          for (int q = 0; q < 4; ++q)
            stage_acc<BN>(lds + b * CHUNK_ROWS * BN, 32 * wm + (lane & 31), 32 * (wn * TN + j) + 8 * q + 4 * (lane >> 5),
                          reinterpret_cast<const float*>(&acc[b][i][j]) + 4 * q);
    }
    __syncthreads();
    for (int s = threadIdx.x; s < CHUNK_ROWS * ROW_PIECES; s += ALL) {
      const int lr = s / ROW_PIECES, c = (s % ROW_PIECES) * PIECE, n = n0 + c;
      const int r = (lr >> 5) * 32 * TM + 32 * i + (lr & 31);
      const bool live = r < rows && n < p.N;
      const int64_t o = (int64_t)(row0 + r) * p.ldc + n;
      float a[PIECE];
      staged<BN>(lds, lr, c, a);
      if constexpr (EPI == PLAIN) {
        if (live) store_piece<T>(reinterpret_cast<T*>(p.O0) + o, a);
      } else if constexpr (EPI == GATE_UP) {
        float u[PIECE], h[PIECE];
        staged<BN>(lds + CHUNK_ROWS * BN, lr, c, u);
#pragma unroll
        for (int t = 0; t < PIECE; ++t) {
          a[t] = pk_to_float<T>(pk_from_float<T>(a[t]));     // g and u are tensors of T
          u[t] = pk_to_float<T>(pk_from_float<T>(u[t]));
        }
        if (sizeof(T) == 2 && p.hw_sigmoid) {
#pragma unroll
          for (int t = 0; t < PIECE; ++t) h[t] = (a[t] * __builtin_amdgcn_rcpf(1.f + __expf(-a[t]))) * u[t];
        } else {
#pragma unroll
          for (int t = 0; t < PIECE; ++t) h[t] = (a[t] / (1.f + expf(-a[t]))) * u[t];
        }
        if (live) {
          if (p.O0) store_piece<T>(reinterpret_cast<T*>(p.O0) + o, a);
          if (p.O1) store_piece<T>(reinterpret_cast<T*>(p.O1) + o, u);
          store_piece<T>(reinterpret_cast<T*>(p.O2) + o, h);
        }
      } else {
        float ds = 0.f;
        if (live) {
          float g[PIECE], u[PIECE], hs[PIECE];
          load_piece<T>(reinterpret_cast<const T*>(p.Gin) + o, g);
          load_piece<T>(reinterpret_cast<const T*>(p.Uin) + o, u);
          const float sc = EPI == BWD_SCALED ? p.scores[p.row_map[row0 + r]] : 1.f;
#pragma unroll
          for (int t = 0; t < PIECE; ++t) {
            const float sg = 1.f / (1.f + expf(-g[t]));
            const float d = pk_to_float<T>(pk_from_float<T>(sc * a[t]));      // d_h is a tensor of T
            const float hv = (g[t] * sg) * u[t];
            ds += a[t] * hv;
            hs[t] = sc * hv;
            const float d_u = d * (g[t] * sg);
            g[t] = d * u[t] * (sg * (1.f + g[t] * (1.f - sg)));
            u[t] = d_u;
          }
          store_piece<T>(reinterpret_cast<T*>(p.O0) + o, g);
          store_piece<T>(reinterpret_cast<T*>(p.O1) + o, u);
          if (EPI == BWD_SCALED) store_piece<T>(reinterpret_cast<T*>(p.O2) + o, hs);
        }
        if constexpr (EPI == BWD_SCALED) {
#pragma unroll
          for (int off = 1; off < ROW_PIECES; off <<= 1) ds += __shfl_xor(ds, off);
          if (live && c == 0) p.ds_part[(int64_t)nt * p.total_rows + row0 + r] = ds;
        }
      }
    }
  }
}

// *part_cols: columns per part of the score gradient (those of a tile)
template <typename T, int WM, int WN, int TM, int TN, int KS, bool B_KC, int EPI>
inline int launch_tiles(RaggedM p, int64_t A_rows, int* part_cols, int kernel_id, hipStream_t s) {
  constexpr int BM = 32 * WM * TM, BN = 32 * WN * TN;
  p.n_tiles = (int32_t)pk_ceil_div(p.N, BN);
  const int64_t units = (pk_ceil_div(A_rows, BM) + p.E) * p.n_tiles;
  if (units > 0x7fffff00ll) return PK_ERR_SHAPE;
  if (part_cols) *part_cols = BN;
  const dim3 grid((unsigned)(pk_ceil_div(units, CHUNK * NXCD) * CHUNK * NXCD)), block(64 * WM * WN * KS);
  constexpr bool MAY_BE_SPARSE = sizeof(T) == 4 && (WM * WN > 1 || EPI != PLAIN);
  if (MAY_BE_SPARSE && pk_rules::absent_rows_left_out(EPI == GATE_UP, A_rows, p.E, BM, p.n_tiles, pk_ceil_div(p.K, kBK<T>) * p.nseg, CUS))
    PK_LAUNCH_NOCHECK(kernel_id, s, (ragged_m_kernel<T, WM, WN, TM, TN, KS, B_KC, EPI, MAY_BE_SPARSE>), grid, block, 0, s, p);
  else
    PK_LAUNCH_NOCHECK(kernel_id, s, (ragged_m_kernel<T, WM, WN, TM, TN, KS, B_KC, EPI, false>), grid, block, 0, s, p);
  PK_RETURN_IF_LAUNCH_FAILED();
  return PK_OK;
}
// any_order: the sums over k (and the parts of a score gradient) may be ordered otherwise than they are with the tiles that
// the number of 64 x 64 tiles alone selects.  A token with one expert and a normalised score has a gate gradient of zero, and what
// is left of it in floating point is the rounding of that order, in its own layer and in those in front of it: the callers
// keep it for such tokens and for products that know nothing of the router (the forward, the operators one by one).  Without a
// split all of these tiles, and the persistent kernels, add along k in the same order; a split (reduction_groups) moves it.
// few_rows: rows an expert up to which the 64 x 64 tiles are the faster ones however many tiles there are (each
// product's own; the caller says with what it measured).
template <typename T, bool B_KC, int EPI>
inline int launch_ragged_m(const RaggedM& p, int64_t A_rows, int cus, bool any_order, int64_t few_rows, int* part_cols, int kernel_id,
                           hipStream_t s) {
  // 128 x 128 tiles halve what a product reads from LDS per multiplication, and fit a CU once or twice: they need a
  // tile for every CU and some more (bf16, us, 64 x 64 -> 128 x 128: down, 2048 x 1024, 8 experts, 256 rows, 320 tiles
  // 31.3 -> 28.9; 384 rows, 448 tiles 36.1 -> 28.8; 8 experts 2048 x 768, 192 rows, 256 tiles 20.6 -> 20.0;
  // 24 experts 768 x 256, 192 rows, 288 tiles 11.2 -> 12.8), those with the SwiGLU backward half a round more
  // (1536 x 384, 64 experts: 128 rows, 288 tiles 35.8 -> 46.0, 192 rows, 384 tiles 53.4 -> 48.4).
  // Not for the pair of products with the SwiGLU behind it: 128 accumulator registers a wave leave one
  // workgroup to a CU (128 experts 2048 x 768, 32 rows 155 -> 185, 256 rows 402 -> 433), and not in fp32, where the matrix
  // cores are the bound and the finer tiles fill the last round better (16 experts 1024 x 512, 16,384 rows:
  // gate/up 335 -> 435, down 176 -> 215, d_h 197 -> 251, d_x 340 -> 414).
  // Below two tiles for every CU all of them have to fit at once, also where every expert's last one is nearly empty: with
  // uneven counts some CUs are left with a third (64 x 64 -> 128 x 128, even / counts ~ 1 / sqrt(rank): d_x, 32 experts
  // 2048 x 768, 24 rows, 608 tiles at most 45 -> 39 / 47 -> 40, 32 rows, 640 tiles 47 -> 40 / 46 -> 63; 64 experts
  // 1024 x 512, 16 rows 29 -> 26 / 27 -> 26, 32 rows, 640 tiles 28 -> 25 / 29 -> 38; 896 x 384, 64 rows, 672 tiles
  // 31 -> 27 / 32 -> 38; down, 32 experts 2048 x 512, 48 rows, 704 tiles 31 -> 33 / 32 -> 39).  From 128 rows an expert on that
  // last tile weighs less (16 experts 2048 x 1024, 188 rows, 624 tiles: down 49 -> 37, d_x 68 -> 52, skewed).
  if constexpr (sizeof(T) == 2 && EPI != GATE_UP) {
    const int64_t cols = pk_ceil_div(p.N, 128), big = (A_rows / 128 + (p.E + 1) / 2) * cols;
    const int64_t most = (A_rows / 128 + (A_rows < p.E ? A_rows : p.E)) * cols;
    const bool fill = EPI == PLAIN ? 4 * big >= 5 * (int64_t)cus && (big >= 2 * (int64_t)cus || A_rows >= 128 * p.E || 5 * most <= 12 * (int64_t)cus)
                                   : 4 * big >= 6 * (int64_t)cus;
    if (EPI == BWD_SCALED && !any_order ? big >= 2 * (int64_t)cus : A_rows > few_rows * p.E && fill)
      return launch_tiles<T, 2, 2, 2, 2, 1, B_KC, EPI>(p, A_rows, part_cols, kernel_id, s);
  }
  // row tiles that hold rows, about: every expert's last one is half full
  const int64_t row_tiles = A_rows / 64 + (A_rows < p.E ? A_rows : p.E) / 2;
  const int64_t tiles = row_tiles * pk_ceil_div(p.N, 64), k_tiles = pk_ceil_div(p.K, kBK<T>) * p.nseg;
  // An fp32 tile of 64 x 64 is 1,024 cycles of the matrix cores per k-tile, whoever shares it, so the finer tiles win wherever
  // the coarse ones leave CUs without one or a last round nearly empty (us, 64 x 64 with a split reduction where there
  // are CUs for it -> the tile chosen; tiles of 64 x 64 against 256 CUs):
  if constexpr (sizeof(T) == 4) {
    const int64_t rows = A_rows / (A_rows < p.E ? A_rows : p.E);
    //  32 x 32, four groups: 70 tiles, 408 x 472, d_x 23 -> 14; 96 tiles, 1024 x 512, d_h 26 -> 15; 96 tiles,
    //  512 x 256, d_x 16 -> 10; 126 tiles, 704 x 408, d_h 22 -> 18 (64 x 32: 18)
    if (any_order && 8 * tiles <= 3 * (int64_t)cus) return launch_tiles<T, 1, 1, 1, 1, 4, B_KC, EPI>(p, A_rows, part_cols, kernel_id, s);
    //  half as wide: 128 tiles, 1024 x 512, gate/up 44 -> 30, d_h 27 -> 22
    if (2 * tiles <= cus) {
      if (reduction_groups(2 * tiles, k_tiles, cus) > 1) return launch_tiles<T, 2, 1, 1, 1, 2, B_KC, EPI>(p, A_rows, part_cols, kernel_id, s);
      return launch_tiles<T, 2, 1, 1, 1, 1, B_KC, EPI>(p, A_rows, part_cols, kernel_id, s);
    }
    //  half as high, where most of a tile would be padding: 64 experts 896 x 384, 8 rows, 240 tiles, gate/up 73 -> 45, 16 rows, 288
    //  tiles 68 -> 47, d_h 43 -> 28; 64 experts 512 x 256, 8 rows, 320 tiles, down 16 -> 13, d_x 27 -> 19; 128 experts
    //  1024 x 256, 31 rows, 504 tiles, d_h 52 -> 42, but gate/up 83 -> 97; 64 experts 896 x 384, 2 rows, 476 tiles, down 26 -> 31
    //  (the same order as long as the 64 x 64 tiles would take two groups)
    const bool flat = 2 * tiles <= 3 * (int64_t)cus ? rows <= 16 : (EPI == BWD || EPI == BWD_SCALED) && rows <= 32 && tiles <= 2 * (int64_t)cus;
    if (flat && (any_order || reduction_groups(tiles, k_tiles, cus) == 2))
      return launch_tiles<T, 1, 2, 1, 1, 2, B_KC, EPI>(p, A_rows, part_cols, kernel_id, s);
    //  half as wide again, where the CUs would have one or two tiles: 280 tiles, 408 x 472, d_x 47 -> 29, down 26 -> 18;
    //  320 tiles, 1024 x 512, d_h 52 -> 40; 384 tiles, d_x 49 -> 39; but 490 tiles, 408 x 472, down 27 -> 34; gate/up, which
    //  reads twice the weights for its rows, 320 tiles, 1024 x 512 78 -> 83
    if (any_order && EPI != GATE_UP && tiles > cus && 2 * tiles <= 3 * (int64_t)cus && k_tiles >= 4)
      return launch_tiles<T, 2, 1, 1, 1, 2, B_KC, EPI>(p, A_rows, part_cols, kernel_id, s);
  }
  const int ks = reduction_groups(tiles, k_tiles, cus);
  // (fp32 products with so few tiles are on the finer ones above)
  if constexpr (sizeof(T) == 2)
    if (ks == 4) return launch_tiles<T, 2, 2, 1, 1, EPI == GATE_UP ? 2 : 4, B_KC, EPI>(p, A_rows, part_cols, kernel_id, s);
  if (ks == 2) return launch_tiles<T, 2, 2, 1, 1, 2, B_KC, EPI>(p, A_rows, part_cols, kernel_id, s);
  return launch_tiles<T, 2, 2, 1, 1, 1, B_KC, EPI>(p, A_rows, part_cols, kernel_id, s);
}

// ---------------------------------------------------------------------------------- ragged K
struct RaggedKProblem {
  const void* A; int32_t lda;
  const void* B; int32_t ldb;
  const int32_t* map;       // row map of one operand (neither: some map of as many rows all the same, if the launch has one)
  int32_t map_a, map_b;     // which operand's rows are map[row] / map_div
  void* C;                  // [E][M][N]
  int32_t M, N;
};
struct RaggedK {
  RaggedKProblem prob[3];
  int32_t first[4];         // first tile of problem q within an expert's tiles; first[nprob] = all of them
  int32_t nprob;
  const int32_t* starts;
  pk_units::FastDiv map_div;
  int32_t E, accumulate;
};

// TILE: 64-wide (1) or 128-wide (2) tiles.  MAPPED: some operand's rows are gathered.
template <typename T, int TILE, int KS, bool MAPPED>
__global__ __launch_bounds__(256 * KS, TILE == 2 ? 2 : 4) void ragged_k_kernel(const RaggedK p) {
  constexpr int THREADS = 256;
  constexpr int TM = TILE, TN = TILE, BM = 64 * TILE, BN = BM, BK = kBK<T>, PIECE = kPiece<T>;
  constexpr int L = BM * 8 / THREADS;
  constexpr int A_BYTES = BM * 128, STAGE = 2 * A_BYTES;
  using M = Mn<T, BM>;
  __shared__ __attribute__((aligned(16))) char smem_[KS * 2 * STAGE];

  const int group = __builtin_amdgcn_readfirstlane((int)threadIdx.x / THREADS);      // as in ragged_m_kernel
  const int tid = threadIdx.x % THREADS, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave >> 1, wn = wave & 1;
  char* const smem = smem_ + group * 2 * STAGE;
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
  const int nkt = (rows + BK - 1) / BK, mine = (nkt + KS - 1) / KS;

  // The thread's pieces sit at the same k-rows of both operands.  Columns past M or N read the tile's first piece instead
  // and k-rows past the expert's end its first row: no load stands behind a branch (see ragged_m_kernel).
  int k_row[L], a_col[L], b_col[L];
#pragma unroll
  for (int i = 0; i < L; ++i) {
    const int s = tid + i * THREADS, c = (s % M::CPR) * PIECE;
    k_row[i] = s / M::CPR;
    a_col[i] = m0 + (m0 + c < q.M ? c : 0);
    b_col[i] = n0 + (n0 + c < q.N ? c : 0);
  }
  auto source_row = [&](int kt, int i) {
    const int k = kt * BK + k_row[i];
    return row0 + (k < rows ? k : 0);
  };
  // Row map entries of a k-tile.  MAPPED: they are requested one round of the register sets before the tile's pieces, and
  // divided when these are fetched: memory answers in order, so a wait for them waits for nothing still needed in flight.
  int entry_[DEPTH][L];
  auto lookup = [&](auto d_c, int kt) {
#pragma unroll
    for (int i = 0; i < L; ++i) entry_[decltype(d_c)::value][i] = q.map[source_row(kt, i)];
  };
  u32x4_t ra_[DEPTH][L], rb_[DEPTH][L];
  // k-tile kt into register set d; the entries of the tile after it there are requested on the way
  auto fetch = [&](auto d_c, int kt) {
    auto& ra = ra_[decltype(d_c)::value];
    auto& rb = rb_[decltype(d_c)::value];
    int a_row[L], b_row[L];
#pragma unroll
    for (int i = 0; i < L; ++i) {
      a_row[i] = b_row[i] = source_row(kt, i);
      if constexpr (MAPPED) {
        const int r = pk_units::fastdiv(entry_[decltype(d_c)::value][i], p.map_div);
        a_row[i] = q.map_a ? r : a_row[i];
        b_row[i] = q.map_b ? r : b_row[i];
      }
    }
    if constexpr (MAPPED) lookup(d_c, kt + DEPTH * KS);
#pragma unroll
    for (int i = 0; i < L; ++i)
      ra[i] = *reinterpret_cast<const u32x4_t*>(reinterpret_cast<const T*>(q.A) + (int64_t)a_row[i] * q.lda + a_col[i]);
#pragma unroll
    for (int i = 0; i < L; ++i)
      rb[i] = *reinterpret_cast<const u32x4_t*>(reinterpret_cast<const T*>(q.B) + (int64_t)b_row[i] * q.ldb + b_col[i]);
  };
  auto deposit = [&](auto d_c, int kt, char* st) {
    auto& ra = ra_[decltype(d_c)::value];
    auto& rb = rb_[decltype(d_c)::value];
    const int left = rows - kt * BK;
    if (left < BK) {                           // both: zero times infinity is not zero
      const u32x4_t zero = {0u, 0u, 0u, 0u};
#pragma unroll
      for (int i = 0; i < L; ++i) ra[i] = k_row[i] < left ? ra[i] : zero;
#pragma unroll
      for (int i = 0; i < L; ++i) rb[i] = k_row[i] < left ? rb[i] : zero;
    }
#pragma unroll
    for (int i = 0; i < L; ++i) {
      const int c = (tid + i * THREADS) % M::CPR;
      char* const t = st + k_row[i] * (M::CPR * 16) + ((c ^ M::swz(k_row[i])) << 4);
      *reinterpret_cast<u32x4_t*>(t) = ra[i];
      *reinterpret_cast<u32x4_t*>(t + A_BYTES) = rb[i];
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
    auto step = [&](auto d_c, int kt, bool more) {
      char* const st = smem + decltype(d_c)::value * STAGE;
      deposit(d_c, kt * KS + group, st);
      __syncthreads();
      if (more) fetch(d_c, (kt + DEPTH) * KS + group);
      Frag<T> a[AHEAD][TM], b[AHEAD][TN];
      auto read = [&](int step) {
#pragma unroll
        for (int i = 0; i < TM; ++i) a[step % AHEAD][i] = frag_mn<T, BM>(st, (wm * TM + i) * 32, step, lane);
#pragma unroll
        for (int j = 0; j < TN; ++j) b[step % AHEAD][j] = frag_mn<T, BN>(st + A_BYTES, (wn * TN + j) * 32, step, lane);
      };
#pragma unroll
      for (int step = 0; step < AHEAD - 1; ++step) read(step);
#pragma unroll
      for (int step = 0; step < 4; ++step) {
        if (step + AHEAD - 1 < 4) read(step + AHEAD - 1);
        __builtin_amdgcn_sched_barrier(0);
        mma_tiles<TM, TN>(acc, a[step % AHEAD], b[step % AHEAD]);
        __builtin_amdgcn_sched_barrier(0);
      }
    };
    if constexpr (MAPPED) static_for<DEPTH>([&](auto d) { lookup(d, d * KS + group); });
    __builtin_amdgcn_sched_barrier(0);
    run_k_tiles(mine, [&](auto d) { fetch(d, d * KS + group); }, step);
    if constexpr (KS > 1) {
      add_groups<KS, TM * TN, THREADS>(reinterpret_cast<floatx16_t*>(&acc), reinterpret_cast<float*>(smem_), group, tid);
    }
  } else if (p.accumulate) {
    return;                       // an expert without rows adds nothing
  }

  static_assert(BM * BN * 4 <= KS * 2 * STAGE, "the staged tile reuses the k-tiles' LDS");
  float* const lds = reinterpret_cast<float*>(smem_);
  __syncthreads();                           // the LDS has been read for the last time
  if (group == 0) {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int v = 0; v < 4; ++v)
          stage_acc<BN>(lds, (wm * TM + i) * 32 + (lane & 31), (wn * TN + j) * 32 + 8 * v + 4 * (lane >> 5),
                        reinterpret_cast<const float*>(&acc[i][j]) + 4 * v);
  }
  __syncthreads();
  T* const C = reinterpret_cast<T*>(q.C) + (int64_t)e * q.M * q.N;
  constexpr int ROW_PIECES = BN / PIECE;
  for (int s = threadIdx.x; s < BM * ROW_PIECES; s += THREADS * KS) {
    const int r = s / ROW_PIECES, c = (s % ROW_PIECES) * PIECE;
    if (m0 + r >= q.M || n0 + c >= q.N) continue;
    T* const out = C + (int64_t)(m0 + r) * q.N + n0 + c;
    float f[PIECE];
    staged<BN>(lds, r, c, f);
    if (p.accumulate) {
      float old[PIECE];
      load_piece<T>(out, old);
#pragma unroll
      for (int x = 0; x < PIECE; ++x) f[x] += old[x];
    }
    store_piece<T>(out, f);
  }
}

template <typename T>
inline int launch_ragged_k(RaggedK p, int64_t A_rows, int cus, int kernel_id, hipStream_t s) {
  auto plan = [&](int bm) {
    int64_t tiles = 0;
    for (int q = 0; q < p.nprob; ++q) {
      p.first[q] = (int32_t)tiles;
      tiles += pk_ceil_div(p.prob[q].M, bm) * pk_ceil_div(p.prob[q].N, bm);
    }
    p.first[p.nprob] = (int32_t)tiles;
    return tiles * p.E;
  };
  // 128 x 128 tiles with two of them for every CU, unless they are that much more padding: in fp32 the two are within
  // 7 % of each other (us, 64 x 64 -> 128 x 128: 16 experts 1024 x 512, 250 rows 159 -> 148, 32 experts, 60 rows 109 -> 109;
  // 408 x 472, 14 % more padding, 71 -> 95), in bf16 the larger are a tenth faster (24 experts 1000 x 360, 172 rows 38 -> 33,
  // 16 experts 1024 x 512, 250 rows 39 -> 34; 408 x 472 22 -> 22)
  int64_t units = plan(128), area_128 = 0, area_64 = 0;
  for (int q = 0; q < p.nprob; ++q) {
    area_128 += pk_ceil_div(p.prob[q].M, 128) * pk_ceil_div(p.prob[q].N, 128) * 4;
    area_64 += pk_ceil_div(p.prob[q].M, 64) * pk_ceil_div(p.prob[q].N, 64);
  }
  const bool large = units >= 2 * (int64_t)cus && 100 * area_128 <= (sizeof(T) == 4 ? 105 : 125) * area_64;
  if (!large) units = plan(64);
  if (units > 0x7fffff00ll) return PK_ERR_SHAPE;
  if (units == 0) return PK_OK;
  const dim3 grid((unsigned)(pk_ceil_div(units, CHUNK * NXCD) * CHUNK * NXCD));
  const int ks = large ? 1 : reduction_groups(units, pk_ceil_div(pk_ceil_div(A_rows, p.E), kBK<T>), cus);
  const int32_t* map = nullptr;
  for (int q = 0; q < p.nprob; ++q)
    if (p.prob[q].map) map = p.prob[q].map;
  for (int q = 0; q < p.nprob; ++q)
    if (!p.prob[q].map) p.prob[q].map = map;
#define PK_RAGGED_K(TILE, KS)                                                                                                          \
  do {                                                                                                                                 \
    if (map) PK_LAUNCH_NOCHECK(kernel_id, s, (ragged_k_kernel<T, TILE, KS, true>), grid, dim3(256 * KS), 0, s, p);      \
    else PK_LAUNCH_NOCHECK(kernel_id, s, (ragged_k_kernel<T, TILE, KS, false>), grid, dim3(256 * KS), 0, s, p);            \
  } while (0)
  if (large) PK_RAGGED_K(2, 1);
  else if (ks == 4) PK_RAGGED_K(1, 4);
  else if (ks == 2) PK_RAGGED_K(1, 2);
  else PK_RAGGED_K(1, 1);
#undef PK_RAGGED_K
  PK_RETURN_IF_LAUNCH_FAILED();
  return PK_OK;
}

}  // namespace pk_tile
