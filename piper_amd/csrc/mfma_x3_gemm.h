// Dense GEMM C[M,N] = sum_k A(m,k) * B(k,n) with fp32-accurate products on the bf16 matrix
// cores: an fp32 operand is split exactly into three bf16 planes (v = hi + mid + lo, 8 mantissa
// bits each), a bf16 operand is its own single plane, and every pair of planes whose product is
// not below 2^-24 of the leading one is multiplied with v_mfma_f32_32x32x16_bf16 into one fp32
// accumulator (3 MFMAs for bf16 x fp32, 6 for fp32 x fp32).  Plane products are exact in fp32, so
// the result differs from an fp32 FMA chain only by summation order and the dropped 2^-24 terms.
// Against v_mfma_f32_32x32x2_f32 this is 5.3x (bf16 x fp32) / 2.7x (fp32 x fp32) fewer matrix-core
// cycles.  Same Params, tiling, split-K and epilogue as mfma_f32_gemm.h.  An operand whose k index
// is not the contiguous one is kept in LDS as [k][row] (8-byte stores of the 4 fetched elements)
// and turned into MFMA fragments by the transposing LDS read (ds_read_b64_tr_b16).
// An fp32 operand can also be handed over already split (split3_t: three bf16 planes in memory, made
// once by split_planes_kernel): every workgroup that loads a tile of an fp32 operand otherwise
// splits it again (about 20 vector instructions per MFMA with tiles this small).  The planes are
// 6 bytes per element where the fp32 value is 4, so this pays only where the split arithmetic is
// what the kernel waits for: measured, the gate weight gradient (a long reduction over the tokens,
// d_logits re-read by every column tile) gains a fifth, the forward and the d_x GEMM lose.
#pragma once
#include "mfma_f32_gemm.h"
#include <type_traits>

namespace pk_x3mm {

using pk_f32mm::Params;
constexpr int BK = 32;
constexpr int LDK = BK + 8;   // bf16 per LDS row: 80-byte rows keep 16-byte fragment reads aligned
constexpr int MN_PAD = 8;     // bf16 of padding per [k][row] LDS row

typedef short shortx4_t __attribute__((ext_vector_type(4)));
typedef short shortx8_t __attribute__((ext_vector_type(8)));

// MFMA operand fragment (lane -> row lane%32, k = kk + 8*(lane/32) + 0..7) of a [row][k] tile
__device__ __forceinline__ bf16x8_t frag_kc(const bf16_t* tile, int row0, int kk, int lane) {
  return *reinterpret_cast<const bf16x8_t*>(tile + (row0 + (lane & 31)) * LDK + kk + 8 * (lane >> 5));
}
// the same fragment out of a [k][row] tile with `ld` bf16 per k-row: within 16 lanes, lane i
// points at 4 consecutive rows of k-row i/4 and receives 4 consecutive k of row i
__device__ __forceinline__ bf16x8_t frag_mn(const bf16_t* tile, int ld, int row0, int kk, int lane) {
  const int i = lane & 15;
  const int krow = kk + 8 * (lane >> 5) + (i >> 2);
  const int row = row0 + 16 * ((lane >> 4) & 1) + 4 * (i & 3);
  const bf16_t* ptr = tile + krow * ld + row;
  const shortx4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) shortx4_t*)(ptr));
  const shortx4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) shortx4_t*)(ptr + 4 * ld));
  return __builtin_bit_cast(bf16x8_t, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
}

// operand element types: float (split on load), bf16_t (one plane), split3_t (three bf16 planes in
// memory: plane q of element i at base[q * plane_stride + i])
struct split3_t {};
template <typename T> struct Planes;
template <> struct Planes<float> { static constexpr int N = 3; };
template <> struct Planes<bf16_t> { static constexpr int N = 1; };
template <> struct Planes<split3_t> { static constexpr int N = 3; };
template <typename T> struct Mem { typedef T type; };
template <> struct Mem<split3_t> { typedef bf16_t type; };      // what the operand pointer points at

// fp32 [n] -> three bf16 planes [3][n]: hi = bf16(v), mid = bf16(v - hi), lo = bf16(v - hi - mid)
__global__ __launch_bounds__(256) void split_planes_kernel(const float* __restrict__ src, bf16_t* __restrict__ dst, int64_t n) {
  const int64_t i = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4;
  if (i + 4 <= n) {
    const float4 v = *reinterpret_cast<const float4*>(src + i);
    const float f[4] = {v.x, v.y, v.z, v.w};
    bf16x4_t pl[3];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const bf16_t hi = (bf16_t)f[j];
      const float r1 = f[j] - (float)hi;
      const bf16_t mid = (bf16_t)r1;
      pl[0][j] = hi; pl[1][j] = mid; pl[2][j] = (bf16_t)(r1 - (float)mid);
    }
#pragma unroll
    for (int q = 0; q < 3; ++q) *reinterpret_cast<bf16x4_t*>(dst + q * n + i) = pl[q];
  } else {
    for (int64_t e = i; e < n; ++e) {
      const bf16_t hi = (bf16_t)src[e];
      const float r1 = src[e] - (float)hi;
      const bf16_t mid = (bf16_t)r1;
      dst[e] = hi; dst[n + e] = mid; dst[2 * n + e] = (bf16_t)(r1 - (float)mid);
    }
  }
}

template <int P>
__device__ __forceinline__ void split(float v, bf16_t (&out)[P]) {
  out[0] = (bf16_t)v;
  if (P > 1) {
    const float r1 = v - (float)out[0];
    out[1] = (bf16_t)r1;
    if (P > 2) out[2] = (bf16_t)(r1 - (float)out[1]);
  }
}
template <int P>
__device__ __forceinline__ void zero_planes(bf16x4_t (&out)[P]) {
  const bf16x4_t zero = {(bf16_t)0.f, (bf16_t)0.f, (bf16_t)0.f, (bf16_t)0.f};
#pragma unroll
  for (int q = 0; q < P; ++q) out[q] = zero;
}
// Four consecutive elements of an operand as they come from memory (Raw: fp32 values, or the planes),
// and as planes of four bf16.  They are split when they go to LDS: a split at the fetch waits for the
// load there and then (forward 61 -> 50 us, d_x 103 -> 84 us at 16,384 tokens, 128 experts, 2048 wide).
template <typename T> struct Raw { bf16x4_t v[Planes<T>::N]; };
template <> struct Raw<float> { floatx4_t v; };
template <typename T>
__device__ __forceinline__ void zero_raw(Raw<T>& r) {
  if constexpr (std::is_same<T, float>::value) r.v = floatx4_t{0.f, 0.f, 0.f, 0.f};
  else zero_planes<Planes<T>::N>(r.v);
}
template <typename T>
__device__ __forceinline__ void fetch4(const typename Mem<T>::type* src, int64_t plane_stride, Raw<T>& out) {
  if constexpr (std::is_same<T, float>::value) {
    out.v = *reinterpret_cast<const floatx4_t*>(src);
  } else {
#pragma unroll
    for (int q = 0; q < Planes<T>::N; ++q) out.v[q] = *reinterpret_cast<const bf16x4_t*>(src + q * plane_stride);
  }
}
template <typename T, bool PAIRS = true>
__device__ __forceinline__ void to_planes(const Raw<T>& r, bf16x4_t (&out)[Planes<T>::N]) {
  constexpr int P = Planes<T>::N;
  if constexpr (std::is_same<T, float>::value && !PAIRS) {
    bf16_t pl[4][P];
#pragma unroll
    for (int j = 0; j < 4; ++j) split<P>(r.v[j], pl[j]);
#pragma unroll
    for (int q = 0; q < P; ++q)
#pragma unroll
      for (int j = 0; j < 4; ++j) out[q][j] = pl[j][q];
  } else if constexpr (std::is_same<T, float>::value) {
    // split(), two values to a conversion: the pair is also where the rounded values are taken from
    typedef float floatx2_t __attribute__((ext_vector_type(2)));
    typedef bf16_t bf16x2_t __attribute__((ext_vector_type(2)));
    static_assert(P == 3, "three planes");
#pragma unroll
    for (int j = 0; j < 4; j += 2) {
      floatx2_t v = {r.v[j], r.v[j + 1]};
#pragma unroll
      for (int q = 0; q < 3; ++q) {
        const bf16x2_t b = __builtin_convertvector(v, bf16x2_t);
        out[q][j] = b[0];
        out[q][j + 1] = b[1];
        const uint32_t u = __builtin_bit_cast(uint32_t, b);
        v[0] -= __builtin_bit_cast(float, u << 16);
        v[1] -= __builtin_bit_cast(float, u & 0xffff0000u);
      }
    }
  } else {
#pragma unroll
    for (int q = 0; q < P; ++q) out[q] = r.v[q];
  }
}

template <int WM, int WN, bool A_KC, bool B_KC, typename TA, typename TB>
struct Lds {
  static constexpr int BM = 32 * WM, BN = 32 * WN;
  static constexpr int LDA = BM + MN_PAD, LDB = BN + MN_PAD;     // [k][row] layouts
  __attribute__((aligned(16))) bf16_t As[Planes<TA>::N][A_KC ? BM * LDK : BK * LDA];
  __attribute__((aligned(16))) bf16_t Bs[Planes<TB>::N][B_KC ? BN * LDK : BK * LDB];
};

// What the products below have in common: a thread's share of a k-tile in registers, its way into the LDS, and the matrix
// instructions.  Every thread holds 4 consecutive elements of the contiguous index per load (every plane of them for a pre-split operand).
template <int WM, int WN, bool A_KC, bool B_KC, typename TA, typename TB>
struct KTile {
  typedef Lds<WM, WN, A_KC, B_KC, TA, TB> Tiles;
  static constexpr int BM = 32 * WM, BN = 32 * WN, THREADS = 64 * WM * WN;
  static constexpr int PA = Planes<TA>::N, PB = Planes<TB>::N;
  static constexpr int NA = BM * BK / (THREADS * 4), NB = BN * BK / (THREADS * 4);
  static_assert(NA >= 1 && NB >= 1, "tile too small for the thread count");
  Raw<TA> a[NA];
  Raw<TB> b[NB];

  __device__ static __forceinline__ void slot(int idx, bool kc, int R, int& row, int& k) {
    if (kc) { k = (idx % (BK / 4)) * 4; row = idx / (BK / 4); }
    else { row = (idx % (R / 4)) * 4; k = idx / (R / 4); }
  }
  // one 8-byte store per plane: along k of a [row][k] tile for a K-contiguous operand, along the
  // rows of a [k][row] tile otherwise
  template <int P, typename Operand>
  __device__ static __forceinline__ void store4(Operand& tiles, bool kc, int ld_mn, int row, int k, const bf16x4_t (&v)[P]) {
#pragma unroll
    for (int q = 0; q < P; ++q) *reinterpret_cast<bf16x4_t*>(&tiles[q][kc ? row * LDK + k : k * ld_mn + row]) = v[q];
  }
  // into the LDS, cleared from k-index `have` on
  __device__ __forceinline__ void store(Tiles& lds, int tid, int have) {
#pragma unroll
    for (int i = 0; i < NA; ++i) {
      int m, k;
      slot(tid + i * THREADS, A_KC, BM, m, k);
      if (have < BK && k >= have) zero_raw<TA>(a[i]);
      bf16x4_t v[PA];
      to_planes<TA>(a[i], v);
      store4(lds.As, A_KC, Tiles::LDA, m, k, v);
    }
#pragma unroll
    for (int i = 0; i < NB; ++i) {
      int n, k;
      slot(tid + i * THREADS, B_KC, BN, n, k);
      if (have < BK && k >= have) zero_raw<TB>(b[i]);
      bf16x4_t v[PB];
      to_planes<TB>(b[i], v);
      store4(lds.Bs, B_KC, Tiles::LDB, n, k, v);
    }
  }
  __device__ static __forceinline__ void multiply(const Tiles& lds, int wm, int wn, int lane, floatx16_t& acc) {
#pragma unroll
    for (int kk = 0; kk < BK; kk += 16) {
      bf16x8_t fa[PA], fb[PB];
#pragma unroll
      for (int pl = 0; pl < PA; ++pl) fa[pl] = A_KC ? frag_kc(lds.As[pl], wm * 32, kk, lane) : frag_mn(lds.As[pl], Tiles::LDA, wm * 32, kk, lane);
#pragma unroll
      for (int pl = 0; pl < PB; ++pl) fb[pl] = B_KC ? frag_kc(lds.Bs[pl], wn * 32, kk, lane) : frag_mn(lds.Bs[pl], Tiles::LDB, wn * 32, kk, lane);
      // small terms first
#pragma unroll
      for (int s = PA + PB - 2; s >= 0; --s)
#pragma unroll
        for (int pa = 0; pa < PA; ++pa) {
          const int pb = s - pa;
          if (pb >= 0 && pb < PB && s <= 2) acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[pa], fb[pb], acc, 0, 0, 0);
        }
    }
  }
};

// How k-tiles are requested ahead (see product).  2: two in flight, for the products whose reduction is long: the forward from bf16
// and the weight gradients.  1: one, for the fp32 forward, whose split takes the registers of the second (64 experts 1024 wide,
// 10,000 tokens 18.5 -> 17.6 us).  0: one, ordered by the compiler, for d_x: its reduction over the experts is one to four k-tiles.
template <bool A_KC, bool B_KC, typename TA>
constexpr int in_flight() { return A_KC && !B_KC ? 0 : A_KC && std::is_same<TA, float>::value ? 1 : 2; }

// What bounds these products is the instructions and the waits around their matrix instructions, 6 or 12 a wave and k-tile.  The
// addresses are worked out once and advance by a constant, and the fp32 values are split two to a conversion: 100 vector
// instructions for two k-tiles of the bf16 forward, where forming the addresses of every load, masking it and splitting values one
// by one took 260.  The older of two k-tiles in flight is waited for by count, as nothing in the loop is conditional; without the
// scheduling barriers the compiler puts the requests behind the products and converts the younger tile first.  Four waves a
// SIMD (128 registers) matter more than a second k-tile, and more than the two registers that the fp32 weight gradient spills for
// them (three waves, nothing spilled: in one launch 2048 wide, 128 experts, 1,000 tokens 27.4 -> 30.2, 16,000 304 -> 309).  us, before -> now, 128 experts 2048 wide unless said: forward 16,384 tokens
// 53 -> 47, 4,096 19.2 -> 18.6, 8 experts, 16,384 37 -> 25; weight gradient 16,384 60 -> 56,
// fp32, 64 experts 1024 wide, 4,000 15.0 -> 11.4; d_x 16,384 96 -> 85; the router's backward in one launch (router_grads_kernel)
// 16,384 202 -> 189, 4,096 62 -> 58, 3,000 36 -> 33.
// (Its weight gradient's tiles dealt out among those of the gather instead of in front of them: 190 -> 195 to 262.)
//
// acc of one wave: rows m0 + 32 wm .., columns n0 + 32 wn .. of the product over k in [kbeg, kend).
template <int WM, int WN, bool A_KC, bool B_KC, typename TA, typename TB, int FLIGHT = 2>
__device__ __forceinline__ void product(const Params& p, Lds<WM, WN, A_KC, B_KC, TA, TB>& lds, int64_t m0, int64_t n0, int64_t kbeg,
                                        int64_t kend, floatx16_t& acc) {
  constexpr int BM = 32 * WM, BN = 32 * WN, THREADS = 64 * WM * WN;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int wm = wave / WN, wn = wave % WN;
  typedef typename Mem<TA>::type MA;
  typedef typename Mem<TB>::type MB;
  const MA* A = reinterpret_cast<const MA*>(p.A);
  const MB* B = reinterpret_cast<const MB*>(p.B);

#pragma unroll
  for (int v = 0; v < 16; ++v) acc[v] = 0.f;

  // No load stands behind a branch: rows past the ends are read from the last ones, and their results are not stored.
  typedef KTile<WM, WN, A_KC, B_KC, TA, TB> Tile;
  constexpr int NA = Tile::NA, NB = Tile::NB;
  const MA* pa[NA];
  const MB* pb[NB];
#pragma unroll
  for (int i = 0; i < NA; ++i) {
    int m, k;
    Tile::slot(tid + i * THREADS, A_KC, BM, m, k);
    pa[i] = A + min(m0 + m, p.M - (A_KC ? 1 : 4)) * p.sam + (A_KC ? kbeg + k : (kbeg + k) * p.sak);
  }
#pragma unroll
  for (int i = 0; i < NB; ++i) {
    int n, k;
    Tile::slot(tid + i * THREADS, B_KC, BN, n, k);
    pb[i] = B + min(n0 + n, p.N - (B_KC ? 1 : 4)) * p.sbn + (B_KC ? kbeg + k : (kbeg + k) * p.sbk);
  }
  const int64_t step_a = A_KC ? BK : BK * p.sak, step_b = B_KC ? BK : BK * p.sbk;
  const int64_t left = kend - kbeg;            // (nothing, or less, where the splits outnumber the k-tiles)
  const int full = left > 0 ? (int)(left / BK) : 0, rest = left > 0 ? (int)(left % BK) : 0;
  // the next k-tile, which is a whole one
  auto request = [&](Tile& t) {
#pragma unroll
    for (int i = 0; i < NA; ++i) { fetch4<TA>(pa[i], p.plane_a, t.a[i]); pa[i] += step_a; }
#pragma unroll
    for (int i = 0; i < NB; ++i) { fetch4<TB>(pb[i], p.plane_b, t.b[i]); pb[i] += step_b; }
  };
  // the next k-tile, of which only `have` (a multiple of 4 along a contiguous k) are there, the others from the last of them
  auto request_rest = [&](Tile& t, int have) {
#pragma unroll
    for (int i = 0; i < NA; ++i) {
      int m, k;
      Tile::slot(tid + i * THREADS, A_KC, BM, m, k);
      const int64_t back = max(0, k - (have - (A_KC ? 4 : 1)));
      fetch4<TA>(pa[i] - (A_KC ? back : back * p.sak), p.plane_a, t.a[i]);
    }
#pragma unroll
    for (int i = 0; i < NB; ++i) {
      int n, k;
      Tile::slot(tid + i * THREADS, B_KC, BN, n, k);
      const int64_t back = max(0, k - (have - (B_KC ? 4 : 1)));
      fetch4<TB>(pb[i] - (B_KC ? back : back * p.sbk), p.plane_b, t.b[i]);
    }
  };
  auto use = [&](Tile& t, int have, auto next) {
    t.store(lds, tid, have);
    __syncthreads();
    next();
    if constexpr (FLIGHT > 0) __builtin_amdgcn_sched_barrier(0);       // requested before the products, and the next tile not waited for before their end
    Tile::multiply(lds, wm, wn, lane, acc);
    __syncthreads();
    if constexpr (FLIGHT > 0) __builtin_amdgcn_sched_barrier(0);
  };
  auto nothing = [] {};
  if constexpr (FLIGHT <= 1) {
    Tile t;
    if (full > 0) {
      request(t);
      for (int j = 1; j < full; ++j) use(t, BK, [&] { request(t); });
      use(t, BK, [&] { if (rest) request_rest(t, rest); });
    } else if (rest) {
      request_rest(t, rest);
    }
    if (rest) use(t, rest, nothing);
  } else {
    // two k-tiles in flight; the loop has one exit and nothing in it is conditional, so that it waits for the older tile's loads only
    Tile t[2];
    int j = 0;
    if (full > 3) {
      request(t[0]);
      __builtin_amdgcn_sched_barrier(0);
      request(t[1]);
      __builtin_amdgcn_sched_barrier(0);
      do {
        use(t[0], BK, [&] { request(t[0]); });
        use(t[1], BK, [&] { request(t[1]); });
        j += 2;
      } while (j + 3 < full);
    } else {
      if (full > 0) request(t[0]);
      if (full > 1) request(t[1]);
    }
    if (full - j == 3) {
      use(t[0], BK, [&] { request(t[0]); });
      use(t[1], BK, nothing);
      use(t[0], BK, nothing);
    } else {
      if (full - j >= 1) use(t[0], BK, nothing);
      if (full - j >= 2) use(t[1], BK, nothing);
    }
    if (rest) {
      request_rest(t[0], rest);
      use(t[0], rest, nothing);
    }
  }
}

// The same of a reduction of at most AHEAD k-tiles along both operands' contiguous index, all of them requested at once.  Its loads,
// masks and splits are formed one by one: with those of product() it takes a microsecond more (us, 128 experts 2048 wide, 509
// tokens 9.7 -> 10.7, 1,777 12.0 -> 13.1, fp32 1024 wide, 1,000 7.8 -> 9.1), as a workgroup alone on its CU has nothing to do meanwhile.
template <int WM, int WN, typename TA, typename TB, int AHEAD>
__device__ __forceinline__ void product_at_once(const Params& p, Lds<WM, WN, true, true, TA, TB>& lds, int64_t m0, int64_t n0, int64_t kbeg,
                                                int64_t kend, floatx16_t& acc) {
  typedef KTile<WM, WN, true, true, TA, TB> Tile;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int wm = wave / WN, wn = wave % WN;
  typedef typename Mem<TA>::type MA;
  typedef typename Mem<TB>::type MB;
  const MA* A = reinterpret_cast<const MA*>(p.A);
  const MB* B = reinterpret_cast<const MB*>(p.B);

#pragma unroll
  for (int v = 0; v < 16; ++v) acc[v] = 0.f;

  // (past the ends from the last elements, as a branch would hold up the loads behind it)
  auto load_tile = [&](Tile& t, int64_t k0) {
#pragma unroll
    for (int i = 0; i < Tile::NA; ++i) {
      int m, k;
      Tile::slot(tid + i * Tile::THREADS, true, Tile::BM, m, k);
      fetch4<TA>(A + min(m0 + m, p.M - 1) * p.sam + min(k0 + k, kend - 4) * p.sak, p.plane_a, t.a[i]);
    }
#pragma unroll
    for (int i = 0; i < Tile::NB; ++i) {
      int n, k;
      Tile::slot(tid + i * Tile::THREADS, true, Tile::BN, n, k);
      fetch4<TB>(B + min(k0 + k, kend - 4) * p.sbk + min(n0 + n, p.N - 1) * p.sbn, p.plane_b, t.b[i]);
    }
  };
  auto store_tile = [&](Tile& t, int64_t k0) {
#pragma unroll
    for (int i = 0; i < Tile::NA; ++i) {
      int m, k;
      Tile::slot(tid + i * Tile::THREADS, true, Tile::BM, m, k);
      if (k0 + k >= kend) zero_raw<TA>(t.a[i]);
      bf16x4_t v[Tile::PA];
      to_planes<TA, false>(t.a[i], v);
      Tile::store4(lds.As, true, 0, m, k, v);
    }
#pragma unroll
    for (int i = 0; i < Tile::NB; ++i) {
      int n, k;
      Tile::slot(tid + i * Tile::THREADS, true, Tile::BN, n, k);
      if (k0 + k >= kend) zero_raw<TB>(t.b[i]);
      bf16x4_t v[Tile::PB];
      to_planes<TB, false>(t.b[i], v);
      Tile::store4(lds.Bs, true, 0, n, k, v);
    }
  };
  Tile t[AHEAD];
#pragma unroll
  for (int i = 0; i < AHEAD; ++i) load_tile(t[i], kbeg + i * BK);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int i = 0; i < AHEAD; ++i)
    if (kbeg + i * BK < kend) {
      store_tile(t[i], kbeg + i * BK);
      __syncthreads();
      Tile::multiply(lds, wm, wn, lane, acc);
      __syncthreads();
    }
}

// output tile (bx, by) of split bz
template <int WM, int WN, bool A_KC, bool B_KC, typename TA, typename TB, int AHEAD = 0, int FLIGHT = 2>
__device__ __forceinline__ void gemm_tile(const Params& p, Lds<WM, WN, A_KC, B_KC, TA, TB>& lds, int bx, int by, int bz) {
  constexpr int BM = 32 * WM, BN = 32 * WN;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int wm = wave / WN, wn = wave % WN;
  const int64_t m0 = (int64_t)by * BM, n0 = (int64_t)bx * BN;
  const int64_t kchunk = ((p.K + p.splits - 1) / p.splits + BK - 1) / BK * BK;
  const int64_t kbeg = (int64_t)bz * kchunk;
  const int64_t kend = kbeg + kchunk < p.K ? kbeg + kchunk : p.K;
  floatx16_t acc;
  if constexpr (AHEAD > 0) product_at_once<WM, WN, TA, TB, AHEAD>(p, lds, m0, n0, kbeg, kend, acc);
  else product<WM, WN, A_KC, B_KC, TA, TB, FLIGHT>(p, lds, m0, n0, kbeg, kend, acc);

  float* C = p.C + (p.splits > 1 ? (int64_t)bz * p.M * p.N : 0);
  const int64_t n = n0 + wn * 32 + (lane & 31);
  if (n < p.N) {
    const float bias = (p.bias && p.splits == 1) ? p.bias[n] : 0.f;
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      const int64_t m = m0 + wm * 32 + 8 * (v >> 2) + 4 * (lane >> 5) + (v & 3);
      if (m < p.M) {
        float r = acc[v] + bias;
        if (p.accumulate && p.splits == 1) r += C[m * p.N + n];
        C[m * p.N + n] = r;
      }
    }
  }
}
template <int WM, int WN, bool A_KC, bool B_KC, typename TA, typename TB>
__global__ __launch_bounds__(64 * WM * WN, 4) void kernel(const Params p) {
  __shared__ Lds<WM, WN, A_KC, B_KC, TA, TB> lds;
  gemm_tile<WM, WN, A_KC, B_KC, TA, TB, 0, in_flight<A_KC, B_KC, TA>()>(p, lds, blockIdx.x, blockIdx.y, blockIdx.z);
}
template <int WM, int WN, typename TA, typename TB, int AHEAD>
__global__ __launch_bounds__(64 * WM * WN) void at_once_kernel(const Params p) {
  __shared__ Lds<WM, WN, true, true, TA, TB> lds;
  gemm_tile<WM, WN, true, true, TA, TB, AHEAD>(p, lds, blockIdx.x, blockIdx.y, blockIdx.z);
}

// The gradient of the region's input in one pass: out[t] = sum_k rows[inv_perm[t*K + k]] + d_logits[t] .
// w_gate, the second term being this GEMM.  Its tile goes through LDS, and every thread then adds the K
// gathered rows for 16 bytes of a token (the sum over k first, the GEMM's value last, rounded once: what
// the GEMM into an fp32 [T, H] tensor and gather_reduce_kernel behind it compute), so that tensor is
// neither written nor read.  STREAM: the gathered rows are too many to stay in a cache.
struct GatherAdd {
  const void* rows;           // [T * K, H], element type TG
  const int32_t* inv_perm;    // [T * K]
  void* out;                  // [T, H]
  int32_t K;
};
template <int WM, int WN>
struct GatherLds {
  typedef Lds<WM, WN, true, false, float, float> Tiles;
  static constexpr int LDO = 32 * WN + 4;
  static constexpr int BYTES = sizeof(Tiles) > 32 * WM * LDO * 4 ? (int)sizeof(Tiles) : 32 * WM * LDO * 4;
};
template <int WM, int WN, typename TG, bool STREAM>
__device__ __forceinline__ void gather_tile(const Params& p, const GatherAdd& ga, char* smem, int bx, int by) {
  constexpr int BM = 32 * WM, BN = 32 * WN, THREADS = 64 * WM * WN;
  typedef typename GatherLds<WM, WN>::Tiles Tiles;
  constexpr int LDO = GatherLds<WM, WN>::LDO;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int wm = wave / WN, wn = wave % WN;
  const int64_t m0 = (int64_t)by * BM, n0 = (int64_t)bx * BN;
  floatx16_t acc;
  product<WM, WN, true, false, float, float, 1>(p, *reinterpret_cast<Tiles*>(smem), m0, n0, 0, p.K, acc);
  float* const tile = reinterpret_cast<float*>(smem);       // (product ends with a barrier)
#pragma unroll
  for (int v = 0; v < 16; ++v)
    tile[(wm * 32 + 8 * (v >> 2) + 4 * (lane >> 5) + (v & 3)) * LDO + wn * 32 + (lane & 31)] = acc[v];
  __syncthreads();
  constexpr int N = PkVec16<TG>::N, PIECES = BN / N;        // 16-byte pieces of a token's columns
  constexpr int KB = 8;
  const int H = (int)p.N;
  for (int i = tid; i < BM * PIECES; i += THREADS) {
    const int r = i / PIECES, c = (i % PIECES) * N;
    const int64_t t = m0 + r;
    if (t >= p.M || n0 + c >= H) continue;
    float sum[N];
#pragma unroll
    for (int j = 0; j < N; ++j) sum[j] = 0.f;
    const int32_t* inv = ga.inv_perm + t * ga.K;
    for (int k0 = 0; k0 < ga.K; k0 += KB) {
      PkVec16<TG> v[KB];
#pragma unroll
      for (int j = 0; j < KB; ++j) {
        const int64_t row = inv[k0 + j < ga.K ? k0 + j : ga.K - 1];
        const auto* src = reinterpret_cast<const decltype(v[j].v)*>(reinterpret_cast<const TG*>(ga.rows) + row * H + n0 + c);
        if (STREAM) v[j].v = __builtin_nontemporal_load(src);
        else v[j].v = *src;
      }
#pragma unroll
      for (int j = 0; j < KB; ++j)
        if (k0 + j < ga.K) {
#pragma unroll
          for (int e = 0; e < N; ++e) sum[e] += v[j].get(e);
        }
    }
    PkVec16<TG> o;
#pragma unroll
    for (int e = 0; e < N; ++e) o.set(e, sum[e] + tile[r * LDO + c + e]);
    *reinterpret_cast<decltype(o.v)*>(reinterpret_cast<TG*>(ga.out) + t * H + n0 + c) = o.v;
  }
}
template <int WM, int WN, typename TG, bool STREAM>
__global__ __launch_bounds__(64 * WM * WN, 4) void gather_kernel(const Params p, const GatherAdd ga) {
  __shared__ __attribute__((aligned(16))) char smem[GatherLds<WM, WN>::BYTES];
  gather_tile<WM, WN, TG, STREAM>(p, ga, smem, blockIdx.x, blockIdx.y);
}

// The operands must allow 4-element loads (pk_f32mm::vec4_ok); the caller falls back to
// pk_f32mm::launch otherwise.
template <int WM, int WN, bool A_KC, bool B_KC, typename TA, typename TB>
inline bool usable(const Params& p) {
  using pk_f32mm::vec4_ok;
  typedef typename Mem<TA>::type MA;
  typedef typename Mem<TB>::type MB;
  if (std::is_same<TA, split3_t>::value && p.plane_a % 4 != 0) return false;
  if (std::is_same<TB, split3_t>::value && p.plane_b % 4 != 0) return false;
  return (A_KC ? (p.sak == 1 && vec4_ok<MA>(p.A, p.K, p.sam)) : (p.sam == 1 && vec4_ok<MA>(p.A, p.M, p.sak))) &&
         (B_KC ? (p.sbk == 1 && vec4_ok<MB>(p.B, p.K, p.sbn)) : (p.sbn == 1 && vec4_ok<MB>(p.B, p.N, p.sbk)));
}

template <int WM, int WN, bool A_KC, bool B_KC, typename TA, typename TB>
inline int launch(const Params& p, int kernel_id, hipStream_t s) {
  if (!usable<WM, WN, A_KC, B_KC, TA, TB>(p)) {
    if constexpr (std::is_same<TA, split3_t>::value || std::is_same<TB, split3_t>::value) return PK_ERR_ALIGN;   // the caller splits only what this kernel can read
    else return pk_f32mm::launch<WM, WN, A_KC, B_KC, TA, TB>(p, kernel_id, s);
  }
  if (p.M <= 0 || p.N <= 0) return PK_OK;
  dim3 grid((unsigned)pk_ceil_div(p.N, 32 * WN), (unsigned)pk_ceil_div(p.M, 32 * WM), (unsigned)p.splits);
  if (grid.y > 65535u || grid.z > 65535u) return PK_ERR_SHAPE;
  // A workgroup that has a CU to itself waits for every k-tile's loads in turn: a reduction of up to 256, which is what the gate's
  // splits leave, is requested as a whole.  Where workgroups share a CU the registers for it cost more (gate, us, 128
  // experts 2048 wide: 300 tokens 13.7 -> 11.8, 1,777 tokens, 224 workgroups 14.1 -> 12.6, 3,000 tokens, 376 16.7 -> 18.9;
  // 64 experts, 1,500 tokens 12.1 -> 8.8; fp32, 128 experts 1024 wide, 1,000 tokens 10.8 -> 9.9, 4,000 14.7 -> 16.2).
  if constexpr (A_KC && B_KC) {
    const int64_t k_tiles = pk_ceil_div(pk_ceil_div(p.K, p.splits), BK);
    if ((int64_t)grid.x * grid.y * grid.z <= 256 && k_tiles <= 8) {
      if (k_tiles <= 4) PK_LAUNCH_NOCHECK(kernel_id, s, (at_once_kernel<WM, WN, TA, TB, 4>), grid, dim3(64 * WM * WN), 0, s, p);
      else PK_LAUNCH_NOCHECK(kernel_id, s, (at_once_kernel<WM, WN, TA, TB, 8>), grid, dim3(64 * WM * WN), 0, s, p);
      PK_RETURN_IF_LAUNCH_FAILED();
      return PK_OK;
    }
  }
  PK_LAUNCH_NOCHECK(kernel_id, s, (kernel<WM, WN, A_KC, B_KC, TA, TB>), grid, dim3(64 * WM * WN), 0, s, p);
  PK_RETURN_IF_LAUNCH_FAILED();
  return PK_OK;
}

// d_logits: p.A [T, E], w_gate: p.B [E, H] (p.M = T, p.N = H, p.K = E).  PK_ERR_ALIGN: a base is not 16-byte
// aligned, which the caller's contract asks for (widths without whole pieces go to the two kernels).
// 32 tokens x 128 columns (16,384 tokens, the router backward as a whole: 212 us; 64 x 128: 214, 64 x 64: 222;
// with the GEMM and the gather apart 270)
constexpr int kGatherWM = 1, kGatherWN = 4;
// one launch per 65,535 row blocks, what grid.y holds: the GEMM with 64-row blocks in front of a separate
// gather takes twice that many tokens, and so does the forward
constexpr int64_t kGatherSlice = (int64_t)65535 * 32 * kGatherWM;
template <typename TG>
inline bool gather_usable(const Params& p, const GatherAdd& ga) {
  return usable<kGatherWM, kGatherWN, true, false, float, float>(p) && p.N % PkVec16<TG>::N == 0 && pk_aligned16(ga.rows) && pk_aligned16(ga.out);
}
template <typename TG>
inline bool gather_streams(const Params& p, const GatherAdd& ga) {
  return p.M * ga.K * p.N * (int64_t)sizeof(TG) > (int64_t)192 * 1024 * 1024;
}
template <typename TG>
inline int launch_gather(const Params& p, const GatherAdd& ga, int kernel_id, hipStream_t s) {
  constexpr int WM = kGatherWM, WN = kGatherWN;
  if (!gather_usable<TG>(p, ga)) return PK_ERR_ALIGN;
  const bool stream_rows = gather_streams<TG>(p, ga);
  constexpr int64_t SLICE = kGatherSlice;
  for (int64_t t0 = 0; t0 < p.M; t0 += SLICE) {
    Params q = p;
    GatherAdd gq = ga;
    q.M = p.M - t0 < SLICE ? p.M - t0 : SLICE;
    q.A = static_cast<const float*>(p.A) + t0 * p.sam;
    gq.inv_perm = ga.inv_perm + t0 * ga.K;
    gq.out = static_cast<TG*>(ga.out) + t0 * p.N;
    const dim3 grid((unsigned)pk_ceil_div(p.N, 32 * WN), (unsigned)pk_ceil_div(q.M, 32 * WM));
    if (stream_rows) PK_LAUNCH_NOCHECK(kernel_id, s, (gather_kernel<WM, WN, TG, true>), grid, dim3(64 * WM * WN), 0, s, q, gq);
    else PK_LAUNCH_NOCHECK(kernel_id, s, (gather_kernel<WM, WN, TG, false>), grid, dim3(64 * WM * WN), 0, s, q, gq);
    PK_RETURN_IF_LAUNCH_FAILED();
  }
  return PK_OK;
}

}  // namespace pk_x3mm
