// Routing: gate logits, wavefront softmax/top-k (+ backward), stable counting sort by expert.
#include "pk_common.h"
#include "gate_tail.h"
#include "topk.h"
#include "mfma_x3_gemm.h"
#include <mutex>

namespace {

// ------------------------------------------------------------------ top-k
constexpr int kRouteThreads = 256;  // 4 waves, one token per wave

// Split-K partial results of the gate GEMM, summed by whoever reads the logits first.
struct GatePartials {
  const float* part;    // [splits][T][E], or nullptr: the logits are complete
  const float* bias;    // [E] or nullptr
  int splits;
};

// PARTIALS: the logits are still split-K partial results; they are summed here (in split order, then
// the bias: what reduce_partials_kernel would store) and written out on the way, which saves a launch
// and a pass over [T, E].
template <int EPL, bool PARTIALS>
__device__ __forceinline__ void route_topk_token(int t, int lane, const GatePartials gp, float* __restrict__ logits, int T, int E, int K,
                                                 int route_norm, float route_scale, float& out_s, int& out_e) {
  float* row = logits + (int64_t)t * E;
  float val[1][EPL], score[1];
  int expert[1];
  if (PARTIALS) {
    const int64_t n = (int64_t)T * E;
#pragma unroll
    for (int j = 0; j < EPL; ++j) {
      const int e = lane + 64 * j;
      float s = 0.f;
      if (e < E) {
        const float* src = gp.part + (int64_t)t * E + e;
        float v[8];
#pragma unroll
        for (int z = 0; z < 8; ++z) v[z] = z < gp.splits ? src[z * n] : 0.f;
#pragma unroll
        for (int z = 0; z < 8; ++z)
          if (z < gp.splits) s += v[z];
        if (gp.bias) s += gp.bias[e];
        row[e] = s;
      }
      val[0][j] = s;
    }
  }
  if (!PARTIALS) {
#pragma unroll
    for (int j = 0; j < EPL; ++j) val[0][j] = lane + 64 * j < E ? row[lane + 64 * j] : 0.f;
  }
  topk_of<EPL, 1>(val, lane, E, K, route_norm, route_scale, score, expert);
  out_s = score[0];
  out_e = expert[0];
}

template <int EPL, bool PARTIALS>
__global__ __launch_bounds__(kRouteThreads) void route_topk_kernel(
    const GatePartials gp, float* __restrict__ logits, int T, int E, int K, int route_norm, float route_scale,
    float* __restrict__ top_scores, int32_t* __restrict__ top_idx) {
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int t = blockIdx.x * (kRouteThreads / 64) + wave;
  if (t >= T) return;
  float s;
  int e;
  route_topk_token<EPL, PARTIALS>(t, lane, gp, logits, T, E, K, route_norm, route_scale, s, e);
  if (lane < K) {
    top_scores[(int64_t)t * K + lane] = s;
    top_idx[(int64_t)t * K + lane] = e;
  }
}

// The same with the histogram that sort_scatter_kernel wants: a workgroup takes the 16 tokens of a chunk, a wave each (128 experts,
// top 8, us: 1,777 tokens, top-k 5.0 + histogram 4.4 + placing 7.2 -> 6.2 + 7.0; 300 tokens, top-k 5.0 + sort_small_kernel
// 8.5 -> 11.8; 100 tokens 10.0 -> 11.4).
constexpr int kTopkHistTokens = 16, kTopkHistExperts = 128;
template <int EPL, bool PARTIALS>
__global__ __launch_bounds__(64 * kTopkHistTokens) void route_topk_hist_kernel(const GatePartials gp, float* __restrict__ logits, int T, int E, int K,
                                                                               int route_norm, float route_scale, float* __restrict__ top_scores,
                                                                               int32_t* __restrict__ top_idx, int32_t* __restrict__ chunk_hist) {
  __shared__ int32_t hist[kTopkHistExperts];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int t = blockIdx.x * kTopkHistTokens + wave;
  if (threadIdx.x < kTopkHistExperts) hist[threadIdx.x] = 0;
  __syncthreads();
  if (t < T) {
    float s;
    int e;
    route_topk_token<EPL, PARTIALS>(t, lane, gp, logits, T, E, K, route_norm, route_scale, s, e);
    if (lane < K) {
      top_scores[(int64_t)t * K + lane] = s;
      top_idx[(int64_t)t * K + lane] = e;
      atomicAdd(&hist[e], 1);
    }
  }
  __syncthreads();
  if ((int)threadIdx.x < E) chunk_hist[(int64_t)blockIdx.x * E + threadIdx.x] = hist[threadIdx.x];
}

// Where the score gradients come from and where d_logits goes besides its own tensor.
struct RouteBwdIo {
  const float* d_top_scores;    // [T, K], or nullptr:
  const float* part;            //   the d_h GEMM's partial sums [n_part][A], in sorted row order
  const int32_t* inv_perm;      //   flat slot -> sorted row
  int64_t A;
  int32_t n_part;
  bf16_t* planes;               // optional: d_logits as three bf16 planes [3][T * E] for the gate weight gradient
};
template <int EPL>
__global__ __launch_bounds__(kRouteThreads) void route_topk_bwd_kernel(
    const float* __restrict__ logits, const int32_t* __restrict__ top_idx,
    const RouteBwdIo io, int T, int E, int K, int route_norm,
    float route_scale, float* __restrict__ d_logits) {
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int t = blockIdx.x * (kRouteThreads / 64) + wave;
  if (t >= T) return;
  const float* row = logits + (int64_t)t * E;

  float val[EPL];
  float mx = -INFINITY;
#pragma unroll
  for (int j = 0; j < EPL; ++j) {
    const int e = lane + 64 * j;
    val[j] = (e < E) ? row[e] : -INFINITY;
    mx = fmaxf(mx, val[j]);
  }
  mx = from_orderable(wave_max_u32(orderable(mx)));
  float p[EPL];
  float part = 0.f;
#pragma unroll
  for (int j = 0; j < EPL; ++j) {
    p[j] = (lane + 64 * j < E) ? expf(val[j] - mx) : 0.f;
    part += p[j];
  }
  const float denom = wave_sum_f32(part);
#pragma unroll
  for (int j = 0; j < EPL; ++j) p[j] = p[j] / denom;

  // lanes k < K: selected expert, its probability, incoming gradient
  int my_e = -1;
  float s = 0.f, dw = 0.f;
  if (lane < K) {
    my_e = top_idx[(int64_t)t * K + lane];
    s = expf(row[my_e] - mx) / denom;
    if (io.d_top_scores) {
      dw = io.d_top_scores[(int64_t)t * K + lane];
    } else {      // summed in partial order, like dscore_reduce_kernel
      const int64_t r = io.inv_perm[(int64_t)t * K + lane];
      for (int q0 = 0; q0 < io.n_part; q0 += 8) {
        float v[8];
#pragma unroll
        for (int q = 0; q < 8; ++q) v[q] = q0 + q < io.n_part ? io.part[(q0 + q) * io.A + r] : 0.f;
#pragma unroll
        for (int q = 0; q < 8; ++q)
          if (q0 + q < io.n_part) dw += v[q];
      }
    }
  }
  float ds;
  if (route_norm) {
    const float S = wave_sum_f32(s) + 1e-20f;
    const float dot = wave_sum_f32(dw * s);
    ds = route_scale * (dw / S - dot / (S * S));
  } else {
    ds = route_scale * dw;
  }
  if (lane >= K) ds = 0.f;
  const float D = wave_sum_f32(ds * s);  // sum_j dp_j p_j

  float dp[EPL];
#pragma unroll
  for (int j = 0; j < EPL; ++j) dp[j] = 0.f;
  for (int k = 0; k < K; ++k) {
    const int ek = __builtin_amdgcn_readlane(my_e, k);
    const float dsk = __uint_as_float((uint32_t)__builtin_amdgcn_readlane((int)__float_as_uint(ds), k));
#pragma unroll
    for (int j = 0; j < EPL; ++j)
      if (lane + 64 * j == ek) dp[j] = dsk;
  }
#pragma unroll
  for (int j = 0; j < EPL; ++j) {
    const int e = lane + 64 * j;
    if (e < E) {
      const float d = p[j] * (dp[j] - D);
      const int64_t at = (int64_t)t * E + e;
      d_logits[at] = d;
      if (io.planes) {
        const int64_t n = (int64_t)T * E;
        bf16_t pl[3];
        pk_x3mm::split<3>(d, pl);
        io.planes[at] = pl[0]; io.planes[n + at] = pl[1]; io.planes[2 * n + at] = pl[2];
      }
    }
  }
}

// ------------------------------------------------------------------ counting sort
constexpr int kSortChunk = 512;  // flat slots per chunk

__global__ __launch_bounds__(64) void sort_hist_kernel(const int32_t* __restrict__ idx, int A,
                                                       int E, int32_t* __restrict__ chunk_hist) {
  extern __shared__ int32_t hist[];  // [E]
  for (int e = threadIdx.x; e < E; e += 64) hist[e] = 0;
  __syncthreads();
  const int base = blockIdx.x * kSortChunk;
  for (int i = threadIdx.x; i < kSortChunk; i += 64) {
    const int s = base + i;
    if (s < A) {
      const int e = idx[s];
      if ((unsigned)e < (unsigned)E) atomicAdd(&hist[e], 1);  // out-of-range ids are dropped
    }
  }
  __syncthreads();
  for (int e = threadIdx.x; e < E; e += 64) chunk_hist[(int64_t)blockIdx.x * E + e] = hist[e];
}

// Lanes of the wave that hold the same expert id as this one (ids below 1,024; inactive lanes: none).
__device__ __forceinline__ unsigned long long same_expert_lanes(int e, bool active, int id_bits) {
  unsigned long long same = __ballot(active);
  for (int b = 0; b < id_bits; ++b) {
    const unsigned long long bal = __ballot((e >> b) & 1);
    same &= ((e >> b) & 1) ? bal : ~bal;
  }
  return same;
}
// One wave places slots [s0, s0 + n), in order: `cursor` (LDS, private to the wave) holds the next free
// position per expert.  The rank of a slot among the 64 of a step is a population count, so equal
// experts keep their slot order.
__device__ __forceinline__ void place_slots(const int32_t* __restrict__ idx, int s0, int n, int A, int E, int id_bits, int32_t* cursor,
                                            int32_t* __restrict__ perm, int32_t* __restrict__ inv_perm) {
  const int lane = threadIdx.x & 63;
  const unsigned long long lt_mask = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
  for (int i = 0; i < n; i += 64) {
    const int s = s0 + i + lane;
    int e = (i + lane < n && s < A) ? idx[s] : -1;
    const bool active = (unsigned)e < (unsigned)E;      // out-of-range ids are dropped
    const unsigned long long same = same_expert_lanes(e, active, id_bits);
    int pos = 0;
    if (active) pos = cursor[e] + __popcll(same & lt_mask);
    __builtin_amdgcn_wave_barrier();
    if (active) {
      if (lane == 63 - __clzll(same)) cursor[e] += __popcll(same);     // the last lane of a group advances the cursor
      perm[pos] = s;
      if (inv_perm) inv_perm[s] = pos;
    }
    __builtin_amdgcn_wave_barrier();
  }
}
__host__ __device__ inline int id_bits_for(int E) {
  int b = 0;
  while ((1 << b) < E) ++b;
  return b;
}
// Exclusive prefix sum over v[0, n) in LDS by the whole block (n <= blockDim.x rounded up to a power of
// two); every thread passes its own element and gets its exclusive sum.
__device__ __forceinline__ int block_exclusive_scan(int mine, int32_t* wave_sums) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nw = blockDim.x >> 6;
  int incl = mine;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const int v = __shfl_up(incl, off, PK_WAVE);
    if (lane >= off) incl += v;
  }
  if (lane == 63) wave_sums[wave] = incl;
  __syncthreads();
  int before = 0;
  for (int w = 0; w < nw; ++w) before += w < wave ? wave_sums[w] : 0;
  __syncthreads();
  return before + incl - mine;
}
// order[rank] = e: experts by descending row count, ties by index.  cnt: LDS, rank: LDS scratch [E].
__device__ __forceinline__ void write_order(const int32_t* cnt, int32_t* rank, int E, int32_t* __restrict__ order) {
  for (int e = threadIdx.x; e < E; e += blockDim.x) rank[e] = 0;
  __syncthreads();
  int parts = blockDim.x / E;                    // threads that share an expert's comparisons
  if (parts < 1) parts = 1;
  for (int i = threadIdx.x; i < E * parts; i += blockDim.x) {
    const int e = i % E, part = i / E, c = cnt[e];
    int r = 0;
    for (int o = part; o < E; o += parts) {
      const int oc = cnt[o];
      r += (oc > c || (oc == c && o < e)) ? 1 : 0;
    }
    if (r) atomicAdd(&rank[e], r);
  }
  __syncthreads();
  for (int e = threadIdx.x; e < E; e += blockDim.x) order[rank[e]] = e;
}

// The whole sort in one workgroup of 16 waves, for inputs short enough that one CU's scattered stores
// (about one lane per cycle) do not matter: wave w owns the w-th sixteenth of the slots, counts its
// experts in LDS, the counts become first positions, and it places its slots.  Three launches took
// 16 us at 192 slots and 19 us at 4,072 (mostly gaps and latency), this one 5 and 11 us; at 8,192 the
// two kernels below are as quick.
constexpr int kSmallSortWaves = 16, kSmallSortSlots = 4096, kSmallSortExperts = 512;
struct SortOut {
  int32_t *counts, *starts, *perm, *inv_perm, *order;     // counts, inv_perm, order may be null
};
struct SmallSortLds {
  int32_t hist[kSmallSortWaves * kSmallSortExperts];      // [wave][E]
  int32_t cnt[kSmallSortExperts], rank[kSmallSortExperts], wave_sums[kSmallSortWaves];
};
__device__ __forceinline__ void sort_small(const int32_t* idx, int A, int E, const SortOut& out, SmallSortLds& l) {
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int per = ((A + kSmallSortWaves - 1) / kSmallSortWaves + 63) & ~63;      // slots per wave
  const int s0 = wave * per;
  for (int i = threadIdx.x; i < kSmallSortWaves * E; i += blockDim.x) l.hist[i] = 0;
  __syncthreads();
  for (int i = lane; i < per; i += 64) {
    const int s = s0 + i;
    if (s < A) {
      const int e = idx[s];
      if ((unsigned)e < (unsigned)E) atomicAdd(&l.hist[wave * E + e], 1);
    }
  }
  __syncthreads();
  const int e = threadIdx.x;
  int total = 0;
  if (e < E) {
#pragma unroll
    for (int w = 0; w < kSmallSortWaves; ++w) total += l.hist[w * E + e];
  }
  const int start = block_exclusive_scan(total, l.wave_sums);
  if (e < E) {
    int run = start;
    for (int w = 0; w < kSmallSortWaves; ++w) {
      const int n = l.hist[w * E + e];
      l.hist[w * E + e] = run;
      run += n;
    }
    l.cnt[e] = total;
    if (out.counts) out.counts[e] = total;
    out.starts[e] = start;
    if (e == E - 1) out.starts[E] = run;
  }
  __syncthreads();
  place_slots(idx, s0, per, A, E, id_bits_for(E), &l.hist[wave * E], out.perm, out.inv_perm);
  if (out.order) write_order(l.cnt, l.rank, E, out.order);
}
__global__ __launch_bounds__(64 * kSmallSortWaves) void sort_small_kernel(const int32_t* __restrict__ idx, int A, int E, const SortOut out) {
  __shared__ SmallSortLds l;
  sort_small(idx, A, E, out, l);
}
// Top-k and sort in one launch for a decode step: the 16 waves take the tokens in turn and hand the
// chosen experts over in LDS.
constexpr int kRouteSortTokens = 32, kRouteSortSlots = 1024;
template <int EPL, bool PARTIALS>
__global__ __launch_bounds__(64 * kSmallSortWaves) void route_sort_small_kernel(const GatePartials gp, float* __restrict__ logits, int T, int E, int K,
                                                                                int route_norm, float route_scale, float* __restrict__ top_scores,
                                                                                int32_t* __restrict__ top_idx, const SortOut out) {
  __shared__ SmallSortLds l;
  __shared__ int32_t chosen[kRouteSortSlots];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  for (int t = wave; t < T; t += kSmallSortWaves) {
    float s;
    int e;
    route_topk_token<EPL, PARTIALS>(t, lane, gp, logits, T, E, K, route_norm, route_scale, s, e);
    if (lane < K) {
      top_scores[t * K + lane] = s;
      top_idx[t * K + lane] = e;
      chosen[t * K + lane] = e;
    }
  }
  __syncthreads();
  sort_small(chosen, T * K, E, out, l);
}

// Inputs of more chunks than self_scan_chunks: one workgroup turns the chunk histograms into first positions.
// The 1024 threads form G = 1024 / cols groups of cols columns (E rounded up to a power of two); group g of
// expert e walks chunks [g * cpg, (g + 1) * cpg) twice, eight values at a time (one round trip per eight
// chunks): once for the group's sum, once to replace chunk_hist[c][e] by the first output position of
// expert e's rows of chunk c.
__global__ __launch_bounds__(1024) void sort_scan_kernel(int32_t* __restrict__ chunk_hist, int nchunks, int E, int32_t* __restrict__ counts,
                                                         int32_t* __restrict__ starts, int32_t* __restrict__ order) {
  __shared__ int32_t part[1024];       // [g][e]: rows of expert e in the chunks of group g
  __shared__ int32_t cnt[PK_MAX_EXPERTS], first[PK_MAX_EXPERTS], wave_sums[16];
  int cols = 1;
  while (cols < E) cols <<= 1;
  const int G = 1024 / cols;
  const int e = threadIdx.x % cols, g = threadIdx.x / cols;
  const int cpg = (nchunks + G - 1) / G;
  const int c0 = g * cpg, c1 = min(nchunks, c0 + cpg);
  constexpr int WALK = 8;
  int mine = 0;
  if (e < E)
    for (int c = c0; c < c1; c += WALK) {
      int v[WALK];
#pragma unroll
      for (int i = 0; i < WALK; ++i) v[i] = c + i < c1 ? chunk_hist[(int64_t)(c + i) * E + e] : 0;
#pragma unroll
      for (int i = 0; i < WALK; ++i) mine += v[i];
    }
  part[threadIdx.x] = mine;
  __syncthreads();
  int total = 0, before = 0;           // rows of expert e in all chunks / in the chunks of earlier groups
  for (int k = 0; k < G; ++k) {
    const int v = part[k * cols + e];
    total += v;
    before += k < g ? v : 0;
  }
  const int start = block_exclusive_scan(g == 0 ? total : 0, wave_sums);      // (columns past E hold zeros)
  if (g == 0 && e < E) {
    cnt[e] = total;
    first[e] = start;
    if (counts) counts[e] = total;
    starts[e] = start;
    if (e == E - 1) starts[E] = start + total;
  }
  __syncthreads();
  if (e < E) {
    int run = first[e] + before;
    for (int c = c0; c < c1; c += WALK) {
      int v[WALK];
#pragma unroll
      for (int i = 0; i < WALK; ++i) v[i] = c + i < c1 ? chunk_hist[(int64_t)(c + i) * E + e] : 0;
#pragma unroll
      for (int i = 0; i < WALK; ++i)
        if (c + i < c1) {
          chunk_hist[(int64_t)(c + i) * E + e] = run;
          run += v[i];
        }
    }
  }
  __syncthreads();
  if (order) write_order(cnt, first, E, order);
}

// After sort_hist_kernel one workgroup per chunk works out for itself where every expert starts and how
// many of its rows come from earlier chunks -- all of them read all the chunk histograms, a few tens of kB
// out of the L2, which is quicker than sort_scan_kernel in between that everybody waits for -- and then
// places its chunk with four waves.  Workgroup 0 also writes counts, starts and order.  What is read grows
// with the square of the chunks, so SCANNED leaves it to sort_scan_kernel beyond self_scan_chunks.
constexpr int kScatterThreads = 1024, kScatterWaves = 4;
// Where the two ways meet.  The whole sort, us, without -> with the scan kernel:
//   experts      513 chunks       1,024 chunks     2,048 chunks      8,192 chunks
//        8      12.2 -> 16.4      15.6 -> 19.5     30.0 -> 25.7       191 -> 65
//       32      15.5 -> 16.7      24.3 -> 21.5     59.5 -> 31.8       593 -> 96
//      128      29.3 -> 26.0      57.8 -> 39.7      171 -> 68        2910 -> 236
//    1,024       159 -> 171        410 -> 269      1537 -> 472
inline int self_scan_chunks(int64_t E) { return E <= 16 ? 1024 : 512; }
template <bool SCANNED>
__global__ __launch_bounds__(kScatterThreads) void sort_scatter_kernel(const int32_t* __restrict__ idx, int A, int E, int chunk_slots,
                                                                       const int32_t* __restrict__ chunk_hist, int nchunks,
                                                                       int32_t* __restrict__ counts, int32_t* __restrict__ starts,
                                                                       int32_t* __restrict__ perm, int32_t* __restrict__ inv_perm,
                                                                       int32_t* __restrict__ order) {
  extern __shared__ int32_t lds[];                   // cnt [E], before [E], cursor [kScatterWaves][E]
  __shared__ int32_t wave_sums[kScatterThreads / 64];
  int32_t* const cnt = lds;
  int32_t* const before = lds + E;
  int32_t* const cursor = lds + 2 * E;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int chunk = blockIdx.x;
  for (int i = threadIdx.x; i < (2 + kScatterWaves) * E; i += blockDim.x) lds[i] = 0;
  __syncthreads();
  if constexpr (!SCANNED) {
    // 1024 threads = G groups of E columns; group g adds up chunks g, g + G, ..., eight loads at a time
    int cols = 1;
    while (cols < E) cols <<= 1;
    const int e = threadIdx.x % cols, g = threadIdx.x / cols, G = blockDim.x / cols;
    constexpr int WALK = 8;
    int total = 0, early = 0;
    if (e < E)
      for (int c = g; c < nchunks; c += G * WALK) {
        int v[WALK];
#pragma unroll
        for (int i = 0; i < WALK; ++i) v[i] = c + i * G < nchunks ? chunk_hist[(int64_t)(c + i * G) * E + e] : 0;
#pragma unroll
        for (int i = 0; i < WALK; ++i) {
          total += v[i];
          early += c + i * G < chunk ? v[i] : 0;
        }
      }
    if (e < E) {
      atomicAdd(&cnt[e], total);
      atomicAdd(&before[e], early);
    }
  }
  // the wave's own share of the chunk, counted before anything is placed
  const int per = ((chunk_slots + kScatterWaves - 1) / kScatterWaves + 63) & ~63;      // slots of a wave
  const int s0 = chunk * chunk_slots + wave * per, n = min(per, chunk_slots - wave * per);
  if (wave < kScatterWaves)
    for (int i = lane; i < n; i += 64) {
      const int s = s0 + i;
      if (s < A) {
        const int e = idx[s];
        if ((unsigned)e < (unsigned)E) atomicAdd(&cursor[wave * E + e], 1);
      }
    }
  __syncthreads();
  const int e = threadIdx.x;
  const int total = !SCANNED && e < E ? cnt[e] : 0;
  const int start = SCANNED ? 0 : block_exclusive_scan(total, wave_sums);
  if (e < E) {
    int run = SCANNED ? chunk_hist[(int64_t)chunk * E + e] : start + before[e];
#pragma unroll
    for (int w = 0; w < kScatterWaves; ++w) {
      const int placed = cursor[w * E + e];
      cursor[w * E + e] = run;
      run += placed;
    }
    if (!SCANNED && chunk == 0) {
      if (counts) counts[e] = total;
      starts[e] = start;
      if (e == E - 1) starts[E] = start + total;
    }
  }
  __syncthreads();
  if (wave < kScatterWaves) place_slots(idx, s0, n, A, E, id_bits_for(E), cursor + wave * E, perm, inv_perm);
  if (!SCANNED && chunk == 0 && order) write_order(cnt, before, E, order);
}

// ------------------------------------------------------------------ norm, gate and top-k in one launch
// A workgroup takes 16 tokens through the whole front of the region: the norm (its rows stay in LDS), the gate's
// products, softmax and top-k, and the histogram of the chosen experts that sort_scatter_kernel wants.  What it replaces is
// four or five launches of 3 to 14 us each that are mostly latency: see front_pays for where it pays.
// The products are those of pk_x3mm::kernel, plane by plane and split by split, so that the logits are the same bit for
// bit: a wave takes one split of the reduction for 32 experts, splits the weights into their three planes on the way
// through LDS that only it uses (no barriers), and the waves' sums are added in the order of the splits.  Half of a
// 32 x 32 MFMA tile has no tokens; with 32 a workgroup there are half as many workgroups, and the matrix cores are not
// what is waited for: splitting the weights, once per 16 tokens, is.
constexpr int kFrontTokens = 16, kFrontWaves = 8, kFrontExperts = 128, kFrontMaxVecs = 4;
constexpr int64_t kFrontRowBytes = 64 * kFrontMaxVecs * 16;      // a row of x: 4 KB, 64 KB of LDS for 16 of them
struct Front {
  const void* x;              // [T, H]
  const void* norm_w;         // [H], or nullptr: no norm
  void* xn;                   // the norm's outputs
  float* rstd;                //   (optional)
  const float* w;
  const float* bias;          // optional
  float* logits;
  float* top_scores;          // nullptr: logits only
  int32_t* top_idx;
  int32_t* chunk_hist;        // [workgroups][E], optional
  int32_t T, H, E, K, route_norm;
  int32_t splits, kchunk;     // of the reduction: as many, and as deep, as pk_x3mm::kernel has them
  float eps, route_scale;
};
__host__ __device__ inline int front_row_stride(int H, int es) { return (H + 31) / 32 * 32 * es + 16; }
inline size_t front_lds_bytes(int64_t H, int es, int experts_padded) {
  const size_t rows = (size_t)kFrontTokens * front_row_stride((int)H, es);
  const size_t sums = (size_t)(kFrontWaves + 1) * kFrontTokens * experts_padded * sizeof(float);
  return rows > sums ? rows : sums;
}
template <typename TX, int ET, int VECS>      // tiles of 32 experts; 16-byte vectors of a row that a lane holds
__global__ __launch_bounds__(64 * kFrontWaves) void gate_front_kernel(const Front p) {
  constexpr int N = PkVec16<TX>::N, ES = (int)sizeof(TX), EP = 32 * ET, EPL = (EP + 63) / 64;
  constexpr int PA = pk_x3mm::Planes<TX>::N, PB = 3, LDK = pk_x3mm::LDK;
  extern __shared__ __attribute__((aligned(16))) char front_lds[];
  __shared__ int32_t hist[kFrontExperts];
  __shared__ __attribute__((aligned(16))) bf16_t planes_lds[kFrontWaves][PB][32 * LDK];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int H = p.H, nv = H / N, ld = front_row_stride(H, ES);
  const int t0 = blockIdx.x * kFrontTokens;

  // ---- everything that does not depend on anything is requested first: the rows, the norm's weight, the first piece of the
  // gate's (no branch in between, or the compiler waits for all of it at the first use).  Past an end: the last one again.
  constexpr int ROWS = kFrontTokens / kFrontWaves;
  typedef decltype(PkVec16<TX>::v) vec_t;
  PkVec16<TX> v[ROWS][VECS], nw[VECS];
#pragma unroll
  for (int h = 0; h < ROWS; ++h) {
    const vec_t* src = reinterpret_cast<const vec_t*>(reinterpret_cast<const TX*>(p.x) + (int64_t)min(t0 + wave + h * kFrontWaves, p.T - 1) * H);
#pragma unroll
    for (int m = 0; m < VECS; ++m) v[h][m].v = src[min(lane + 64 * m, nv - 1)];
  }
  {
    const vec_t* src = reinterpret_cast<const vec_t*>(p.norm_w ? p.norm_w : p.x);
#pragma unroll
    for (int m = 0; m < VECS; ++m) nw[m].v = src[min(lane + 64 * m, nv - 1)];
  }
  // the wave's q-th share: split z of the reduction for 32 experts from 32 tile on (pieces: 32-deep steps; 0: no share)
  const int tiles = (p.E + 31) / 32;
  auto share = [&](int q, int& z, int& tile, int& k0, int& pieces) {
    const int i = wave + q * kFrontWaves;
    z = i % p.splits;
    tile = i / p.splits;
    k0 = z * p.kchunk;
    pieces = tile < tiles ? (min(p.kchunk, H - k0) + 31) >> 5 : 0;
  };
  struct Regs { floatx4_t w[4]; };      // 32 rows of w, 32 deep: eight lanes to a row
  auto request = [&](Regs& q, int tile, int k0) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int e = min(32 * tile + 8 * i + (lane >> 3), p.E - 1), k = k0 + 4 * (lane & 7);      // (a column that is not stored)
      q.w[i] = *reinterpret_cast<const floatx4_t*>(p.w + (int64_t)e * H + (k < H ? k : 0));      // (set to zero below)
    }
  };
  int z, tile, k0, pieces;
  share(0, z, tile, k0, pieces);
  Regs cur;
  request(cur, min(tile, tiles - 1), k0 < H ? k0 : 0);

  // ---- rows into LDS, normalised on the way: y = x * rstd * w as rmsnorm_fwd_kernel computes it, with the sums of its four
  // waves kept apart and added in its order, so that the result is the same bit for bit
#pragma unroll
  for (int h = 0; h < ROWS; ++h)
#pragma unroll
    for (int m = 0; m < VECS; ++m)
#pragma unroll
      for (int i = 0; i < N; ++i)
        if (lane + 64 * m >= nv) v[h][m].set(i, 0.f);
  if (p.norm_w) {
    float rs[ROWS];
#pragma unroll
    for (int h = 0; h < ROWS; ++h) {
      float ss[4] = {0.f, 0.f, 0.f, 0.f}, sum = 0.f;
#pragma unroll
      for (int m = 0; m < VECS; ++m)
#pragma unroll
        for (int i = 0; i < N; ++i) ss[m & 3] = fmaf(v[h][m].get(i), v[h][m].get(i), ss[m & 3]);
#pragma unroll
      for (int c = 0; c < 4; ++c) sum += c < VECS ? pk_wave_sum(ss[c]) : 0.f;
      rs[h] = rsqrtf(sum / (float)H + p.eps);
    }
#pragma unroll
    for (int h = 0; h < ROWS; ++h)
#pragma unroll
      for (int m = 0; m < VECS; ++m)
#pragma unroll
        for (int i = 0; i < N; ++i) v[h][m].set(i, (v[h][m].get(i) * rs[h]) * nw[m].get(i));
#pragma unroll
    for (int h = 0; h < ROWS; ++h) {
      const int t = t0 + wave + h * kFrontWaves;
      if (t >= p.T) continue;
      if (lane == 0 && p.rstd) p.rstd[t] = rs[h];
      vec_t* const dst = reinterpret_cast<vec_t*>(reinterpret_cast<TX*>(p.xn) + (int64_t)t * H);
#pragma unroll
      for (int m = 0; m < VECS; ++m)
        if (lane + 64 * m < nv) dst[lane + 64 * m] = v[h][m].v;
    }
  }
#pragma unroll
  for (int h = 0; h < ROWS; ++h) {
    char* const row = front_lds + (wave + h * kFrontWaves) * ld;
#pragma unroll
    for (int m = 0; m < VECS; ++m)
      if (lane + 64 * m < nv) reinterpret_cast<vec_t*>(row)[lane + 64 * m] = v[h][m].v;
    if (H + lane < (H + 31) / 32 * 32) reinterpret_cast<TX*>(row)[H + lane] = pk_from_float<TX>(0.f);
  }
  if (tid < kFrontExperts) hist[tid] = 0;
  __syncthreads();

  // ---- products
  auto& planes = planes_lds[wave];
  float keep[ET][8];
#pragma unroll
  for (int q = 0; q < ET; ++q) {
    floatx16_t acc;
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[i] = 0.f;
    int z2, tile2, k2, pieces2;
    share(q + 1, z2, tile2, k2, pieces2);
    if (pieces <= 0 && q + 1 < ET && pieces2 > 0) request(cur, tile2, k2);      // (a split past the end)
    for (int n = 0; n < pieces; ++n, k0 += 32) {
      const Regs now = cur;
      if (n + 1 < pieces) request(cur, tile, k0 + 32);
      else if (q + 1 < ET && pieces2 > 0) request(cur, tile2, k2);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        pk_x3mm::Raw<float> raw;
        raw.v = now.w[i];
        if (k0 + 4 * (lane & 7) >= H) pk_x3mm::zero_raw<float>(raw);
        bf16x4_t pl[PB];
        pk_x3mm::to_planes<float>(raw, pl);
#pragma unroll
        for (int b = 0; b < PB; ++b) *reinterpret_cast<bf16x4_t*>(&planes[b][(8 * i + (lane >> 3)) * LDK + 4 * (lane & 7)]) = pl[b];
      }
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
      for (int kk = 0; kk < 32; kk += 16) {
        bf16x8_t a[PA], b[PB];
        const TX* src = reinterpret_cast<const TX*>(front_lds + (lane & 15) * ld) + k0 + kk + 8 * (lane >> 5);      // rows 16..31: again
        if constexpr (PA == 1) {
          a[0] = *reinterpret_cast<const bf16x8_t*>(src);
        } else {
#pragma unroll
          for (int half = 0; half < 2; ++half) {
            pk_x3mm::Raw<float> raw;
            raw.v = *reinterpret_cast<const floatx4_t*>(src + 4 * half);
            bf16x4_t pl[PB];
            pk_x3mm::to_planes<float>(raw, pl);
#pragma unroll
            for (int c = 0; c < PA; ++c)
#pragma unroll
              for (int i = 0; i < 4; ++i) a[c][4 * half + i] = pl[c][i];
          }
        }
#pragma unroll
        for (int c = 0; c < PB; ++c) b[c] = pk_x3mm::frag_kc(planes[c], 0, kk, lane);
#pragma unroll
        for (int s = PA + PB - 2; s >= 0; --s)      // small terms first
#pragma unroll
          for (int pa = 0; pa < PA; ++pa) {
            const int pb = s - pa;
            if (pb >= 0 && pb < PB && s <= 2) acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[pa], b[pb], acc, 0, 0, 0);
          }
      }
      // the next piece's planes go to where other lanes have just read
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) keep[q][i] = acc[i];
    z = z2; tile = tile2; k0 = k2; pieces = pieces2;
  }
  __syncthreads();                         // the rows have been read for the last time
  // keep[q][i]: token 8 (i / 4) + 4 (l / 32) + i % 4, expert l % 32 of the q-th share
  float* const part = reinterpret_cast<float*>(front_lds);                       // [split][token][EP]
  float* const sums = part + kFrontWaves * kFrontTokens * EP;                    // [token][EP]
#pragma unroll
  for (int q = 0; q < ET; ++q) {
    share(q, z, tile, k0, pieces);
    if (tile < tiles) {
#pragma unroll
      for (int i = 0; i < 8; ++i)
        part[(z * kFrontTokens + 8 * (i >> 2) + 4 * (lane >> 5) + (i & 3)) * EP + 32 * tile + (lane & 31)] = keep[q][i];
    }
  }
  __syncthreads();
  for (int i = tid; i < kFrontTokens * EP; i += 64 * kFrontWaves) {
    const int r = i / EP, e = i % EP;
    float s = 0.f;
    for (int w = 0; w < p.splits; ++w) s += part[w * kFrontTokens * EP + i];
    if (e < p.E) {
      if (p.bias) s += p.bias[e];
      if (t0 + r < p.T) p.logits[(int64_t)(t0 + r) * p.E + e] = s;
    }
    sums[i] = s;
  }
  if (!p.top_scores) return;
  __syncthreads();
  float val[ROWS][EPL], score[ROWS];
  int expert[ROWS];
#pragma unroll
  for (int h = 0; h < ROWS; ++h)
#pragma unroll
    for (int j = 0; j < EPL; ++j) val[h][j] = lane + 64 * j < p.E ? sums[(wave + h * kFrontWaves) * EP + lane + 64 * j] : 0.f;
  topk_of<EPL, ROWS>(val, lane, p.E, p.K, p.route_norm, p.route_scale, score, expert);
#pragma unroll
  for (int h = 0; h < ROWS; ++h) {
    const int64_t t = t0 + wave + h * kFrontWaves;
    if (t < p.T && lane < p.K) {
      p.top_scores[t * p.K + lane] = score[h];
      p.top_idx[t * p.K + lane] = expert[h];
      atomicAdd(&hist[expert[h]], 1);
    }
  }
  if (!p.chunk_hist) return;
  __syncthreads();
  if (tid < p.E) p.chunk_hist[(int64_t)blockIdx.x * p.E + tid] = hist[tid];
}

__global__ __launch_bounds__(1024) void counts_to_starts_kernel(const void* __restrict__ counts,
                                                                int is_i64, int E,
                                                                int32_t* __restrict__ starts) {
  __shared__ int32_t scan[PK_MAX_EXPERTS];
  const int e = threadIdx.x;
  int c = 0;
  if (e < E) c = is_i64 ? (int)reinterpret_cast<const int64_t*>(counts)[e]
                        : reinterpret_cast<const int32_t*>(counts)[e];
  scan[e] = c;
  __syncthreads();
  for (int off = 1; off < 1024; off <<= 1) {
    const int v = (e >= off) ? scan[e - off] : 0;
    __syncthreads();
    scan[e] += v;
    __syncthreads();
  }
  if (e < E) {
    starts[e] = scan[e] - c;
    if (e == E - 1) starts[E] = scan[e];
  }
}

// ------------------------------------------------------------------ small helpers
// d_bias[e] (+)= sum_t d_logits[t,e]; one block per expert
__device__ __forceinline__ void colsum(int e, const float* __restrict__ d_logits, int64_t T, int E, float* __restrict__ d_bias, int accumulate,
                                       float* red /* 16 floats of LDS */) {
  float s = 0.f;
  for (int64_t t = threadIdx.x; t < T; t += 256) s += d_logits[t * E + e];
  s = pk_block_sum(s, red);
  if (threadIdx.x == 0) d_bias[e] = accumulate ? d_bias[e] + s : s;
}
__global__ __launch_bounds__(256) void colsum_kernel(const float* __restrict__ d_logits, int64_t T, int E, float* __restrict__ d_bias,
                                                     int accumulate) {
  __shared__ float red[16];
  colsum(blockIdx.x, d_logits, T, E, d_bias, accumulate, red);
}

// The same sum for long inputs in two steps with contiguous reads: block b adds up the rows
// [b * per, (b+1) * per) of d_logits (256 threads = RP rows x E/4 column groups of 16 bytes, a
// thread walks every RP-th row with eight rows in flight, the RP partial rows are added in order
// through LDS), then one thread per column adds the kColsumBlocks partial rows in block order.
// One block per expert reading a column touches every cache line of d_logits from every XCD.
inline bool colsum_in_parts(int64_t T, int64_t E) { return T >= 32 * kColsumBlocks && E % 4 == 0 && E <= 1024; }
__device__ __forceinline__ void colsum_partial(int block, int nblocks, const float* __restrict__ d_logits, int64_t T, int E,
                                               float* __restrict__ part, float* red /* 1,024 floats of LDS */) {
  const int cols4 = E / 4, RP = 256 / cols4;
  const int r = threadIdx.x / cols4, c = threadIdx.x % cols4;
  const int64_t per = (T + nblocks - 1) / nblocks;
  const int64_t t0 = (int64_t)block * per, t1 = t0 + per < T ? t0 + per : T;
  float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
  if (r < RP) {
    const float4* src = reinterpret_cast<const float4*>(d_logits) + c;
    int64_t t = t0 + r;
    for (; t + 7 * RP < t1; t += 8 * RP) {
      float4 v[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) v[i] = src[(t + i * RP) * cols4];
#pragma unroll
      for (int i = 0; i < 8; ++i) { acc.x += v[i].x; acc.y += v[i].y; acc.z += v[i].z; acc.w += v[i].w; }
    }
    for (; t < t1; t += RP) {
      const float4 v = src[t * cols4];
      acc.x += v.x; acc.y += v.y; acc.z += v.z; acc.w += v.w;
    }
    reinterpret_cast<float4*>(red)[r * cols4 + c] = acc;
  }
  __syncthreads();
  for (int e = threadIdx.x; e < E; e += 256) {
    float s = 0.f;
    for (int q = 0; q < RP; ++q) s += red[q * E + e];
    part[(int64_t)block * E + e] = s;
  }
}
__global__ __launch_bounds__(256) void colsum_partial_kernel(const float* __restrict__ d_logits, int64_t T, int E, float* __restrict__ part) {
  __shared__ float red[1024];
  colsum_partial(blockIdx.x, gridDim.x, d_logits, T, E, part, red);
}

// What the router's backward owes once d_logits is there, in one launch: blocks [0, w_blocks) are output tiles of the
// gate weight gradient (split over the tokens), then come the partial column sums for the gate bias, then the tiles of
// the region's input gradient.  None of them fills the chip for long at a few thousand tokens or fewer, and
// each needs nothing from the others (1,030 tokens, 1000 wide, 24 experts: 7.5 + 5.8 us in two launches, 8.0 in one; with
// the partial sums added up by blocks of the norm's backward 24 -> 14.4 us, the training step 191 -> 182).
struct RouterGrads {
  pk_f32mm::Params w, x;
  pk_x3mm::GatherAdd gather;
  int32_t w_blocks, w_nx, w_ny, col_blocks, gather_nx;
  float* col_part;            // where the column sums go: partial sums of kColsumBlocks row ranges,
  float* d_bias;              //   or without them the gradient itself, a block per expert
  int32_t accumulate;
};
template <typename TX, bool STREAM>
__global__ __launch_bounds__(256, 4) void router_grads_kernel(const RouterGrads p) {
  using namespace pk_x3mm;
  typedef Lds<2, 2, false, false, split3_t, TX> WLds;
  constexpr int GATHER = GatherLds<kGatherWM, kGatherWN>::BYTES, BYTES = (int)sizeof(WLds) > GATHER ? (int)sizeof(WLds) : GATHER;
  static_assert(BYTES >= 4096, "the column sums' LDS");
  __shared__ __attribute__((aligned(16))) char smem[BYTES];
  int b = blockIdx.x;
  if (b < p.w_blocks) {
    const int xy = p.w_nx * p.w_ny, z = b / xy;
    b -= z * xy;
    gemm_tile<2, 2, false, false, split3_t, TX>(p.w, *reinterpret_cast<WLds*>(smem), b % p.w_nx, b / p.w_nx, z);
    return;
  }
  b -= p.w_blocks;
  if (b < p.col_blocks) {
    const float* d_logits = reinterpret_cast<const float*>(p.x.A);
    float* const red = reinterpret_cast<float*>(smem);
    if (p.col_part) colsum_partial(b, p.col_blocks, d_logits, p.x.M, (int)p.x.K, p.col_part, red);
    else colsum(b, d_logits, p.x.M, (int)p.x.K, p.d_bias, p.accumulate, red);
    return;
  }
  b -= p.col_blocks;
  gather_tile<kGatherWM, kGatherWN, TX, STREAM>(p.x, p.gather, smem, b % p.gather_nx, b / p.gather_nx);
}

// Scratch of pk_sort_by_expert_static: the per-chunk histograms of the counting sort.  Every GPU
// the library runs on holds its own copy of the array (PK_SORT_STATIC_WORDS * 4 bytes) until the
// process ends.  In host code the name `scratch` is only a handle for hipGetSymbolAddress: the
// address a kernel can use is looked up once per device, with that device current, and kept.
static __device__ __align__(256) int32_t scratch[PK_SORT_STATIC_WORDS];

int32_t* sort_scratch_for_current_device() {
  constexpr int MAX_DEV = PK_MAX_DEVICES;
  static int32_t* ptr[MAX_DEV] = {};
  static std::mutex mu;
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= MAX_DEV) return nullptr;
  std::lock_guard<std::mutex> lock(mu);
  if (!ptr[dev]) {
    void* p = nullptr;
    if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess || !p) return nullptr;
    ptr[dev] = static_cast<int32_t*>(p);
  }
  return ptr[dev];
}

}  // namespace

extern "C" {

int pk_version(void) { return 100; }

int pk_init(void) {
  if (!sort_scratch_for_current_device()) return PK_ERR_UNSUPPORTED;
  return pk_init_grouped_gemm();
}

const char* pk_status_string(int status) {
  switch (status) {
    case PK_OK: return "ok";
    case PK_ERR_ARG: return "invalid argument (null pointer, negative size or bad enum)";
    case PK_ERR_SHAPE: return "shape not supported by the kernels";
    case PK_ERR_ALIGN: return "pointer or leading dimension is not 16-byte aligned";
    case PK_ERR_WORKSPACE: return "workspace too small";
    case PK_ERR_UNSUPPORTED: return "dtype/option combination not supported";
    default: return status > 0 ? "HIP runtime error (status is the hipError_t value)" : "unknown status";
  }
}

// Splits of the router's forward reduction: 128 deep, up to eight.  Where the row tiles leave CUs idle the GEMM takes as
// long as one workgroup's k-tiles (512 wide, 1,000 tokens, 256 -> 128 deep: training step 238 -> 234 us, 1024 wide
// op by op 246 -> 234 us); gate_gemm halves the splits again where rows are many.
static int gate_fwd_splits(int64_t H) {
  int64_t sp = H / 128;
  return (int)(sp < 1 ? 1 : (sp > 8 ? 8 : sp));
}

// The reduction is split only as far as it takes to give every CU two workgroups: each split
// writes and re-reads a [T, E] fp32 partial result, which soon outweighs reading x.
static int gate_splits(int64_t T, int64_t H) {
  int sp = gate_fwd_splits(H);
  while (sp > 1 && pk_ceil_div(T, 64) * (sp / 2) >= 512) sp /= 2;
  return sp;
}

static int64_t align256(int64_t n) { return (n + 255) / 256 * 256; }
// bytes of the three bf16 planes of an fp32 array of n elements (0: cannot be pre-split)
static int64_t plane_bytes(int64_t n) { return n % 4 == 0 ? align256(3 * n * (int64_t)sizeof(bf16_t)) : 0; }
// fp32 [n] -> bf16 planes [3][n] at dst
static int split_planes(const float* src, bf16_t* dst, int64_t n, int kernel_id, hipStream_t s) {
  PK_LAUNCH_NOCHECK(kernel_id, s, pk_x3mm::split_planes_kernel, dim3((unsigned)pk_ceil_div(n, 1024)), dim3(256), 0, s, src, dst, n);
  PK_RETURN_IF_LAUNCH_FAILED();
  return PK_OK;
}

static int64_t gate_fwd_partial_bytes(int64_t T, int64_t H, int64_t E) {
  const int sp = gate_fwd_splits(H);
  return sp > 1 ? (int64_t)sp * T * E * (int64_t)sizeof(float) : 0;
}

int64_t pk_gate_workspace_bytes(int64_t T, int64_t H, int64_t E) {
  if (T < 0 || H <= 0 || E <= 0) return PK_ERR_ARG;
  return gate_fwd_partial_bytes(T, H, E);
}

}  // extern "C"

// The gate for a few tokens: one wave per expert and TOKENS tokens, lanes along the reduction, fp32 FMAs.
// The GEMM pads the tokens to 64 and walks the reduction in latency-bound k-tiles: 14 us at one token,
// 18 us at 24 (width 2048, 128 experts); here the loads of eight steps are in flight at once.
constexpr int kGateTokens = 4, kGateSmallMax = 64;
template <typename T, int TOKENS>
__global__ __launch_bounds__(256) void gate_small_kernel(const T* __restrict__ x, const float* __restrict__ w, const float* __restrict__ bias,
                                                         float* __restrict__ logits, int tokens, int H, int E) {
  constexpr int STEPS = TOKENS == 1 ? 8 : 4;
  const int lane = threadIdx.x & 63;
  const int e = blockIdx.x * 4 + (threadIdx.x >> 6);
  const int t0 = blockIdx.y * TOKENS;
  if (e >= E) return;
  float acc[TOKENS];
  const T* xr[TOKENS];
#pragma unroll
  for (int j = 0; j < TOKENS; ++j) {
    acc[j] = 0.f;
    xr[j] = x + (int64_t)min(t0 + j, tokens - 1) * H;      // past the end: the last token again, not stored
  }
  const float* wr = w + (int64_t)e * H;
  for (int k0 = 4 * lane; k0 < H; k0 += 256 * STEPS) {
    float wv[STEPS][4], xv[STEPS][TOKENS][4];
#pragma unroll
    for (int s = 0; s < STEPS; ++s) {
      const int k = k0 + 256 * s;
      const int kk = k < H ? k : 0;
      pk_f32mm::load4<float>(wr + kk, wv[s]);
#pragma unroll
      for (int j = 0; j < TOKENS; ++j) pk_f32mm::load4<T>(xr[j] + kk, xv[s][j]);
    }
#pragma unroll
    for (int s = 0; s < STEPS; ++s)
      if (k0 + 256 * s < H) {
#pragma unroll
        for (int j = 0; j < TOKENS; ++j)
#pragma unroll
          for (int i = 0; i < 4; ++i) acc[j] = fmaf(xv[s][j][i], wv[s][i], acc[j]);
      }
  }
#pragma unroll
  for (int j = 0; j < TOKENS; ++j) {
    const float s = wave_sum_f32(acc[j]);
    if (lane == 0 && t0 + j < tokens) logits[(int64_t)(t0 + j) * E + e] = s + (bias ? bias[e] : 0.f);
  }
}

// The norm and the gate for a few tokens in one launch: a workgroup takes four experts of one token and computes the token's
// norm for itself, as rmsnorm_fwd_kernel does (256 threads, the same sums); the products are those of gate_small_kernel,
// so that both results are the same bit for bit.  One token, 2048 x 128 experts: 2.4 + 3.0 us in two launches, 4.5 in one.
template <typename TX, bool NORM>
__global__ __launch_bounds__(256) void norm_gate_small_kernel(const TX* __restrict__ x, const TX* __restrict__ norm_w, float eps, TX* __restrict__ xn,
                                                              float* __restrict__ rstd, const float* __restrict__ w, const float* __restrict__ bias,
                                                              float* __restrict__ logits, int H, int E) {
  constexpr int N = PkVec16<TX>::N;
  typedef decltype(PkVec16<TX>::v) vec_t;
  extern __shared__ __attribute__((aligned(16))) char gate_row[];
  __shared__ float red[16];
  TX* const row = reinterpret_cast<TX*>(gate_row);
  const int lane = threadIdx.x & 63, t = blockIdx.y, nv = H / N;
  const int e = blockIdx.x * 4 + (threadIdx.x >> 6);
  // the first 2,048 columns of the weight and the bias: requested in front of the norm
  constexpr int STEPS = 8;
  const float* const wr = w + (int64_t)min(e, E - 1) * H;
  floatx4_t wv[STEPS];
#pragma unroll
  for (int s = 0; s < STEPS; ++s) wv[s] = *reinterpret_cast<const floatx4_t*>(wr + min(4 * lane + 256 * s, H - 4));
  const float b = bias ? bias[min(e, E - 1)] : 0.f;
  const TX* const src = x + (int64_t)t * H;
  float ss = 0.f;
  for (int v = threadIdx.x; v < nv; v += 256) {
    PkVec16<TX> f;
    f.v = reinterpret_cast<const vec_t*>(src)[v];
    reinterpret_cast<vec_t*>(row)[v] = f.v;
    if (NORM) {
#pragma unroll
      for (int i = 0; i < N; ++i) ss = fmaf(f.get(i), f.get(i), ss);
    }
  }
  if (NORM) {
    const float rs = rsqrtf(pk_block_sum(ss, red) / (float)H + eps);
    if (rstd && blockIdx.x == 0 && threadIdx.x == 0) rstd[t] = rs;
    for (int v = threadIdx.x; v < nv; v += 256) {
      PkVec16<TX> f, g;
      f.v = reinterpret_cast<vec_t*>(row)[v];
      g.v = reinterpret_cast<const vec_t*>(norm_w)[v];
#pragma unroll
      for (int i = 0; i < N; ++i) f.set(i, (f.get(i) * rs) * g.get(i));
      reinterpret_cast<vec_t*>(row)[v] = f.v;
      if (blockIdx.x == 0) reinterpret_cast<vec_t*>(xn + (int64_t)t * H)[v] = f.v;
    }
  }
  __syncthreads();
  if (e >= E) return;
  float acc = 0.f;
  for (int k0 = 4 * lane; k0 < H; k0 += 256 * STEPS) {
    float xv[STEPS][4];
#pragma unroll
    for (int s = 0; s < STEPS; ++s) pk_f32mm::load4<TX>(row + min(k0 + 256 * s, H - 4), xv[s]);
    if (k0 != 4 * lane) {
#pragma unroll
      for (int s = 0; s < STEPS; ++s) wv[s] = *reinterpret_cast<const floatx4_t*>(wr + min(k0 + 256 * s, H - 4));
    }
#pragma unroll
    for (int s = 0; s < STEPS; ++s)
      if (k0 + 256 * s < H) {
#pragma unroll
        for (int i = 0; i < 4; ++i) acc = fmaf(xv[s][i], wv[s][i], acc);
      }
  }
  acc = wave_sum_f32(acc);
  if (lane == 0) logits[(int64_t)t * E + e] = acc + b;
}

constexpr int64_t kNormGateMaxWidth = 8192;      // columns of a row in LDS
// (declared where it is used as well: decode.hip)
int pk_norm_gate_small(const void* x, int dtype, const void* norm_w, float eps, void* xn, float* rstd, const float* w_gate, const float* gate_bias,
                       float* logits, int64_t T, int64_t H, int64_t E, hipStream_t s) {
  const dim3 grid((unsigned)pk_ceil_div(E, 4), (unsigned)T), block(256);
#define PK_NORM_GATE(TYPE, NORM)                                                                                                  \
  PK_LAUNCH_NOCHECK(pk_timing::K_GATE_LOGITS, s, (norm_gate_small_kernel<TYPE, NORM>), grid, block, (size_t)H * sizeof(TYPE), s, (const TYPE*)x, \
                    (const TYPE*)norm_w, eps, (TYPE*)xn, rstd, w_gate, gate_bias, logits, (int)H, (int)E)
  if (dtype == PK_BF16) { if (norm_w) PK_NORM_GATE(bf16_t, true); else PK_NORM_GATE(bf16_t, false); }
  else { if (norm_w) PK_NORM_GATE(float, true); else PK_NORM_GATE(float, false); }
#undef PK_NORM_GATE
  PK_RETURN_IF_LAUNCH_FAILED();
  return PK_OK;
}

// Whether gate_front_kernel takes a gate of these sizes.  It gives the bits of the launches that it replaces, so each entry point
// has its own answer: how many launches those are.  Every workgroup reads all of w_gate and splits it, for whole tiles of 32
// experts: some 5 us in bf16, with top-k, sort and norm 12, and 0.12 us for 1,024 elements of that; in fp32 half as much again
// (x is split as well).  The launches it replaces hardly depend on the weight's size, but on the tokens.  Us, those -> this one
// (launched back to back, graph; top 4):
//                             65 tokens      1,024        2,048        4,096        4,097        8,192
//   norm .. sort, 1024 x  24  16.5 -> 13.6   21 -> 14     25 -> 15     30 -> 17     30 -> 24     36 -> 29
//                 1024 x  64  17.0 -> 18.1   23 -> 19     27 -> 20     33 -> 23     34 -> 35     38 -> 38
//                  768 x 128  19.3 -> 24.3   25 -> 26     30 -> 28     40 -> 32     40 -> 47     44 -> 49
//           fp32, 1000 x  64  18.0 -> 24.6   25 -> 26     30 -> 28     35 -> 31     35 -> 50     44 -> 56
//   gate .. sort,  768 x  64                              21 -> 17
//                 2048 x  24  16.1 -> 17.2                                          24 -> 29     31 -> 38
//   gate alone,    512 x  64   8.9 ->  6.9   10 ->  7     10 ->  7     11 ->  7     11 -> 12     15 -> 13
//                 2048 x  32  12.0 -> 11.0   13 -> 11     13 -> 11     14 -> 12     16 -> 20     20 -> 27
//                  768 x 128   9.8 -> 14.7   11 -> 16     13 -> 16     18 -> 16     19 -> 29     24 -> 30
// Once the CUs have taken a workgroup or two each (front_lds_bytes says which), the next ones wait a whole round for them.
enum FrontCall { FRONT_LOGITS, FRONT_TOPK, FRONT_SORT, FRONT_NORM };
constexpr int64_t kFrontMaxTokens = 8192;
static bool front_pays(FrontCall call, int es, int64_t T, int64_t H, int64_t E) {
  if (E * H > 96 * 1024) return false;
  const int experts = E <= 32 ? 32 : E <= 64 ? 64 : kFrontExperts;
  const bool narrow = E <= 32, long_rows = H * es > 3072;
  const int64_t work = pk_ceil_div(E, 32) * 32 * H * (es == 2 ? 2 : 3) / 2 / 1024;
  constexpr int64_t LDS = 160 * 1024, PLANES = (int64_t)kFrontWaves * 3 * 32 * pk_x3mm::LDK * 2 + kFrontExperts * 4;
  const int64_t per_cu = std::max<int64_t>(1, std::min<int64_t>(2, LDS / ((int64_t)front_lds_bytes(H, es, experts) + PLANES)));
  if (pk_ceil_div(T, kFrontTokens) > 256 * per_cu) {      // a second round
    if (call == FRONT_NORM) return narrow || (E <= 64 && work <= 32);
    return call != FRONT_TOPK && narrow && H * es <= 2048 && (work <= 16 || T > 6000);
  }
  if (call == FRONT_NORM) return work <= (T < 2048 ? 64 : 128);
  if (long_rows && (call == FRONT_SORT ? T <= 512 : call == FRONT_TOPK && T <= 2048)) return false;
  if (narrow) return work <= 64;
  return work <= (T < 1024 || (T <= 2048 && call != FRONT_SORT) ? 32 : T < 4096 ? 64 : 80);
}
static bool front_ok(FrontCall call, const void* x, int x_dtype, const void* w_gate, int64_t T, int64_t H, int64_t E) {
  const int es = (int)pk_dtype_size(x_dtype);
  if (T <= kGateSmallMax || T > kFrontMaxTokens || E > kFrontExperts || H % (16 / es) != 0 || H * es > kFrontRowBytes || !pk_aligned16(x) ||
      !pk_aligned16(w_gate))
    return false;
  return front_pays(call, es, T, H, E);
}
// Whether the sort goes by its histograms of 16 tokens each: every workgroup of sort_scatter_kernel reads all of them
// (229 of 64 experts: 8.2 us against 5.3 + 6.0 with histograms of 512 slots in a launch of their own).
static bool front_sorts(int64_t T, int64_t E) { return pk_ceil_div(T, kFrontTokens) * E <= 16 * 1024; }
static int launch_front(const Front& p, int x_dtype, hipStream_t s) {
  const dim3 grid((unsigned)pk_ceil_div(p.T, kFrontTokens)), block(64 * kFrontWaves);
  const int vecs = (int)pk_ceil_div(p.H * (int64_t)pk_dtype_size(x_dtype), 64 * 16);
#define PK_FRONT(TYPE, ET, VECS)                                                                                        \
  PK_LAUNCH_NOCHECK(pk_timing::K_GATE_LOGITS, s, (gate_front_kernel<TYPE, ET, VECS>), grid, block,                      \
                    front_lds_bytes(p.H, (int)sizeof(TYPE), 32 * ET), s, p)
#define PK_FRONT_VECS(TYPE, ET)                   \
  do {                                            \
    if (vecs <= 1) PK_FRONT(TYPE, ET, 1);         \
    else if (vecs <= 2) PK_FRONT(TYPE, ET, 2);    \
    else PK_FRONT(TYPE, ET, 4);                   \
  } while (0)
#define PK_FRONT_TYPE(TYPE)                       \
  do {                                            \
    if (p.E <= 32) PK_FRONT_VECS(TYPE, 1);        \
    else if (p.E <= 64) PK_FRONT_VECS(TYPE, 2);   \
    else PK_FRONT_VECS(TYPE, 4);                  \
  } while (0)
  if (x_dtype == PK_BF16) PK_FRONT_TYPE(bf16_t);
  else PK_FRONT_TYPE(float);
#undef PK_FRONT_TYPE
#undef PK_FRONT_VECS
#undef PK_FRONT
  PK_RETURN_IF_LAUNCH_FAILED();
  return PK_OK;
}
static Front front_params(const void* x, const float* w_gate, const float* gate_bias, float* logits, int64_t T, int64_t H, int64_t E) {
  Front p = {};
  p.x = x; p.w = w_gate; p.bias = gate_bias; p.logits = logits;
  p.T = (int32_t)T; p.H = (int32_t)H; p.E = (int32_t)E;
  p.splits = gate_splits(T, H);
  p.kchunk = (int32_t)pk_ceil_div(pk_ceil_div(H, p.splits), pk_x3mm::BK) * pk_x3mm::BK;
  return p;
}

// The gate GEMM.  *splits > 1: `workspace` holds that many partial results [T, E] and logits is not
// written yet (no bias either); otherwise the logits are complete.
static int gate_gemm(const void* x, int x_dtype, const float* w_gate, const float* gate_bias, float* logits, int64_t T, int64_t H,
                     int64_t E, void* workspace, int64_t workspace_bytes, hipStream_t s, int* splits) {
  if (T < 0 || H <= 0 || E <= 0 || !pk_dtype_ok(x_dtype)) return PK_ERR_ARG;
  *splits = 1;
  if (T == 0) return PK_OK;
  if (!x || !w_gate || !logits) return PK_ERR_ARG;
  if (T <= kGateSmallMax && H % 4 == 0 && pk_aligned16(x) && pk_aligned16(w_gate)) {
    const dim3 grid((unsigned)pk_ceil_div(E, 4), (unsigned)pk_ceil_div(T, T == 1 ? 1 : kGateTokens)), block(256);
#define PK_GATE_SMALL(TYPE, N)                                                                                                  \
  PK_LAUNCH_NOCHECK(pk_timing::K_GATE_LOGITS, s, (gate_small_kernel<TYPE, N>), grid, block, 0, s, (const TYPE*)x, w_gate, gate_bias, \
                    logits, (int)T, (int)H, (int)E)
    if (x_dtype == PK_BF16) { if (T == 1) PK_GATE_SMALL(bf16_t, 1); else PK_GATE_SMALL(bf16_t, kGateTokens); }
    else { if (T == 1) PK_GATE_SMALL(float, 1); else PK_GATE_SMALL(float, kGateTokens); }
#undef PK_GATE_SMALL
    PK_RETURN_IF_LAUNCH_FAILED();
    return PK_OK;
  }
  int sp = gate_splits(T, H);
  if (sp > 1 && (!workspace || workspace_bytes < gate_fwd_partial_bytes(T, H, E))) sp = 1;
  // (Handing this GEMM the weight already split into bf16 planes does not shorten it: the kernel
  // waits on its loads and barriers, not on the instructions of the split.)
  pk_f32mm::Params p = {};
  p.A = x; p.B = w_gate;
  p.C = sp > 1 ? reinterpret_cast<float*>(workspace) : logits;
  p.bias = sp > 1 ? nullptr : gate_bias;
  p.M = T; p.N = E; p.K = H;
  p.sam = H; p.sak = 1; p.sbk = 1; p.sbn = H;
  p.splits = sp; p.accumulate = 0;
  *splits = sp;
  const bool xb = x_dtype == PK_BF16;
  if (E > 64)  // 64-token x 128-expert tiles, 8 waves
    return xb ? pk_x3mm::launch<2, 4, true, true, bf16_t, float>(p, pk_timing::K_GATE_LOGITS, s)
              : pk_x3mm::launch<2, 4, true, true, float, float>(p, pk_timing::K_GATE_LOGITS, s);
  // 64-token x 64-expert tiles, 4 waves
  return xb ? pk_x3mm::launch<2, 2, true, true, bf16_t, float>(p, pk_timing::K_GATE_LOGITS, s)
            : pk_x3mm::launch<2, 2, true, true, float, float>(p, pk_timing::K_GATE_LOGITS, s);
}

extern "C" {

int pk_gate_logits(const void* x, int x_dtype, const float* w_gate, const float* gate_bias,
                   float* logits, int64_t T, int64_t H, int64_t E, void* workspace,
                   int64_t workspace_bytes, pk_stream_t stream) {
  hipStream_t s = (hipStream_t)stream;
  if (H > 0 && E > 0 && pk_dtype_ok(x_dtype) && x && w_gate && logits && front_ok(FRONT_LOGITS, x, x_dtype, w_gate, T, H, E))
    return launch_front(front_params(x, w_gate, gate_bias, logits, T, H, E), x_dtype, s);
  int splits = 1;
  const int rc = gate_gemm(x, x_dtype, w_gate, gate_bias, logits, T, H, E, workspace, workspace_bytes, s, &splits);
  if (rc != PK_OK || splits == 1) return rc;
  const int64_t n = T * E;
  PK_LAUNCH_NOCHECK(pk_timing::K_GATE_LOGITS, s, pk_f32mm::reduce_partials_kernel,
                    dim3((unsigned)pk_ceil_div(n, 256)), dim3(256), 0, s,
                    reinterpret_cast<const float*>(workspace), logits, n, splits, 0, gate_bias, (int)E);
  PK_RETURN_IF_LAUNCH_FAILED();
  return PK_OK;
}

// Workgroups that share the reduction over the tokens in the weight-gradient GEMM: one per 256 tokens,
// and with few output tiles (H/64 x E/64) more, down to 64 tokens each, until there are two for a CU
// (509 tokens, 512 x 16, fp32: 26 us on 8 workgroups, 9 us on 64).
static int gate_bwd_splits(int64_t T, int64_t H, int64_t E) {
  const int64_t tiles = pk_ceil_div(H, 64) * pk_ceil_div(E, 64);
  int64_t sp = T / 256, fill = 512 / tiles < T / 64 ? 512 / tiles : T / 64;
  if (fill > sp) sp = fill;
  return (int)(sp < 1 ? 1 : (sp > 16 ? 16 : sp));
}

// workspace of the backward: [partial column sums of d_logits, for the bias][split-K partials of d_w_gate]
// [d_logits as three bf16 planes, for the weight gradient]
static int64_t gate_bwd_colsum_bytes(int64_t E) { return align256((int64_t)kColsumBlocks * E * (int64_t)sizeof(float)); }
static int64_t gate_bwd_partial_bytes(int64_t T, int64_t H, int64_t E) {
  const int sp = gate_bwd_splits(T, H, E);
  return gate_bwd_colsum_bytes(E) + align256(sp > 1 ? (int64_t)sp * E * H * (int64_t)sizeof(float) : 0);
}

int64_t pk_gate_bwd_workspace_bytes(int64_t T, int64_t H, int64_t E) {
  if (T < 0 || H <= 0 || E <= 0) return PK_ERR_ARG;
  return gate_bwd_partial_bytes(T, H, E) + plane_bytes(T * E);
}

}  // extern "C"

// planes_ready: d_logits already lies split in the workspace, where this function would put it
static int gate_bwd(const float* d_logits, const void* x, int x_dtype, const float* w_gate,
                    float* d_x_f32, float* d_w_gate, float* d_gate_bias, int accumulate,
                    int64_t T, int64_t H, int64_t E, void* workspace, int64_t workspace_bytes, bool planes_ready,
                    pk_stream_t stream) {
  if (T < 0 || H <= 0 || E <= 0 || !pk_dtype_ok(x_dtype)) return PK_ERR_ARG;
  if (!d_logits && T > 0) return PK_ERR_ARG;
  hipStream_t s = (hipStream_t)stream;
  using pk_x3mm::split3_t;
  const int64_t part_bytes = gate_bwd_partial_bytes(T, H, E);
  const bool have_ws = workspace && reinterpret_cast<uintptr_t>(workspace) % 16 == 0;
  const bool have_part = have_ws && workspace_bytes >= part_bytes;
  if (d_x_f32 && T > 0) {
    if (!w_gate) return PK_ERR_ARG;
    pk_f32mm::Params p = {};
    p.A = d_logits; p.B = w_gate; p.C = d_x_f32;
    p.M = T; p.N = H; p.K = E;
    p.sam = E; p.sak = 1; p.sbk = H; p.sbn = 1;
    p.splits = 1; p.accumulate = 0;
    int rc = pk_x3mm::launch<2, 2, true, false, float, float>(p, pk_timing::K_GATE_LOGITS_BWD, s);
    if (rc != PK_OK) return rc;
  }
  if (d_w_gate) {
    if (!x && T > 0) return PK_ERR_ARG;
    int sp = gate_bwd_splits(T, H, E);
    if (sp > 1 && !have_part) sp = 1;
    pk_f32mm::Params p = {};
    p.B = x;
    float* const w_part = reinterpret_cast<float*>(reinterpret_cast<char*>(workspace) + gate_bwd_colsum_bytes(E));
    p.C = sp > 1 ? w_part : d_w_gate;
    p.M = E; p.N = H; p.K = T;
    p.sam = 1; p.sak = E; p.sbk = H; p.sbn = 1;
    p.splits = sp; p.accumulate = (sp == 1 && accumulate) ? 1 : 0;
    // d_logits, whose every tile is read by H / 64 workgroups, is split into its three bf16 planes
    // once when the workspace has room for them (this GEMM at 16,384 tokens: 74 -> 61 us, the split
    // included); the kernel splits the tiles it loads otherwise
    const int64_t pb = plane_bytes(T * E);
    const bool presplit = T > 0 && have_ws && pb > 0 && E % 4 == 0 && workspace_bytes >= part_bytes + pb &&
                          reinterpret_cast<uintptr_t>(d_logits) % 16 == 0;
    int rc = PK_ERR_ALIGN;
    if (presplit) {
      bf16_t* planes = reinterpret_cast<bf16_t*>(reinterpret_cast<char*>(workspace) + part_bytes);
      if (!planes_ready) {
        rc = split_planes(d_logits, planes, T * E, pk_timing::K_GATE_LOGITS_BWD, s);
        if (rc != PK_OK) return rc;
      }
      p.A = planes; p.plane_a = T * E;
      rc = x_dtype == PK_BF16 ? pk_x3mm::launch<2, 2, false, false, split3_t, bf16_t>(p, pk_timing::K_GATE_LOGITS_BWD, s)
                              : pk_x3mm::launch<2, 2, false, false, split3_t, float>(p, pk_timing::K_GATE_LOGITS_BWD, s);
    }
    if (rc == PK_ERR_ALIGN) {  // no planes, or x cannot be read four elements at a time
      p.A = d_logits;
      rc = x_dtype == PK_BF16 ? pk_x3mm::launch<2, 2, false, false, float, bf16_t>(p, pk_timing::K_GATE_LOGITS_BWD, s)
                              : pk_x3mm::launch<2, 2, false, false, float, float>(p, pk_timing::K_GATE_LOGITS_BWD, s);
    }
    if (rc != PK_OK) return rc;
    if (sp > 1) {
      const int64_t n = E * H;
      PK_LAUNCH_NOCHECK(pk_timing::K_GATE_LOGITS_BWD, s, pk_f32mm::reduce_partials_kernel,
                        dim3((unsigned)pk_ceil_div(n, 256)), dim3(256), 0, s,
                        (const float*)w_part, d_w_gate, n, sp, accumulate ? 1 : 0, (const float*)nullptr, 1);
      PK_RETURN_IF_LAUNCH_FAILED();
    }
  }
  if (d_gate_bias) {
    if (colsum_in_parts(T, E) && workspace && workspace_bytes >= gate_bwd_colsum_bytes(E) &&
        reinterpret_cast<uintptr_t>(d_logits) % 16 == 0) {
      float* part = reinterpret_cast<float*>(workspace);
      PK_LAUNCH_NOCHECK(pk_timing::K_MISC, s, colsum_partial_kernel, dim3(kColsumBlocks), dim3(256), 0, s, d_logits, T,
                        (int)E, part);
      PK_RETURN_IF_LAUNCH_FAILED();
      GateTail tail = {};
      tail.col_part = part; tail.d_bias = d_gate_bias; tail.E = (int32_t)E; tail.col_blocks = kColsumBlocks;
      tail.bias_blocks = (int32_t)pk_ceil_div(E, 256); tail.accumulate = accumulate ? 1 : 0;
      const int rc = launch_gate_tail(tail, s);
      if (rc != PK_OK) return rc;
    } else {
      PK_LAUNCH_NOCHECK(pk_timing::K_MISC, s, colsum_kernel, dim3((unsigned)E), dim3(256), 0, s, d_logits, T, (int)E,
                         d_gate_bias, accumulate ? 1 : 0);
      PK_RETURN_IF_LAUNCH_FAILED();
    }
  }
  return PK_OK;
}

// One launch for the gate weight gradient (d_logits lies split into planes behind the partial sums of the workspace),
// the bias's column sums and the region's input gradient.  PK_ERR_UNSUPPORTED: some operand does not allow the loads
// that the kernel makes; nothing has been launched.
template <typename TX>
static int router_grads(const pk_f32mm::Params& px, const pk_x3mm::GatherAdd& ga, const void* x, float* d_w_gate, float* d_gate_bias,
                        int accumulate, int64_t T, int64_t H, int64_t E, void* workspace, GateTail* tail, hipStream_t s) {
  using pk_x3mm::split3_t;
  char* const ws = reinterpret_cast<char*>(workspace);
  float* const w_part = reinterpret_cast<float*>(ws + gate_bwd_colsum_bytes(E));
  const int sp = gate_bwd_splits(T, H, E);
  RouterGrads p = {};
  p.x = px;
  p.gather = ga;
  p.w.A = ws + gate_bwd_partial_bytes(T, H, E); p.w.plane_a = T * E;
  p.w.B = x; p.w.C = sp > 1 ? w_part : d_w_gate;
  p.w.M = E; p.w.N = H; p.w.K = T;
  p.w.sam = 1; p.w.sak = E; p.w.sbk = H; p.w.sbn = 1;
  p.w.splits = sp; p.w.accumulate = sp == 1 && accumulate ? 1 : 0;
  if (!pk_x3mm::usable<2, 2, false, false, split3_t, TX>(p.w) || !pk_x3mm::gather_usable<TX>(px, ga) ||
      reinterpret_cast<uintptr_t>(px.A) % 16 != 0 || (d_w_gate && !pk_aligned16(d_w_gate)))
    return PK_ERR_UNSUPPORTED;
  p.w_nx = (int32_t)pk_ceil_div(H, 64);
  p.w_ny = (int32_t)pk_ceil_div(E, 64);
  p.gather_nx = (int32_t)pk_ceil_div(H, 32 * pk_x3mm::kGatherWN);
  const int64_t w_blocks = (int64_t)p.w_nx * p.w_ny * sp, gather = p.gather_nx * pk_ceil_div(T, 32 * pk_x3mm::kGatherWM);
  if (w_blocks + gather + PK_MAX_EXPERTS > 0x7fffffffll) return PK_ERR_UNSUPPORTED;
  p.w_blocks = (int32_t)w_blocks;
  p.d_bias = d_gate_bias;
  p.accumulate = accumulate ? 1 : 0;
  if (d_gate_bias && colsum_in_parts(T, E)) {
    p.col_part = reinterpret_cast<float*>(ws);
    p.col_blocks = kColsumBlocks;
    tail->col_part = p.col_part; tail->d_bias = d_gate_bias; tail->E = (int32_t)E; tail->col_blocks = p.col_blocks;
    tail->bias_blocks = (int32_t)pk_ceil_div(E, 256);
  } else if (d_gate_bias) {
    p.col_blocks = (int32_t)E;
  }
  if (sp > 1) {
    tail->part = w_part; tail->d_w = d_w_gate; tail->n = E * H; tail->splits = sp;
    tail->w_blocks = (int32_t)pk_ceil_div(E * H, 1024);
  }
  tail->accumulate = accumulate ? 1 : 0;
  const dim3 grid((unsigned)(w_blocks + p.col_blocks + gather));
  if (pk_x3mm::gather_streams<TX>(px, ga))
    PK_LAUNCH_NOCHECK(pk_timing::K_GATHER_REDUCE, s, (router_grads_kernel<TX, true>), grid, dim3(256), 0, s, p);
  else
    PK_LAUNCH_NOCHECK(pk_timing::K_GATHER_REDUCE, s, (router_grads_kernel<TX, false>), grid, dim3(256), 0, s, p);
  PK_RETURN_IF_LAUNCH_FAILED();
  return PK_OK;
}

extern "C" {

int pk_gate_logits_bwd(const float* d_logits, const void* x, int x_dtype, const float* w_gate,
                       float* d_x_f32, float* d_w_gate, float* d_gate_bias, int accumulate,
                       int64_t T, int64_t H, int64_t E, void* workspace, int64_t workspace_bytes,
                       pk_stream_t stream) {
  return gate_bwd(d_logits, x, x_dtype, w_gate, d_x_f32, d_w_gate, d_gate_bias, accumulate, T, H, E, workspace, workspace_bytes, false, stream);
}

#define PK_DISPATCH_EPL(E, LAUNCH)                 \
  do {                                             \
    if ((E) <= 64) { LAUNCH(1); }                  \
    else if ((E) <= 128) { LAUNCH(2); }            \
    else if ((E) <= 256) { LAUNCH(4); }            \
    else if ((E) <= 512) { LAUNCH(8); }            \
    else { LAUNCH(16); }                           \
  } while (0)

int pk_route_topk(const float* logits, int64_t T, int64_t E, int64_t K, int route_norm,
                  float route_scale, float* top_scores, int32_t* top_idx, pk_stream_t stream) {
  if (T < 0 || E <= 0 || K <= 0) return PK_ERR_ARG;
  if (E > PK_MAX_EXPERTS || K > PK_MAX_TOPK || K > E) return PK_ERR_SHAPE;
  if (T == 0) return PK_OK;
  if (!logits || !top_scores || !top_idx) return PK_ERR_ARG;
  hipStream_t s = (hipStream_t)stream;
  const dim3 grid((unsigned)pk_ceil_div(T, kRouteThreads / 64)), block(kRouteThreads);
#define PK_LAUNCH_TOPK(EPL)                                                                 \
  PK_LAUNCH_NOCHECK(pk_timing::K_ROUTE_TOPK, s, (route_topk_kernel<EPL, false>), grid, block, 0, s, GatePartials{}, const_cast<float*>(logits), \
                     (int)T, (int)E, (int)K, route_norm, route_scale, top_scores, top_idx)
  PK_DISPATCH_EPL(E, PK_LAUNCH_TOPK);
#undef PK_LAUNCH_TOPK
  PK_RETURN_IF_LAUNCH_FAILED();
  return PK_OK;
}

int pk_gate_route(const void* x, int x_dtype, const float* w_gate, const float* gate_bias, int64_t T, int64_t H, int64_t E, int64_t K,
                  int route_norm, float route_scale, float* logits, float* top_scores, int32_t* top_idx, void* workspace,
                  int64_t workspace_bytes, pk_stream_t stream) {
  if (K <= 0) return PK_ERR_ARG;
  if (E > PK_MAX_EXPERTS || K > PK_MAX_TOPK || K > E) return PK_ERR_SHAPE;
  if (T > 0 && (!top_scores || !top_idx)) return PK_ERR_ARG;
  if (H > 0 && E > 0 && pk_dtype_ok(x_dtype) && x && w_gate && logits && front_ok(FRONT_TOPK, x, x_dtype, w_gate, T, H, E)) {
    Front p = front_params(x, w_gate, gate_bias, logits, T, H, E);
    p.top_scores = top_scores; p.top_idx = top_idx;
    p.K = (int32_t)K; p.route_norm = route_norm; p.route_scale = route_scale;
    return launch_front(p, x_dtype, (hipStream_t)stream);
  }
  int splits = 1;
  const int rc = gate_gemm(x, x_dtype, w_gate, gate_bias, logits, T, H, E, workspace, workspace_bytes, (hipStream_t)stream, &splits);
  if (rc != PK_OK || T == 0) return rc;
  if (splits == 1) return pk_route_topk(logits, T, E, K, route_norm, route_scale, top_scores, top_idx, stream);
  hipStream_t s = (hipStream_t)stream;
  const dim3 grid((unsigned)pk_ceil_div(T, kRouteThreads / 64)), block(kRouteThreads);
  const GatePartials gp{reinterpret_cast<const float*>(workspace), gate_bias, splits};
#define PK_LAUNCH_TOPK(EPL)                                                                                              \
  PK_LAUNCH_NOCHECK(pk_timing::K_ROUTE_TOPK, s, (route_topk_kernel<EPL, true>), grid, block, 0, s, gp, logits, (int)T, (int)E, \
                    (int)K, route_norm, route_scale, top_scores, top_idx)
  PK_DISPATCH_EPL(E, PK_LAUNCH_TOPK);
#undef PK_LAUNCH_TOPK
  PK_RETURN_IF_LAUNCH_FAILED();
  return PK_OK;
}

static int route_topk_bwd(const float* logits, const int32_t* top_idx, const RouteBwdIo& io, int64_t T, int64_t E, int64_t K, int route_norm,
                          float route_scale, float* d_logits, hipStream_t s) {
  const dim3 grid((unsigned)pk_ceil_div(T, kRouteThreads / 64)), block(kRouteThreads);
#define PK_LAUNCH_TOPK_BWD(EPL)                                                                                          \
  PK_LAUNCH_NOCHECK(pk_timing::K_ROUTE_TOPK_BWD, s, (route_topk_bwd_kernel<EPL>), grid, block, 0, s, logits, top_idx, io, \
                    (int)T, (int)E, (int)K, route_norm, route_scale, d_logits)
  PK_DISPATCH_EPL(E, PK_LAUNCH_TOPK_BWD);
#undef PK_LAUNCH_TOPK_BWD
  PK_RETURN_IF_LAUNCH_FAILED();
  return PK_OK;
}

int pk_route_topk_bwd(const float* logits, const int32_t* top_idx, const float* d_top_scores,
                      int64_t T, int64_t E, int64_t K, int route_norm, float route_scale,
                      float* d_logits, pk_stream_t stream) {
  if (T < 0 || E <= 0 || K <= 0) return PK_ERR_ARG;
  if (E > PK_MAX_EXPERTS || K > PK_MAX_TOPK || K > E) return PK_ERR_SHAPE;
  if (T == 0) return PK_OK;
  if (!logits || !top_idx || !d_top_scores || !d_logits) return PK_ERR_ARG;
  RouteBwdIo io = {};
  io.d_top_scores = d_top_scores;
  return route_topk_bwd(logits, top_idx, io, T, E, K, route_norm, route_scale, d_logits, (hipStream_t)stream);
}

// workspace of pk_region_router_bwd: [what pk_gate_logits_bwd takes][fp32 d_x for operands that the fused
// kernel cannot read in 16-byte pieces]
static bool region_bwd_fused(int x_dtype, int64_t H, int64_t E) { return H % (x_dtype == PK_BF16 ? 8 : 4) == 0 && E % 4 == 0; }
int64_t pk_region_router_bwd_workspace_bytes(int64_t T, int64_t H, int64_t E, int x_dtype) {
  if (T < 0 || H <= 0 || E <= 0 || !pk_dtype_ok(x_dtype)) return PK_ERR_ARG;
  return align256(pk_gate_bwd_workspace_bytes(T, H, E)) + (region_bwd_fused(x_dtype, H, E) ? 0 : T * H * (int64_t)sizeof(float));
}

}  // extern "C"

// *tail: what is left for a later launch (launch_gate_tail, or extra blocks of the norm's backward)
static int region_router_bwd(const float* logits, const int32_t* top_idx, const float* d_top_scores, const float* ds_partial,
                             int64_t n_partial, const int32_t* inv_perm, int route_norm, float route_scale, const void* x, int x_dtype,
                             const float* w_gate, const void* d_rows, void* d_x, float* d_w_gate, float* d_gate_bias, int accumulate,
                             float* d_logits, int64_t T, int64_t H, int64_t E, int64_t K, void* workspace, int64_t workspace_bytes,
                             GateTail* tail, pk_stream_t stream) {
  if (T < 0 || H <= 0 || E <= 0 || K <= 0 || !pk_dtype_ok(x_dtype)) return PK_ERR_ARG;
  if (E > PK_MAX_EXPERTS || K > PK_MAX_TOPK || K > E || T > 0x7fffffffll / K) return PK_ERR_SHAPE;
  if (T > 0 && (!logits || !top_idx || !d_logits || !inv_perm || (!d_top_scores && (!ds_partial || n_partial <= 0)))) return PK_ERR_ARG;
  if (T > 0 && d_x && (!d_rows || !w_gate)) return PK_ERR_ARG;
  const int64_t gate_bytes = align256(pk_gate_bwd_workspace_bytes(T, H, E));
  if (!workspace || workspace_bytes < pk_region_router_bwd_workspace_bytes(T, H, E, x_dtype) || !pk_aligned16(workspace)) return PK_ERR_WORKSPACE;
  hipStream_t s = (hipStream_t)stream;
  int rc;
  bool planes_ready = false;
  if (T > 0) {
    RouteBwdIo io = {};
    io.d_top_scores = d_top_scores;
    io.part = ds_partial; io.n_part = (int32_t)n_partial; io.inv_perm = inv_perm; io.A = T * K;
    if (d_w_gate && plane_bytes(T * E) > 0 && E % 4 == 0) {
      io.planes = reinterpret_cast<bf16_t*>(reinterpret_cast<char*>(workspace) + gate_bwd_partial_bytes(T, H, E));
      planes_ready = true;
    }
    rc = route_topk_bwd(logits, top_idx, io, T, E, K, route_norm, route_scale, d_logits, s);
    if (rc != PK_OK) return rc;
  }
  pk_f32mm::Params p = {};
  p.A = d_logits; p.B = w_gate;
  p.M = T; p.N = H; p.K = E;
  p.sam = E; p.sak = 1; p.sbk = H; p.sbn = 1;
  p.splits = 1;
  const pk_x3mm::GatherAdd ga{d_rows, inv_perm, d_x, (int32_t)K};
  if (planes_ready && d_x && region_bwd_fused(x_dtype, H, E) && T <= pk_x3mm::kGatherSlice) {
    rc = x_dtype == PK_BF16 ? router_grads<bf16_t>(p, ga, x, d_w_gate, d_gate_bias, accumulate, T, H, E, workspace, tail, s)
                            : router_grads<float>(p, ga, x, d_w_gate, d_gate_bias, accumulate, T, H, E, workspace, tail, s);
    if (rc != PK_ERR_UNSUPPORTED) return rc;
  }
  if (d_w_gate || d_gate_bias) {
    rc = gate_bwd(d_logits, x, x_dtype, w_gate, nullptr, d_w_gate, d_gate_bias, accumulate, T, H, E, workspace, gate_bytes, planes_ready, stream);
    if (rc != PK_OK) return rc;
  }
  if (!d_x || T == 0) return PK_OK;
  if (region_bwd_fused(x_dtype, H, E)) {
    rc = x_dtype == PK_BF16 ? pk_x3mm::launch_gather<bf16_t>(p, ga, pk_timing::K_GATHER_REDUCE, s)
                            : pk_x3mm::launch_gather<float>(p, ga, pk_timing::K_GATHER_REDUCE, s);
    return rc;
  }
  float* const d_x32 = reinterpret_cast<float*>(reinterpret_cast<char*>(workspace) + gate_bytes);
  p.C = d_x32;
  rc = pk_x3mm::launch<2, 2, true, false, float, float>(p, pk_timing::K_GATE_LOGITS_BWD, s);
  if (rc != PK_OK) return rc;
  return pk_permute_bwd(d_rows, x_dtype, inv_perm, d_x32, d_x, T, H, K, stream);
}

extern "C" {

int pk_region_router_bwd(const float* logits, const int32_t* top_idx, const float* d_top_scores, const float* ds_partial,
                         int64_t n_partial, const int32_t* inv_perm, int route_norm, float route_scale, const void* x, int x_dtype,
                         const float* w_gate, const void* d_rows, void* d_x, float* d_w_gate, float* d_gate_bias, int accumulate,
                         float* d_logits, int64_t T, int64_t H, int64_t E, int64_t K, void* workspace, int64_t workspace_bytes,
                         pk_stream_t stream) {
  GateTail tail = {};
  const int rc = region_router_bwd(logits, top_idx, d_top_scores, ds_partial, n_partial, inv_perm, route_norm, route_scale, x, x_dtype, w_gate,
                                   d_rows, d_x, d_w_gate, d_gate_bias, accumulate, d_logits, T, H, E, K, workspace, workspace_bytes, &tail,
                                   stream);
  return rc != PK_OK ? rc : launch_gate_tail(tail, (hipStream_t)stream);
}

int64_t pk_region_router_norm_bwd_workspace_bytes(int64_t T, int64_t H, int64_t E, int x_dtype) {
  const int64_t router = pk_region_router_bwd_workspace_bytes(T, H, E, x_dtype);
  return router < 0 ? router : align256(router) + pk_rmsnorm_bwd_workspace_bytes(T, H);
}

int pk_region_router_norm_bwd(const float* logits, const int32_t* top_idx, const float* d_top_scores, const float* ds_partial,
                              int64_t n_partial, const int32_t* inv_perm, int route_norm, float route_scale, const void* xn, int x_dtype,
                              const float* w_gate, const void* d_rows, void* d_xn, float* d_w_gate, float* d_gate_bias, int accumulate,
                              float* d_logits, const void* x, const void* norm_weight, const float* rstd, const void* d_x_addend,
                              void* d_x, void* d_norm_weight, int64_t T, int64_t H, int64_t E, int64_t K, void* workspace,
                              int64_t workspace_bytes, pk_stream_t stream) {
  if (T < 0 || H <= 0 || E <= 0 || !pk_dtype_ok(x_dtype)) return PK_ERR_ARG;
  if (T > 0 && (!d_xn || !x || !norm_weight || !rstd || !d_x)) return PK_ERR_ARG;
  const int64_t router = align256(pk_region_router_bwd_workspace_bytes(T, H, E, x_dtype));
  if (!workspace || workspace_bytes < pk_region_router_norm_bwd_workspace_bytes(T, H, E, x_dtype)) return PK_ERR_WORKSPACE;
  GateTail tail = {};
  const int rc = region_router_bwd(logits, top_idx, d_top_scores, ds_partial, n_partial, inv_perm, route_norm, route_scale, xn, x_dtype, w_gate,
                                   d_rows, d_xn, d_w_gate, d_gate_bias, accumulate, d_logits, T, H, E, K, workspace, router, &tail, stream);
  if (rc != PK_OK) return rc;
  return pk_rmsnorm_bwd_with_tail(d_xn, x, x_dtype, norm_weight, rstd, d_x_addend, d_x, d_norm_weight, accumulate, T, H,
                                  reinterpret_cast<char*>(workspace) + router, workspace_bytes - router, tail, (hipStream_t)stream);
}

int64_t pk_sort_workspace_bytes(int64_t A, int64_t E) {
  if (A < 0 || E <= 0) return PK_ERR_ARG;
  const int64_t nchunks = pk_ceil_div(A > 0 ? A : 1, kSortChunk);
  return nchunks * E * (int64_t)sizeof(int32_t);
}

int pk_sort_by_expert(const int32_t* top_idx, int64_t A, int64_t E, int32_t* counts,
                      int32_t* starts, int32_t* perm, int32_t* inv_perm, int32_t* order,
                      void* workspace, int64_t workspace_bytes, pk_stream_t stream) {
  if (A < 0 || E <= 0) return PK_ERR_ARG;
  if (E > PK_MAX_EXPERTS || A > 0x7fffffffll) return PK_ERR_SHAPE;
  if (!starts || !workspace || (A > 0 && (!top_idx || !perm))) return PK_ERR_ARG;
  if (workspace_bytes < pk_sort_workspace_bytes(A, E)) return PK_ERR_WORKSPACE;
  hipStream_t s = (hipStream_t)stream;
  if (A <= kSmallSortSlots && E <= kSmallSortExperts) {
    PK_LAUNCH_NOCHECK(pk_timing::K_SORT_SCATTER, s, sort_small_kernel, dim3(1), dim3(64 * kSmallSortWaves), 0, s, top_idx, (int)A, (int)E,
                      SortOut{counts, starts, perm, inv_perm, order});
    PK_RETURN_IF_LAUNCH_FAILED();
    return PK_OK;
  }
  const int nchunks = (int)pk_ceil_div(A > 0 ? A : 1, kSortChunk);
  int32_t* chunk_hist = reinterpret_cast<int32_t*>(workspace);
  PK_LAUNCH_NOCHECK(pk_timing::K_SORT_HIST, s, sort_hist_kernel, dim3(nchunks), dim3(64), (size_t)E * sizeof(int32_t), s, top_idx, (int)A, (int)E,
                     chunk_hist);
  PK_RETURN_IF_LAUNCH_FAILED();
  const size_t lds = (size_t)(2 + kScatterWaves) * E * sizeof(int32_t);
  if (nchunks <= self_scan_chunks(E)) {
    PK_LAUNCH_NOCHECK(pk_timing::K_SORT_SCATTER, s, sort_scatter_kernel<false>, dim3(nchunks), dim3(kScatterThreads), lds, s, top_idx, (int)A, (int)E,
                      kSortChunk, chunk_hist, nchunks, counts, starts, perm, inv_perm, order);
    PK_RETURN_IF_LAUNCH_FAILED();
    return PK_OK;
  }
  PK_LAUNCH_NOCHECK(pk_timing::K_SORT_SCAN, s, sort_scan_kernel, dim3(1), dim3(1024), 0, s, chunk_hist, nchunks, (int)E, counts, starts, order);
  PK_RETURN_IF_LAUNCH_FAILED();
  PK_LAUNCH_NOCHECK(pk_timing::K_SORT_SCATTER, s, sort_scatter_kernel<true>, dim3(nchunks), dim3(kScatterThreads), lds, s, top_idx, (int)A, (int)E,
                    kSortChunk, chunk_hist, nchunks, counts, starts, perm, inv_perm, order);
  PK_RETURN_IF_LAUNCH_FAILED();
  return PK_OK;
}

int64_t pk_gate_route_sort_workspace_bytes(int64_t T, int64_t H, int64_t E, int64_t K) {
  if (T < 0 || H <= 0 || E <= 0 || K <= 0) return PK_ERR_ARG;
  const int64_t gate = pk_gate_workspace_bytes(T, H, E), sort = pk_sort_workspace_bytes(T * K, E);
  const int64_t front = pk_ceil_div(T, kFrontTokens) * E * (int64_t)sizeof(int32_t);      // histograms of gate_front_kernel
  const int64_t most = gate > sort ? gate : sort;
  if (T > kFrontMaxTokens || E > kFrontExperts) return most;
  // (the top-k reads the gate's partial results and writes the histograms behind them)
  const int64_t both = front_sorts(T, E) ? align256(gate) + front : 0;
  return std::max(std::max(most, front), both);
}

}  // extern "C"

// norm_w: the norm whose output (xn, written) the gate reads; nullptr: it reads x
static int norm_gate_route_sort(const void* x, int x_dtype, const void* norm_w, float eps, void* xn, float* rstd, const float* w_gate,
                                const float* gate_bias, int64_t T, int64_t H, int64_t E, int64_t K, int route_norm, float route_scale,
                                float* logits, float* top_scores, int32_t* top_idx, int32_t* counts, int32_t* starts, int32_t* perm,
                                int32_t* inv_perm, int32_t* order, void* workspace, int64_t workspace_bytes, pk_stream_t stream) {
  if (T < 0 || K <= 0 || E <= 0) return PK_ERR_ARG;
  if (E > PK_MAX_EXPERTS || K > PK_MAX_TOPK || K > E || T > 0x7fffffffll / K) return PK_ERR_SHAPE;
  if (!starts || !workspace || (T > 0 && (!top_scores || !top_idx || !perm))) return PK_ERR_ARG;
  if (workspace_bytes < pk_gate_route_sort_workspace_bytes(T, H, E, K)) return PK_ERR_WORKSPACE;
  hipStream_t s = (hipStream_t)stream;
  if (H > 0 && pk_dtype_ok(x_dtype) && x && w_gate && logits &&
      front_ok(norm_w ? FRONT_NORM : FRONT_SORT, x, x_dtype, w_gate, T, H, E) &&
      (!norm_w || (xn && pk_aligned16(norm_w) && pk_aligned16(xn)))) {
    Front p = front_params(x, w_gate, gate_bias, logits, T, H, E);
    p.norm_w = norm_w; p.eps = eps; p.xn = xn; p.rstd = rstd;
    p.top_scores = top_scores; p.top_idx = top_idx;
    p.K = (int32_t)K; p.route_norm = route_norm; p.route_scale = route_scale;
    p.chunk_hist = front_sorts(T, E) ? reinterpret_cast<int32_t*>(workspace) : nullptr;
    const int rc = launch_front(p, x_dtype, s);
    if (rc != PK_OK) return rc;
    if (!p.chunk_hist) return pk_sort_by_expert(top_idx, T * K, E, counts, starts, perm, inv_perm, order, workspace, workspace_bytes, stream);
    const int nchunks = (int)pk_ceil_div(T, kFrontTokens);
    PK_LAUNCH_NOCHECK(pk_timing::K_SORT_SCATTER, s, sort_scatter_kernel<false>, dim3(nchunks), dim3(kScatterThreads),
                      (size_t)(2 + kScatterWaves) * E * sizeof(int32_t), s, top_idx, (int)(T * K), (int)E, (int)(kFrontTokens * K), p.chunk_hist,
                      nchunks, counts, starts, perm, inv_perm, order);
    PK_RETURN_IF_LAUNCH_FAILED();
    return PK_OK;
  }
  bool have_logits = false;
  if (norm_w) {
    have_logits = T > 0 && T <= kGateSmallMax && H <= kNormGateMaxWidth && H % (16 / (int64_t)pk_dtype_size(x_dtype)) == 0 && w_gate && logits &&
                  pk_aligned16(x) && pk_aligned16(norm_w) && pk_aligned16(xn) && pk_aligned16(w_gate);
    const int rc = have_logits ? pk_norm_gate_small(x, x_dtype, norm_w, eps, xn, rstd, w_gate, gate_bias, logits, T, H, E, s)
                               : pk_rmsnorm_fwd(x, x_dtype, norm_w, eps, xn, rstd, T, H, stream);
    if (rc != PK_OK) return rc;
    x = xn;
  }
  // 16 tokens a chunk, as behind gate_front_kernel; up to 1,024 slots sort_small_kernel is quicker
  if (T * K > kRouteSortSlots && T > kRouteSortTokens && T <= kFrontMaxTokens && E <= kTopkHistExperts && front_sorts(T, E)) {
    int splits = 1;
    if (!have_logits) {
      const int rc = gate_gemm(x, x_dtype, w_gate, gate_bias, logits, T, H, E, workspace, workspace_bytes, s, &splits);
      if (rc != PK_OK) return rc;
    }
    if (!logits) return PK_ERR_ARG;
    const GatePartials gp{splits > 1 ? reinterpret_cast<const float*>(workspace) : nullptr, gate_bias, splits};
    int32_t* const chunk_hist = reinterpret_cast<int32_t*>(reinterpret_cast<char*>(workspace) + align256(gate_fwd_partial_bytes(T, H, E)));
    const int nchunks = (int)pk_ceil_div(T, kTopkHistTokens);
#define PK_TOPK_HIST(EPL, PARTIALS)                                                                                                                  \
  PK_LAUNCH_NOCHECK(pk_timing::K_ROUTE_TOPK, s, (route_topk_hist_kernel<EPL, PARTIALS>), dim3(nchunks), dim3(64 * kTopkHistTokens), 0, s, gp, logits, \
                    (int)T, (int)E, (int)K, route_norm, route_scale, top_scores, top_idx, chunk_hist)
    if (E <= 64) { if (splits > 1) PK_TOPK_HIST(1, true); else PK_TOPK_HIST(1, false); }
    else { if (splits > 1) PK_TOPK_HIST(2, true); else PK_TOPK_HIST(2, false); }
#undef PK_TOPK_HIST
    PK_RETURN_IF_LAUNCH_FAILED();
    PK_LAUNCH_NOCHECK(pk_timing::K_SORT_SCATTER, s, sort_scatter_kernel<false>, dim3(nchunks), dim3(kScatterThreads),
                      (size_t)(2 + kScatterWaves) * E * sizeof(int32_t), s, top_idx, (int)(T * K), (int)E, (int)(kTopkHistTokens * K), chunk_hist,
                      nchunks, counts, starts, perm, inv_perm, order);
    PK_RETURN_IF_LAUNCH_FAILED();
    return PK_OK;
  }
  if (T == 0 || T > kRouteSortTokens || T * K > kRouteSortSlots || E > kSmallSortExperts) {
    const int rc = have_logits ? pk_route_topk(logits, T, E, K, route_norm, route_scale, top_scores, top_idx, stream)
                               : pk_gate_route(x, x_dtype, w_gate, gate_bias, T, H, E, K, route_norm, route_scale, logits, top_scores, top_idx,
                                               workspace, workspace_bytes, stream);
    if (rc != PK_OK) return rc;
    return pk_sort_by_expert(top_idx, T * K, E, counts, starts, perm, inv_perm, order, workspace, workspace_bytes, stream);
  }
  int splits = 1;
  if (!have_logits) {
    const int rc = gate_gemm(x, x_dtype, w_gate, gate_bias, logits, T, H, E, workspace, workspace_bytes, s, &splits);
    if (rc != PK_OK) return rc;
  }
  const GatePartials gp{splits > 1 ? reinterpret_cast<const float*>(workspace) : nullptr, gate_bias, splits};
  const SortOut out{counts, starts, perm, inv_perm, order};
  const dim3 grid(1), block(64 * kSmallSortWaves);
#define PK_LAUNCH_ROUTE_SORT(EPL)                                                                                                   \
  do {                                                                                                                              \
    if (splits > 1)                                                                                                                 \
      PK_LAUNCH_NOCHECK(pk_timing::K_ROUTE_TOPK, s, (route_sort_small_kernel<EPL, true>), grid, block, 0, s, gp, logits, (int)T, (int)E, (int)K,  \
                        route_norm, route_scale, top_scores, top_idx, out);                                                         \
    else                                                                                                                            \
      PK_LAUNCH_NOCHECK(pk_timing::K_ROUTE_TOPK, s, (route_sort_small_kernel<EPL, false>), grid, block, 0, s, gp, logits, (int)T, (int)E, (int)K, \
                        route_norm, route_scale, top_scores, top_idx, out);                                                         \
  } while (0)
  PK_DISPATCH_EPL(E, PK_LAUNCH_ROUTE_SORT);
#undef PK_LAUNCH_ROUTE_SORT
  PK_RETURN_IF_LAUNCH_FAILED();
  return PK_OK;
}

extern "C" {

int pk_gate_route_sort(const void* x, int x_dtype, const float* w_gate, const float* gate_bias, int64_t T, int64_t H, int64_t E,
                       int64_t K, int route_norm, float route_scale, float* logits, float* top_scores, int32_t* top_idx,
                       int32_t* counts, int32_t* starts, int32_t* perm, int32_t* inv_perm, int32_t* order, void* workspace,
                       int64_t workspace_bytes, pk_stream_t stream) {
  return norm_gate_route_sort(x, x_dtype, nullptr, 0.f, nullptr, nullptr, w_gate, gate_bias, T, H, E, K, route_norm, route_scale, logits,
                              top_scores, top_idx, counts, starts, perm, inv_perm, order, workspace, workspace_bytes, stream);
}

int pk_norm_gate_route_sort(const void* x, int x_dtype, const void* norm_weight, float eps, void* xn, float* rstd, const float* w_gate,
                            const float* gate_bias, int64_t T, int64_t H, int64_t E, int64_t K, int route_norm, float route_scale,
                            float* logits, float* top_scores, int32_t* top_idx, int32_t* counts, int32_t* starts, int32_t* perm,
                            int32_t* inv_perm, int32_t* order, void* workspace, int64_t workspace_bytes, pk_stream_t stream) {
  if (T < 0 || H <= 0 || !pk_dtype_ok(x_dtype) || !(eps >= 0.f) || (T > 0 && (!x || !norm_weight || !xn))) return PK_ERR_ARG;
  return norm_gate_route_sort(x, x_dtype, norm_weight, eps, xn, rstd, w_gate, gate_bias, T, H, E, K, route_norm, route_scale, logits,
                              top_scores, top_idx, counts, starts, perm, inv_perm, order, workspace, workspace_bytes, stream);
}

int pk_sort_by_expert_static(const int32_t* top_idx, int64_t A, int64_t E, int32_t* counts,
                             int32_t* starts, int32_t* perm, int32_t* inv_perm, int32_t* order,
                             pk_stream_t stream) {
  if (A < 0 || E <= 0) return PK_ERR_ARG;
  if (E > PK_MAX_EXPERTS || A > 0x7fffffffll) return PK_ERR_SHAPE;
  // the per-chunk histograms must fit the fixed scratch array
  const int64_t need = pk_sort_workspace_bytes(A, E);
  if (need > (int64_t)sizeof(int32_t) * PK_SORT_STATIC_WORDS) return PK_ERR_WORKSPACE;
  int32_t* ws = sort_scratch_for_current_device();
  if (!ws) return PK_ERR_UNSUPPORTED;
  return pk_sort_by_expert(top_idx, A, E, counts, starts, perm, inv_perm, order, ws, need, stream);
}

int pk_counts_to_starts(const void* counts, int counts_is_i64, int64_t E, int32_t* starts,
                        pk_stream_t stream) {
  if (E <= 0 || !counts || !starts) return PK_ERR_ARG;
  if (E > PK_MAX_EXPERTS) return PK_ERR_SHAPE;
  PK_LAUNCH_NOCHECK(pk_timing::K_COUNTS_TO_STARTS, (hipStream_t)stream, counts_to_starts_kernel, dim3(1), dim3(1024), 0, (hipStream_t)stream, counts,
                     counts_is_i64, (int)E, starts);
  PK_RETURN_IF_LAUNCH_FAILED();
  return PK_OK;
}

}  // extern "C"
