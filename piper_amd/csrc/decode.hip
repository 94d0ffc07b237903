// The region without a backward for a decode step: up to 16 routed rows (one token of top-8, sixteen of top-1), bf16.
// Every launch of the general path is then a few microseconds of latency around little work, and the sort only serves to
// group rows that one wave can hold, so three launches do what six to eight did:
//
//   1  norm and gate logits    (norm_gate_small_kernel)
//   2  top-k, gate/up, SiLU    every workgroup chooses the experts for itself, about a microsecond where a launch of its own
//                              takes three to six, and workgroup 0 writes them down
//   3  down, combine           a workgroup has eight columns and the rows of all experts, so the weighted sum over a
//                              token's experts needs nobody else
//
// Bound by the weights of the chosen experts; what is left is latency, so a wave asks for its whole share of them at
// once.  2048 x 768, 128 experts, top-8, us, general path -> here (the weights alone take 14.5 us a token at 5.2 TB/s):
//   one token   2.7 + 2.8 + 5.8 + 13.2 + 7.5 + 3.0 = 35.0 -> 4.3 + 13.8 + 8.8 = 26.9
//   two         3.1 + 4.7 + 6.2 + 21.1 + 12.2 + 4.1 = 51.3 -> 5.1 + 24.1 + 16.9 = 46.1
#include "pk_common.h"
#include "topk.h"
#include <initializer_list>

// logits = [norm](x) . w_gate^T + gate_bias for a few tokens (route.hip)
int pk_norm_gate_small(const void* x, int dtype, const void* norm_w, float eps, void* xn, float* rstd, const float* w_gate, const float* gate_bias,
                       float* logits, int64_t T, int64_t H, int64_t E, hipStream_t s);

namespace {

constexpr int kDecodeRows = 16;

// Sixteen rows of `w` (r16: the lane's) against the sixteen rows of the other operand, over the reduction elements
// [k0, k1) in steps of 64: a wave's whole share, CHUNK steps of it in flight at once.  Past k1: zeros.
template <int CHUNK>
__device__ __forceinline__ floatx4_t rows_times_rows(const bf16_t* __restrict__ w, const bf16_t* __restrict__ a, int k0, int k1, int g) {
  floatx4_t acc = {0.f, 0.f, 0.f, 0.f};
  for (int c = k0; c < k1; c += 64 * CHUNK) {
    u32x4_t wv[CHUNK][2], av[CHUNK][2];
#pragma unroll
    for (int s = 0; s < CHUNK; ++s)
#pragma unroll
      for (int h = 0; h < 2; ++h) wv[s][h] = *reinterpret_cast<const u32x4_t*>(w + min(c + 64 * s + 32 * h + 8 * g, k1 - 8));
#pragma unroll
    for (int s = 0; s < CHUNK; ++s)
#pragma unroll
      for (int h = 0; h < 2; ++h) av[s][h] = *reinterpret_cast<const u32x4_t*>(a + min(c + 64 * s + 32 * h + 8 * g, k1 - 8));
    __builtin_amdgcn_sched_barrier(0);      // (all of them in front of the first use)
    const u32x4_t zero = {0u, 0u, 0u, 0u};
#pragma unroll
    for (int s = 0; s < CHUNK; ++s)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const bool in = c + 64 * s + 32 * h + 8 * g < k1;
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, in ? av[s][h] : zero),
                                                      __builtin_bit_cast(bf16x8_t, in ? wv[s][h] : zero), acc, 0, 0, 0);
      }
  }
  return acc;      // [v]: row 4 (l / 16) + v of `a`, row l % 16 of `w`
}

// ---- 2: h[slot] = silu(x . w1[e]^T) * (x . w3[e]^T) for the slots (t, k) of one expert and eight columns
struct DecodeRoute {
  const float* logits;
  float* scores;          // written by workgroup 0
  int32_t* idx;
  int32_t T, E, K, route_norm;
  float route_scale;
};
template <int EPL>
__global__ __launch_bounds__(256) void decode_gate_up_kernel(const DecodeRoute rt, const bf16_t* __restrict__ x, const bf16_t* __restrict__ w1,
                                                             const bf16_t* __restrict__ w3, bf16_t* __restrict__ h, int H, int I) {
  __shared__ int32_t chosen[kDecodeRows];
  __shared__ float red[4][256];
  const int tid = threadIdx.x, lane = tid & 63, r = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int slots = rt.T * rt.K, n_tiles = I / 8;
  for (int t = wave; t < rt.T; t += 4) {
    float val[1][EPL], score[1];
    int expert[1];
#pragma unroll
    for (int j = 0; j < EPL; ++j) val[0][j] = lane + 64 * j < rt.E ? rt.logits[(int64_t)t * rt.E + lane + 64 * j] : 0.f;
    topk_of<EPL, 1>(val, lane, rt.E, rt.K, rt.route_norm, rt.route_scale, score, expert);
    if (lane < rt.K) {
      chosen[t * rt.K + lane] = expert[0];
      if (blockIdx.x == 0) {
        rt.scores[t * rt.K + lane] = score[0];
        rt.idx[t * rt.K + lane] = expert[0];
      }
    }
  }
  __syncthreads();
  // the workgroup's slot stands for its expert if it is the first of its slots
  const int slot = blockIdx.x / n_tiles, n0 = (blockIdx.x - slot * n_tiles) * 8;
  const int mine = lane < slots ? chosen[lane] : -1;
  const int e = __builtin_amdgcn_readlane(mine, slot);
  const unsigned long long same = __ballot(mine == e);
  if (__ffsll((long long)same) - 1 != slot) return;
  const int steps = (H + 63) / 64, first = wave * steps / 4, last = (wave + 1) * steps / 4;      // a contiguous share of the reduction
  const bf16_t* const w = (r < 8 ? w1 : w3) + ((int64_t)e * I + n0 + (r & 7)) * H;
  const floatx4_t acc = rows_times_rows<8>(w, x + (int64_t)(min(r, slots - 1) / rt.K) * H, 64 * first, min(64 * last, H), g);
#pragma unroll
  for (int v = 0; v < 4; ++v) red[wave][(4 * g + v) * 16 + r] = acc[v];
  __syncthreads();
  const int row = tid >> 3, c = tid & 7;
  if (row < slots && ((same >> row) & 1)) {
    float gs = 0.f, us = 0.f;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      gs += red[q][row * 16 + c];
      us += red[q][row * 16 + 8 + c];
    }
    const float gf = (float)(bf16_t)gs, uf = (float)(bf16_t)us;      // g and u are tensors of bf16
    h[(int64_t)row * I + n0 + c] = (bf16_t)((gf / (1.f + __expf(-gf))) * uf);
  }
}

// ---- 3: out[t] = sum_k score[t][k] * bf16(h[t][k] . w2[e]^T) (+ residual[t]), eight columns a workgroup.  A wave takes two
// experts at a time: one in the first eight columns of its MFMA tile, one in the others.
__global__ __launch_bounds__(256) void decode_down_kernel(const float* __restrict__ scores, const int32_t* __restrict__ idx, const bf16_t* __restrict__ h,
                                                          const bf16_t* __restrict__ w2, const bf16_t* __restrict__ residual,
                                                          bf16_t* __restrict__ out, int T, int K, int H, int I) {
  __shared__ float y[kDecodeRows][8];
  const int tid = threadIdx.x, lane = tid & 63, r = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int slots = T * K, n0 = blockIdx.x * 8;
  const int mine = lane < slots ? idx[lane] : -1;
  // slots that are the first of their expert, in order
  unsigned long long firsts = 0;
  for (int s = 0; s < slots; ++s) {
    const unsigned long long same = __ballot(mine == __builtin_amdgcn_readlane(mine, s));
    if (__ffsll((long long)same) - 1 == s) firsts |= 1ull << s;
  }
  const int experts = __popcll(firsts);
  for (int p = wave; 2 * p < experts; p += 4) {
    unsigned long long rest = firsts;
    for (int i = 0; i < 2 * p; ++i) rest &= rest - 1;
    const int ea = __builtin_amdgcn_readlane(mine, __ffsll((long long)rest) - 1);
    rest &= rest - 1;
    const int eb = rest ? __builtin_amdgcn_readlane(mine, __ffsll((long long)rest) - 1) : ea;
    const int e = r < 8 ? ea : eb;
    const floatx4_t acc = rows_times_rows<12>(w2 + ((int64_t)e * H + n0 + (r & 7)) * I, h + (int64_t)min(r, slots - 1) * I, 0, I, g);
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int slot = 4 * g + v;
      if (slot < slots && __shfl(mine, slot) == e && (r < 8 || eb != ea)) y[slot][r & 7] = (float)(bf16_t)acc[v];
    }
  }
  __syncthreads();
  const int t = tid >> 3, c = tid & 7;
  if (t >= T) return;
  float acc = 0.f;
  for (int k = 0; k < K; ++k) acc = fmaf(scores[t * K + k], y[t * K + k][c], acc);
  const int64_t o = (int64_t)t * H + n0 + c;
  if (residual) acc = (float)(bf16_t)acc + (float)residual[o];
  out[o] = (bf16_t)acc;
}

struct DecodeWorkspace {
  int64_t xn, logits, scores, idx, h, bytes;
  DecodeWorkspace(int64_t T, int64_t H, int64_t E, int64_t I, int64_t K) {
    int64_t at = 0;
    const auto add = [&](int64_t n) { const int64_t p = at; at += (n + 255) / 256 * 256; return p; };
    xn = add(T * H * 2); logits = add(T * E * 4); scores = add(T * K * 4); idx = add(T * K * 4); h = add(T * K * I * 2);
    bytes = at;
  }
};

}  // namespace

extern "C" {

int64_t pk_region_decode_workspace_bytes(int64_t T, int64_t H, int64_t E, int64_t I, int64_t K, int dtype) {
  if (T < 0 || H <= 0 || E <= 0 || I <= 0 || K <= 0) return PK_ERR_ARG;
  if (dtype != PK_BF16 || T == 0 || T * K > kDecodeRows || K > E || E > PK_MAX_EXPERTS || H % 8 != 0 || I % 8 != 0 || H > 8192 || I > (1 << 20)) return 0;
  return DecodeWorkspace(T, H, E, I, K).bytes;
}

// Against the general path its time grows with the tokens (every workgroup chooses the experts of all of them), with rounds of
// experts (down: two for each of four waves) and with I (down: chunks of 768), and falls with H (down: a workgroup per eight
// columns).  us, general -> here, tokens x experts a token:
//   128 experts 2048 x  768   1x8 53 -> 44   2x8 81 -> 74   8x2 76 -> 73   10x1 59 -> 57   14x1 73 -> 76
//    24         1000 x  360   1x8 31 -> 25   2x8 37 -> 33   8x2 32 -> 29   16x1 35 -> 33
//    64          512 x  512   1x8 29 -> 25   9x1 28 -> 29   2x8 32 -> 39   16x1 31 -> 45
//   128         1024 x  384   1x8 32 -> 27   5x2 33 -> 31   2x6 35 -> 35    2x8 37 -> 39   16x1 37 -> 43
//    64         1536 x  768   1x8 46 -> 39   9x1 46 -> 41   2x8 66 -> 63   14x1 59 -> 58   16x1 61 -> 67
//    16         2048 x 1024   1x8 60 -> 55   5x2 67 -> 64   4x4 70 -> 67    8x2 73 -> 77
//    32         1024 x 1024   1x6 37 -> 35   1x8 41 -> 42   2x6 50 -> 56   16x1 46 -> 63
//     8          512 x  256   2x8 26 -> 23   8x2 26 -> 26  16x1 26 -> 29
//     8         1024 x 4096   1x2 48 -> 40   1x4 61 -> 63   2x8 97 -> 115
//    16         4096 x 4096   1x4 145 -> 138  4x2 202 -> 201  2x8 252 -> 269  16x1 240 -> 300
//    16         8192 x 1024   1x6 137 -> 133  2x4 144 -> 152  2x8 187 -> 215
// Widths that are no multiple of 128 leave the general path smaller steps, and it loses everywhere.  Popular experts (counts ~ 1 /
// sqrt(rank)) leave fewer to read and move the line up: 16 experts 640 x 128, 7x2 26 -> 23; 64 experts 512 x 256, 12x1
// 26 -> 23 (even 27 -> 30), 16x1 26 -> 24 (27 -> 35); 128 experts 1280 x 384, 12x1 32 -> 29 (1024 x 384, even 34 -> 37).
int pk_region_decode_pays(int64_t T, int64_t H, int64_t E, int64_t I, int64_t K) {
  if (T <= 0 || K <= 0 || T > kDecodeRows || K > kDecodeRows || T * K > kDecodeRows) return 0;
  const int64_t n = T * K;
  const bool deep = I > 768 && H < 2 * I;
  if (I > H) return n <= 2 || (n <= 8 && I <= 768);
  if (H > 4096) return n <= 6;
  if (n <= 8) return !deep || n <= 6 || (H > I && T <= 4);
  if (H % 128 != 0 || I % 128 != 0) return I <= 1024;
  if (deep) return 0;
  if (E <= 8) return H <= 2048 && T <= (E <= 4 && I <= 768 ? 16 : 12);
  if (H >= 1536) return T <= (I > 768 ? 5 : 12);
  return n <= (I <= 128 ? 16 : I <= 256 ? 14 : 12);
}

int pk_region_decode(const void* x, int dtype, const void* norm_weight, float eps, const float* w_gate, const float* gate_bias, const void* w1,
                     const void* w2, const void* w3, int route_norm, float route_scale, const void* residual, void* out, int64_t T, int64_t H,
                     int64_t E, int64_t I, int64_t K, void* workspace, int64_t workspace_bytes, pk_stream_t stream) {
  const int64_t need = pk_region_decode_workspace_bytes(T, H, E, I, K, dtype);
  if (need < 0) return PK_ERR_ARG;
  if (need == 0) return PK_ERR_UNSUPPORTED;
  if (!x || !w_gate || !w1 || !w2 || !w3 || !out || (norm_weight && !(eps >= 0.f))) return PK_ERR_ARG;
  if (!workspace || workspace_bytes < need) return PK_ERR_WORKSPACE;
  for (const void* p : {x, norm_weight, (const void*)w_gate, w1, w2, w3, residual, (const void*)out, (const void*)workspace})
    if (!pk_aligned16(p)) return PK_ERR_ALIGN;
  const DecodeWorkspace ws(T, H, E, I, K);
  char* const base = reinterpret_cast<char*>(workspace);
  hipStream_t s = (hipStream_t)stream;
  bf16_t* const xn = reinterpret_cast<bf16_t*>(base + ws.xn);
  float *const logits = reinterpret_cast<float*>(base + ws.logits), *const scores = reinterpret_cast<float*>(base + ws.scores);
  int32_t* const idx = reinterpret_cast<int32_t*>(base + ws.idx);
  bf16_t* const h = reinterpret_cast<bf16_t*>(base + ws.h);
  const dim3 block(256);
  const int rc = pk_norm_gate_small(x, dtype, norm_weight, eps, xn, nullptr, w_gate, gate_bias, logits, T, H, E, s);
  if (rc != PK_OK) return rc;
  const DecodeRoute rt{logits, scores, idx, (int32_t)T, (int32_t)E, (int32_t)K, route_norm, route_scale};
  const dim3 up_grid((unsigned)(T * K * (I / 8)));
#define PK_DECODE_UP(EPL)                                                                                                               \
  PK_LAUNCH_NOCHECK(pk_timing::K_SWIGLU_GATE_UP, s, decode_gate_up_kernel<EPL>, up_grid, block, 0, s, rt, norm_weight ? xn : (const bf16_t*)x, \
                    (const bf16_t*)w1, (const bf16_t*)w3, h, (int)H, (int)I)
  if (E <= 64) PK_DECODE_UP(1);
  else if (E <= 128) PK_DECODE_UP(2);
  else if (E <= 256) PK_DECODE_UP(4);
  else PK_DECODE_UP(16);
#undef PK_DECODE_UP
  PK_RETURN_IF_LAUNCH_FAILED();
  PK_LAUNCH_NOCHECK(pk_timing::K_SWIGLU_DOWN, s, decode_down_kernel, dim3((unsigned)(H / 8)), block, 0, s, (const float*)scores, (const int32_t*)idx,
                    (const bf16_t*)h, (const bf16_t*)w2, (const bf16_t*)residual, (bf16_t*)out, (int)T, (int)K, (int)H, (int)I);
  PK_RETURN_IF_LAUNCH_FAILED();
  return PK_OK;
}

}  // extern "C"
