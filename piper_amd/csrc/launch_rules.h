// Which kernel a grouped product takes, and how its work is cut up, by the sizes alone (the 256-wide bf16 kernels, and what the fp32
// tile products load).  Plain functions of numbers, without a GPU in them, so that a test can ask them too.  cus: CUs, which are
// also the workgroups of the persistent grid.
#pragma once
#include <cstdint>

namespace pk_rules {

constexpr int NXCD = 8;
constexpr int64_t ceil_div(int64_t a, int64_t b) { return (a + b - 1) / b; }

// ---- rows of the persistent kernels' units (256 output columns, for gate/up 128 of each)
enum Product { GATE_UP, DOWN, DX, DX_TRANSPOSED, DH, DH_SCALED };

// 256 rows from this many rows an expert on, unless they leave a workgroup fewer than three units.  (Not gate/up, which goes from 128 to
// 160 rows, and not the scaled SwiGLU backward, which stays on 128: its time goes into the epilogue, loads of g and u, the arithmetic,
// six stores per value, which 256-row units do not shorten, and with 128 accumulator registers that epilogue spills, measured 14 %
// slower at 16,384 tokens even with the packed outputs staged 32 columns at a time.)
constexpr int64_t SHORT_ROWS = 512, LEAST_UNITS = 3;
// d_x already with fewer rows and units: of the three products it reads most of its weights through the transposing LDS
// read, which the taller unit halves (128 -> 256 rows, us, even / skewed counts: 128 experts 2048 x 768, 320 rows
// 333 -> 317 / 333 -> 312, 448 rows 424 -> 376 / 422 -> 394; 272 rows 303 -> 311 / 297 -> 279; 1024 x 512, 320 rows 139 -> 142 /
// 142 -> 142, 384 rows 165 -> 151 / 152 -> 155; 64 experts 2048 x 1024, 352 rows 245 -> 222 / 242 -> 237; 32 experts 2048 x 768,
// 384 rows, 2.25 units per CU 117 -> 103).  Down gains as much with even counts between 128 and 200 rows, and loses more
// with skewed ones (128 experts 2048 x 768, 144 rows: 143 -> 133 / 133 -> 140).
constexpr int64_t DX_SHORT_ROWS = 320, DX_LEAST_UNITS = 2;
// 160 rows, otherwise like the 128-row ones: what fits the LDS (3 x 52 KB).  A unit costs about a fifth more time than one of
// 128 rows and there are fewer of them, above all fewer with a handful of rows (256 rows an expert: two units where half of
// the experts had three).  tall_units_pay says when; 128 (or where named 256) rows -> 160, us, even counts / ~ 1 / sqrt(rank):
// 128 experts 2048 x 768: 256 rows: gate/up 285 -> 260 / 281 -> 273, down 174 -> 164 / 177 -> 170, d_x 280 -> 259 / 280 -> 270; 480
// rows: gate/up 449 -> 418 / 449 -> 426, down 270 -> 253 / 274 -> 247; 224 rows: 266 -> 271 / 260 -> 257, 162 -> 165 / 165 -> 161,
// 253 -> 262 / 264 -> 255; 111 rows 199 -> 197 / 194 -> 198.  64 experts 1536 x 768, 450 rows: 198 -> 178 / 200 -> 179, 115 -> 105 /
// 114 -> 110.  Few rounds of units, where the last one counts: 16 experts 2048 x 1024, 512 rows 114 -> 97 / 109 -> 94, 70 -> 63 / 66 -> 60,
// 108 -> 95 / 104 -> 98; 64 experts 2048 x 768, 256 rows (3.75 rounds -> 3.15) 157 -> 168 / 159 -> 167; 8 experts 1024 x 512, 4,000 rows
// (3.97 -> 3.19) 94 -> 103 / 95 -> 100; 128 experts 1024 x 512, 300 rows (5.7 -> 4.75) 134 -> 140 / 136 -> 144.
// Against 256 rows: gate/up at any size (128 experts 2048 x 768: 512 rows 463 -> 446 / 468 -> 434, 1,024 rows 833 -> 809 / 836 -> 810;
// 16 experts 2048 x 1024, 2,048 rows 302 -> 279 / 310 -> 281), down with a long reduction (64 experts 2048 x 1024, 512 rows 191 -> 179 /
// 191 -> 177; but 2048 x 768, 512 rows 267 -> 277 / 278 -> 263, 1,024 rows 490 -> 494 / 493 -> 493), d_x not (512 rows 423 -> 440 /
// 429 -> 430, 1,024 rows 748 -> 804 / 763 -> 805).
constexpr int64_t TALL_ROWS = 248, TALL_DOWN_K = 1024;
// Whether units of 160 rows are ahead of 128: with more than six rounds of the latter wherever there are fewer of the former, below
// that by the number of rounds, a taller one at six fifths of the time (where that is a draw, from 352 rows an expert on).
constexpr bool tall_units_pay(int64_t A, int64_t E, int64_t cols, int64_t cus) {
  if (A < TALL_ROWS * E) return false;
  const int64_t u128 = (A / 128 + E / 2) * cols, u160 = (A / 160 + E / 2) * cols;
  if (u128 >= 6 * cus) return true;
  const int64_t c128 = 5 * ceil_div(u128, cus), c160 = 6 * ceil_div(u160, cus);
  return c160 < c128 || (c160 == c128 && A >= 352 * E);
}
// cols: columns of units; K: reduction (of one of d_x's two segments)
constexpr int unit_rows(Product what, int64_t A, int64_t E, int64_t cols, int64_t K, int64_t cus) {
  const int64_t units = (A / 256 + E / 2) * cols;
  const bool low = units < (what == DX ? DX_LEAST_UNITS : LEAST_UNITS) * cus || A < (what == DX ? DX_SHORT_ROWS : SHORT_ROWS) * E;
  const bool tall = what == GATE_UP || ((what == DOWN || what == DX) && low) || (what == DOWN && K >= TALL_DOWN_K);
  if (tall && tall_units_pay(A, E, cols, cus)) return 160;
  return low || what == GATE_UP || what == DH_SCALED ? 128 : 256;
}

// ---- weight gradients from row-major operands
enum WgradKernel { TILES, RUNS, RING, BIG };
// Weight gradients from row-major operands (with the transposed copies wgrad_pp_kernel, whose tile is fixed), 256 x 256 tiles by
// rows an expert: few, wgrad_runs_kernel; from WG_BIG_ROWS on 64-deep k-tiles in a 2-stage ring; between them 32-deep ones in a
// 4-stage ring with the loads spread between the MFMAs.  us, runs -> 4-stage ring, gathered rows, even counts / ~ 1 / sqrt(rank): 128 experts
// 2048 x 768: 192 rows 449 -> 476 / 516 -> 503, 256 rows 571 -> 556 / 658 -> 599, 400 rows 783 -> 734 / 876 -> 796; 64 experts 1536 x 768, 400
// rows 299 -> 287 / 327 -> 312; 24 experts 1024 x 768, 400 rows, not gathered, 88 -> 81 / 82 -> 72.  With fewer than two tiles for every CU the
// longest expert's k-loop counts sooner (64 experts 512 x 256, 192 rows, not gathered, 33.2 -> 34.0 / 48.0 -> 43.8).  Accumulating, the runs'
// way to the old values is ahead at any size (128 experts 2048 x 768, 400 rows 907 against 1,080).
constexpr int64_t WG_RUNS_ROWS = 224, WG_RUNS_ROWS_ONE = 160, WG_BIG_ROWS = 512;
// 256 x 256 tiles where they give at least half of the CUs work; otherwise the 64- or 128-wide tiles of tile_gemm.h (us, 256 x 256 or, at
// widths that are not multiples of 256, its former 128 x 128 tiles -> those: 24 experts 640 x 896, 1,000 rows 379 -> 176; 64 experts
// 384 x 640, 1,536 rows 614 -> 287; but 8 experts 1024 x 512, 1,024 rows, 192 tiles 50 against 79).  With fewer experts than XCDs and
// long reductions a last round of few tiles, or an expert longer than the others, costs more than the smaller tiles do: two tiles
// for every CU there (tile_gemm.h's / 256 x 256, even counts, ~ 1 / sqrt(rank): 4 experts 2048 x 1024, 24 rows 22 / 17, 21 / 17, 300 rows 42 /
// 42, 42 / 37, 2,048 rows 155 / 172, 154 / 152; 4 experts 1024 x 1024, 128 rows 18 / 16, 20 / 18, 600 rows 37 / 36, 40 / 44, 2,048 rows 96 / 90,
// 94 / 120; 6 experts 2048 x 768, 300 rows 47 / 43, 47 / 43, 2,048 rows 179 / 176, 189 / 206; 4 experts 2048 x 2048, 300 rows 73 / 62, 74 / 61,
// 2,048 rows 295 / 262, 311 / 269).
constexpr WgradKernel wgrad_kernel(int64_t A, int64_t H, int64_t I, int64_t E, int64_t gradients, bool accumulate, int64_t cus) {
  const int64_t tiles = E * (H / 256) * (I / 256) * gradients;
  if (H % 256 != 0 || I % 256 != 0 || tiles < cus / 2) return TILES;
  if (E < NXCD && A >= WG_BIG_ROWS * E && tiles < 2 * cus) return TILES;
  if (A >= WG_BIG_ROWS * E) return BIG;
  return A < (tiles < 2 * cus ? WG_RUNS_ROWS_ONE : WG_RUNS_ROWS) * E || accumulate ? RUNS : RING;
}
// Tiles of a run (wgrad_runs_kernel).  Longer runs hide more of a tile's start, as long as there are several of them for
// every CU and none is long (us, runs of 1 / 2 / 4 tiles, even counts: 128 experts 2048 x 768, 36 tiles a CU: 16 rows 225 / 222 /
// 230, 32 rows 252 / 240 / 240, 48 rows 290 / 256 / 243, 96 rows 368 / 321 / 310; 64 experts 1536 x 768, 13 tiles: 24 rows
// 90 / 96, 48 rows 118 / 111, 128 rows 161 / 148; 16 experts 2048 x 1024, 6 tiles, 64 rows 61 / 54 / 58, 512 rows,
// ~ 1 / sqrt(rank) 172 / 181; 32 experts 1024 x 512, 3 tiles: 32 rows 30 / 28, 64 rows 31.3 / 32.7 (37 / 34), 128 rows 44 / 45 (46 / 55); 64 experts
// 512 x 256, 1.5 tiles, 100 rows 26 / 23 (32 / 54)).  Two against one in per cent: 64 experts 1024 x 1024, 12 tiles a CU, 8 rows -7 / -1
// uneven, 32 rows -9 / -5; 128 experts 1024 x 512, 12 tiles, 24 rows -4 / -3; 96 experts 1024 x 1024, 18 tiles, 24 rows -9 / -2; 24 experts
// 2048 x 1024, 9 tiles, 24 rows -7 / -6; but 64 experts 1536 x 768, whose 18 tiles make an odd number of pairs, 24 rows +2 / +10; 64 experts
// 512 x 512, 3 tiles, 24 rows -2 / -9, 48 rows +4 / +13; 128 experts 512 x 512, 6 tiles, 64 rows -4 / -3, 128 rows -7 / +14: with
// four tiles a gradient the longest expert's few workgroups are what the launch waits for.
// tiles: of one gradient of one expert; per_cu: of all of them, for a CU
constexpr int wgrad_run(int64_t A, int64_t E, int64_t tiles, int64_t per_cu) {
  if (per_cu >= 24 && A > 32 * E && A <= 192 * E && tiles % 4 == 0) return 4;
  const int64_t two = (per_cu < 6 ? 64 : 192) / (tiles >= 8 ? 1 : per_cu < 6 ? 2 : 3);
  return tiles % 2 == 0 && per_cu >= 3 && A <= two * E && (per_cu < 12 || per_cu >= 24 || A > 32 * E || tiles % 4 == 0) ? 2 : 1;
}
// Workgroup b runs on XCD b % 8.  Units, sorted by expert, come in chunks of neighbours, and chunk c goes to XCD c % 8 in
// "snake" order (0..7, 7..0, 0..7, ...): the tiles of a chunk read the same rows through one L2.  Chunks used to be whole
// experts, which leaves XCDs idle where experts are few or uneven.  us, whole experts
// -> chunks, even counts / ~ 1 / sqrt(rank): 8 experts 2048 x 1024, 256 rows 58 -> 57 / 81 -> 58, 1,024 rows 143 -> 140 /
// 222 -> 147; 32 experts 1024 x 512, 256 rows 59 -> 59 / 73 -> 61; 128 experts 2048 x 768, 64 rows 323 -> 323 / 337 -> 335.
constexpr int dealt_unit(int block, int chunk) {
  const int xcd = block % NXCD, pos = block / NXCD;
  const int turn = pos / chunk;
  return ((turn & 1) ? turn * NXCD + (NXCD - 1 - xcd) : turn * NXCD + xcd) * chunk + pos % chunk;
}
// The chunk for `units` units, `per_expert` of them an expert's: 16 or more for an XCD where there are as many units, at most an
// expert.  It need not divide an expert's units: halved while it is even it stays whole experts where these have an odd number, or few
// chunks (us, so -> this, even counts / ~ 1 / sqrt(rank): 8 experts 1280 x 768, 128 rows 26 -> 26 / 37 -> 24, 1,024 rows 88 -> 89 / 148 -> 83; 12
// experts 1280 x 1280, 256 rows 83 -> 69 / 87 -> 67; 16 experts 768 x 768, 256 rows 38 -> 39 / 49 -> 38; 24 experts 1536 x 768, 1,024 rows
// 251 -> 254 / 265 -> 245).
constexpr int64_t deal_chunk(int64_t units, int64_t per_expert) {
  const int64_t chunk = units / (16 * NXCD);
  return chunk < 1 ? 1 : chunk < per_expert ? chunk : per_expert;
}
// workgroups that it takes: whole turns of eight chunks
constexpr int64_t dealt_blocks(int64_t units, int64_t chunk) { return ceil_div(units, chunk * NXCD) * chunk * NXCD; }

// ---- fp32 products in tiles of 64 x 64 and below
// Whether they leave the rows that are not there out of the loads (the SPARSE kernels of tile_gemm.h, with what that gains): with up
// to half a tile of rows an expert and at least twelve k-tiles, as long as the tiles fit the CUs at once, which hold three of
// gate/up, four of the others.  Beyond that other tiles hide what it saves, and the branches are left (us, all rows read -> left out:
// gate/up 128 experts 1024 x 512, 16 rows, 1,024 tiles 189 -> 224, 100 experts, 8 rows, 800 tiles 184 -> 202, 128 experts 2048 x 768, 8 rows
// 407 -> 440; but 96 experts 1024 x 512, 768 tiles 147 -> 141; d_x 80 experts 1024 x 512, 20 uneven rows, 1,280 tiles 144 -> 158, 96 experts,
// 8 rows 145 -> 161, but 64 experts 1024 x 768, 8 rows, 1,024 tiles 151 -> 143; d_h 128 experts 2048 x 768, 8 rows, 1,536 tiles 245 -> 251,
// 1024 x 512, 16 rows, 1,024 tiles 113 -> 107).
constexpr bool absent_rows_left_out(bool gate_up, int64_t A, int64_t E, int64_t tile_rows, int64_t col_tiles, int64_t k_tiles, int64_t cus) {
  const int64_t experts = A < E ? A : E;
  return 2 * A <= tile_rows * experts && k_tiles >= 12 && experts * col_tiles <= (gate_up ? 3 : 4) * cus;
}

}  // namespace pk_rules
