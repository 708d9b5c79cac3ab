// Which tiles the forward pass and dW take, on how many workgroups, how dX, dW and the joint pass of up to 256 rows store what they write, and when two
// gradients take two passes, as arithmetic on sizes, alignment and the number of CUs: the launches take it from here, and tests/test_tile_plan.py goes
// through it on the host.  Plain C++, nothing of the GPU.
#pragma once
#include <math.h>
#include <stdint.h>

namespace xfc {

inline int ceil_div(int64_t a, int64_t b) { return (int)((a + b - 1) / b); }
inline int64_t round_up(int64_t a, int64_t b) { return (a + b - 1) / b * b; }

// How an output is stored.  CACHED: it stays in the L2 until something pushes it out or the kernel ends, which waits for what its
// eight L2s (32 MB) still hold to be written back.  THROUGH: past the L2 to the Infinity Cache at once (agent scope): nothing is left
// to write back, for outputs about as large as the L2s or smaller; more of them, or pieces of lines, pass the fabric faster when the L2
// has gathered them.  PAST: as what will not be wanted again, past the Infinity Cache too, for outputs that it would not hold.
enum StoreHow { CACHED = 0, PAST = 1, THROUGH = 2 };
// The last two want rows that are whole lines of 128 bytes: a line that two stores, of two labels or of two workgroups, make up is fetched
// and written twice where the L2 may not gather it: 1.1 to 1.6 times the time (see dw_plan, dx_how and back_how).
inline bool whole_lines(const void* p, int64_t ld, int64_t row, int64_t element) {
  return (reinterpret_cast<uintptr_t>(p) | (uintptr_t)(ld * element) | (uintptr_t)(row * element)) % 128 == 0;
}

// ---------------------------------------------------------------------------------------------
// forward pass
// ---------------------------------------------------------------------------------------------
// The labels [0, first) go by `tile`, those after them, if any, by FWD_WIDE128.
enum FwdTile { FWD_64, FWD_128, FWD_WIDE, FWD_WIDE128 };
struct FwdPlan {
  FwdTile tile;
  int64_t first;
};
constexpr int FWD_STAGE = 64;  // dims of a stage
constexpr int fwd_tile_rows(FwdTile t) { return t == FWD_64 ? 64 : t == FWD_WIDE ? 256 : 128; }
constexpr int fwd_tile_labels(FwdTile t) { return t == FWD_WIDE128 ? 128 : 256; }
inline int64_t fwd_ids(FwdTile t, int64_t M, int64_t n) { return ceil_div(M, fwd_tile_rows(t)) * round_up(ceil_div(n, fwd_tile_labels(t)), 8); }
// Large tiles move the fewest bytes through the fetch path, small ones fill the chip with few labels, leave no last round nearly
// empty, and two of them on a CU work at each other's epilogues.  Time in rounds of the large tile, of 256 tiles on as many CUs: a round is
// 8.6 us at 64 dims, 16.5 at 384, 26 at 768, 32 at 1024, 256 small tiles 0.31 of it (with the loss, whose epilogue is the longer,
// 0.28); on the 128-row tile of the eight-wave loop a round is 14.5 to 22 us at 768 dims, and 256 small tiles 0.58 of it.  Measured
// (fwd_grad without pairs, large and small, us): 200 rows x 8,001 labels x 768 dims 27.7 and 10.9, x 30,001 30.7 and 19.7, x
// 60,001 34.6 and 35.7, x 131,073 84 and 73, 256 x 131,072 63 and 81, 512 x 60,001 57 and 70, x 20,001 x 256 21.1 and 13.5, 300 x
// 131,073 x 384 80 and 61, 1024 x 131,072 x 768 219 and 262; 100 rows x 4,097 x 768 14.2 and 10.3, x 60,001 20.7 and 22.8, x 80,001 39.2 and
// 34.3, x 250,001 85 and 96.  Where whole rounds of large tiles leave few labels over, those go by small tiles in a launch of their
// own, 7.5 us and more: whole steps of 512 rows x 131,073 labels x 768 dims 379 -> 370 us, 256 rows 281 -> 273, 512 x 100,001 299 -> 290, with
// the loss 512 x 131,073 414 -> 396.  Whole steps of few labels: 200 x 8,001 62.8 -> 45.4, 300 x 16,001 79 -> 68; top-100 of 200 x 20,001
// 40.4 -> 29.3.
inline FwdPlan fwd_plan(int64_t M, int64_t n, int64_t d, bool loss, int64_t cus) {
  if (M <= 64) return {FWD_64, n};
  auto rounds = [&](FwdTile t, int64_t labels) { return (double)ceil_div(fwd_ids(t, M, labels), cus); };
  if (M <= 128) return {0.58 * rounds(FWD_WIDE128, n) < rounds(FWD_128, n) ? FWD_WIDE128 : FWD_128, n};
  const double small = loss ? 0.28 : 0.31, launch = 7.5 / (7.0 + 1.58 * (double)ceil_div(d, FWD_STAGE));
  const double large = rounds(FWD_WIDE, n);
  FwdPlan best = {FWD_WIDE, n};
  double least = large;
  if (small * rounds(FWD_WIDE128, n) < least) best = {FWD_WIDE128, n}, least = small * rounds(FWD_WIDE128, n);
  // whole rounds, in label tiles that the 8 XCDs divide
  const int64_t first = ((int64_t)large - 1) * cus / ceil_div(M, fwd_tile_rows(FWD_WIDE)) / 8 * 8 * fwd_tile_labels(FWD_WIDE);
  if (first > 0 && first < n && large - 1.0 + launch + small * rounds(FWD_WIDE128, n - first) < least) best = {FWD_WIDE, first};
  return best;
}
// Workgroups of a persistent pass over tiles: as many as the CUs hold (the number of tile ids is a multiple of 8), with the loss no more
// than there are places for its partial sums.  Of the labels that whole rounds leave over the same number again: their sums are
// added to those that are there.
constexpr int64_t ANY_GRID = 0x7fffffff;
inline int64_t persistent_grid(int64_t ids, int per_cu, int64_t cus, int64_t most = ANY_GRID) {
  const int64_t all = per_cu * round_up(cus, 8), grid = all < most ? all : most;
  return grid < ids ? grid : ids;
}
inline int64_t fwd_grid(const FwdPlan& p, int64_t M, int64_t cus, int64_t most) {
  return persistent_grid(fwd_ids(p.tile, M, p.first), p.tile == FWD_WIDE128 ? 2 : 1, cus, most);
}
inline int64_t fwd_rest_grid(const FwdPlan& p, int64_t M, int64_t n, int64_t cus, int64_t most) {
  return p.first < n ? persistent_grid(fwd_ids(FWD_WIDE128, M, n - p.first), 2, cus, most) : 0;
}

// ---------------------------------------------------------------------------------------------
// dW
// ---------------------------------------------------------------------------------------------
enum DwMode { DW_OUT = 0, DW_UPDATE = 1, DW_UPDATE_MASTER = 2 };  // MASTER: fp32 master weights and momentum, fp16 copy of W
constexpr int DW_TILE = 256, DW_SMALL_TILE = 128;  // labels and dims
struct DwPlan {
  bool small;    // tiles of DW_SMALL_TILE
  StoreHow how;  // what is written
};
// Large tiles move the fewest bytes through the fetch path and the L2s; small ones fill the chip with few labels, leave no last round nearly empty, waste less of a
// width that is no multiple of 256, and two of them on a CU work at each other's epilogues.  Compared by rounds of the large ones, four small tiles to one of
// them at a price (in brackets, large and small in us, by themselves unless they are calls):
//   Updates: none while the update's traffic binds, up to a sixth at 1024 rows, whose operands do [32 rows x 8,001 labels x 256 dims 10.9 and 5.7, 128 x 30,001 x
//   768 46 and 37, 600 x 4,097 x 768 22.3 and 11.8, 1024 x 20,001 x 1024 83 and 68, but 1024 x 131,072 x 768 293 and 327], 0.05 more for a state that no cache
//   holds [384 x 700,001 x 384 583 and 537, 1024 x 1,000,001 x 128 728 and 636, but 512 x 655,363 x 768 1000 and 1100].
//   Master weights, 18 bytes each, bind at any rows: none, 0.05 for the most rows and weights [300 x 20,001 x 1024 106 and 82, 512 x 131,072 x 768 393 and 373, 512 x
//   700,001 x 384 1163 and 1064, steps of 512 x 450,001 x 768 1943 and 1911, 128 x 450,001 1532 and 1556, 512 x 655,363 2581 and 2629 or 2828 and 2823, 1024 x
//   655,363 2262 and 2381].  Of up to 64 rows x 256 dims a large tile writes its labels in one piece [steps, small over large, x 450,561 1.04 to 1.07, x 614,401
//   1.00 to 1.03, x 286,721 0.98 to 0.99; other widths 0.98 to 1.03, from 200 rows on 0.96 to 0.98].
//   Gradients that the caches hold: up to a quarter at 1024 rows [300 x 8,001 x 768 13.2 and 10.0, 1024 x 20,000 x 1024 62 and 53].  Others go straight to HBM, in
//   pieces of a tile's width by label, 512 bytes of a small one and 1 KB of a large one: a fifth from 256 rows on
//   [256 x 400,000 x 384 156 and 147, 712 x 80,256 x 512 86.8 and 90.7], two fifths where large ones are whole [512 x 131,072 x 768 121 and 129, 256 x 655,363 x 768
//   505 and 611, 136 x 1,096,208 x 256 243 and 334, 248 x 234,640 x 1024 204 and 227, but 128 x 131,073 x 768 79.7 and 74.7; calls of 128 rows x 110 Mi weights x
//   256, 512, 1024, small over large, 1.05, 1.04, 1.04].  Of up to 64 rows x 65 to 128 dims both write the same pieces, and large ones in longer runs of them [32 x
//   1,000,000 x 128 90 and 100; 64 rows 97 and 92, but calls, small over large, 1.02 to 1.06 from 900,000 labels on and 0.98 x 370,000 to 570,000].
inline bool dw_small_tiles(DwMode mode, int64_t labels, int64_t dims, int64_t rows, bool past, bool lines, int64_t cus) {
  auto rounds = [&](int64_t tile) {  // (a last one nearly empty leaves the others the more of the memory: half of it counts)
    const double n = (double)(ceil_div(dims, tile) * round_up(ceil_div(labels, tile), 8)) / (double)cus;
    return 0.5 * (n + ceil(n));
  };
  const double over = rows > 256 ? (double)((rows < 1024 ? rows : 1024) - 256) : 0.0;
  double price = 1.0 + 0.0002 * over;
  if (mode == DW_UPDATE && past) price += 0.05;
  const int64_t Mi = (int64_t)1 << 20, weights = labels * dims;
  if (mode == DW_OUT) {
    if (past && dims % DW_TILE == 0 && weights > (rows < 128 ? 120 : 100) * Mi) price = 1.4;
    else if (past && rows >= 256) price = 1.2;
    else if (past && rows <= 64 && dims > 64 && dims <= DW_SMALL_TILE) price = 2.2;  // (half of a large tile empty: what it multiplies is little)
    else price += 0.0001 * over;
  }
  if (mode == DW_UPDATE_MASTER) {
    price = 0.99;
    if (rows > 512 || weights > (rows <= 128 ? 160 : 380) * Mi) price = 1.04;
    else if (past && rows <= 64 && dims == DW_TILE) price = 1.03;
  }
  if (!lines && dims > DW_SMALL_TILE && dims < DW_TILE && weights > 24 * Mi && price < 1.1) price = 1.1;
  return price * rounds(DW_SMALL_TILE) < 4.0 * rounds(DW_TILE);
}
// Non-temporal stores where what is written would push out of the caches what the next kernels read, from about their size on.  A
// gradient: six-argument calls of 512 rows x 131,072 labels x 768 dims 384 -> 347 us, 128 rows 212 -> 178, 512 x 200,000 x 256 303
// -> 261, x 80,000 x 768 258 -> 241, but x 32,768 118 -> 120.  Master weights: steps of 512 x 655,363 x 768 2868 -> 2813, 64 x
// 200,001 717 -> 668, 256 x 131,072 x 256 201 -> 193, but 256 x 20,001 x 768 115 -> 123.  fp16 state: 1024 x 2,812,281 x 768 13.81 ->
// 13.67 ms, x 700,001 3.48 -> 3.44, but 800 x 200,001 x 512 684 -> 688, 700 x 131,072 x 256 228 -> 235.  Not only back to back: the
// calls of 512 rows x 131,072 each followed by a copy of 512 MiB 567 -> 522, by 0.6 ms of matrix products 1011 -> 978, waited for 409 -> 373.
// Small ones are written through (see StoreHow).  Over three states in turn and over one (us): master weights 64 rows x 5,001
// labels x 768 dims 49.7, 50.3 -> 45.3, 46.7, 300 x 10,001 94, 86 -> 93, 73, but 100 x 20,001 97.6, 83.9 -> 99.2, 81.2; fp16 state 600 x
// 8,001 77.1, 77.4 -> 72.6, 73.8, 800 x 60,001 306, 305 -> 304, 301, but 1024 x 131,072 687 -> 694.  Gradients, six-argument calls of 128 x
// 20,000 50.9 -> 47.9; by themselves, with G out of HBM, larger ones lose: 256 x 23,293 x 1024 32 -> 37, 512 x 27,823 x 1024 49 -> 61.
// Rows that are not whole lines are stored as usual, all but small ones, and those of 129 to 255 dims and more than 24 Mi weights by large tiles, whose workgroups share
// no line of a label.  Whole calls, by the rules of whole lines and as usual (us): updates of 16 rows x 36 Mi weights of 136 dims 177 and 134, of 776 148 and
// 110, of 1000 136 and 113, x 150 Mi of 136 703 and 511, of 776 624 and 501, 128 rows x 150 Mi of 200 772 and 580; master weights 16 x 36 Mi of 776 248 and
// 220, 128 x 150 Mi of 200 1323 and 1072; gradients of 16 x 150 Mi of 776 404 and 294, 128 x 150 Mi of 200 510 and 394, but 6 to 12 Mi 0.94 to 0.97.
inline DwPlan dw_plan(DwMode mode, int64_t labels, int64_t dims, int64_t rows, bool lines, int64_t cus) {
  const int64_t weights = labels * dims, Mi = (int64_t)1 << 20;
  const bool through = weights <= (mode == DW_OUT ? 16 : mode == DW_UPDATE ? (lines ? 48 : 3) : lines ? 12 : 0) * Mi;
  const bool past = weights > (mode == DW_UPDATE ? 140 : mode == DW_UPDATE_MASTER ? 28 : 40) * Mi;
  return {dw_small_tiles(mode, labels, dims, rows, past, lines, cus), past && lines ? PAST : through ? THROUGH : CACHED};
}

// ---------------------------------------------------------------------------------------------
// dX
// ---------------------------------------------------------------------------------------------
// How dX's partial sums are stored.  Those that the L2s hold much of through them: six-argument calls of 512 rows x 20,000 labels x 768 dims 92.5 -> 90.0
// us, steps of 600 x 8,001 77.0 -> 75.4, x 20,001 115.4 -> 113.7, but 512 x 60,000 192.6 -> 194.2, 1024 x 60,001 x 256 179 -> 184, and longer axes, whose pass is not
// waited for as long, too (dX by itself: 100 x 119,605 x 384 35.2 -> 37.2, 899 x 106,385 x 768 162 -> 167).  Not where rows that are not whole lines go by tiles
// of 256 rows, whose waves share the lines about dim 128: dX by itself through and as usual, 200 rows x 1,001 labels x 200 dims 15.4 and 12.0, 512 x 20,001 x
// 328 30.0 and 26.2, 1024 x 4,001 x 776 31.5 and 29.1; up to 128 dims or rows through 0.94 to 0.95 of as usual, whatever the width.
inline StoreHow dx_how(int64_t rows, int64_t dims, int64_t labels, int64_t bytes, bool lines) {
  const bool apart = lines || rows <= 128 || dims <= 128;
  return apart && bytes <= (int64_t)48 << 20 && labels <= 40000 ? THROUGH : CACHED;
}

// ---------------------------------------------------------------------------------------------
// both gradients of a batch of up to 256 rows
// ---------------------------------------------------------------------------------------------
constexpr int BACK_DIMS = 128;  // of a slice of the joint pass

// How the joint pass stores what it writes, weights and momentum or a gradient.
// PAST, the loads of these arrays with the same hint, from where they push out of the Infinity Cache (256 MB) what the forward pass left there of G and the
// weights.  Whole steps with the hint over without, 9 to 256 rows x 64 to 1024 dims, means at some MiB of weights and momentum:
//                                              80     120     150     180     210     240     320     480
//   a state by itself, back to back          1.10    1.08    1.07    1.05    1.02    1.00    0.99    0.95
//   three states in turn                     1.02    0.96    0.94    0.94    0.94    0.94    0.92    0.91
//   with 0.6 ms of matrix products between   1.08    1.05    1.00    1.00    1.00    1.00    0.98
//   with a copy of 256 MiB between                   0.97    0.97    0.97    0.97    0.96
// (The products' operands are 96 MB, and their columns 110, 150, 180, 200, 220, 245 and 300.)  By itself a state of few rows loses the most, 9 to 64 rows x 150 MiB
// 1.1 to 1.17, 224 and 256 rows x 180 0.96 to 1.08: what it stores through the caches is written back by whoever runs next, which is nobody there.  A
// training step has the encoder's between, so the line is where the last three have come even.  A gradient: two micro-batches of 128 x 50,001 x 384 (110
// MiB with W) without and with 167 and 169, by themselves 158 and 161, with products 793 and 794, of 100 x 90,001 x 384 (198) 270, 260, 907 and 269, 263, 904.
// THROUGH for small updates.  Whole steps, over three states in turn and over one (us): 64 rows x 4,097 labels x 768 dims 25.2 -> 24.0, 100 x 10,001 40.5,
// 40.7 -> 39.1, 38.8, 200 x 20,001 66.5, 60.7 -> 65.7, 59.6; but 100 x 40,001 88.4, 80.1 -> 90.4, 77.8.  (Of a gradient it makes no difference: 200 x 5,001 to
// 256 x 40,001 x 384.)
// Where rows are not whole lines, as a rule neither.  PAST over CACHED, a state by itself, three, and with the copy between: 9 rows x 150 MiB of 136 dims 1.66, 1.14,
// 1.14, of 200 1.66, 1.32, 1.34, of 776 1.51, 1.15, 1.16, 256 rows x 245 MiB of 776 1.22, 1.17, 1.15, 48 x 245 of 56 1.10, 1.05, 1.06 (of 24 and 40 dims 0.97 to
// 1.04); a gradient that is added to 1.0 to 1.29, one that is written 1.05 to 1.4 of 9 rows or 150 Mi weights, but 0.87 to 1.04 of 64 to 256 rows x 70 Mi.
// THROUGH over CACHED 64 rows x 62 MiB of 72 dims 1.24, of 200 1.29, of 776 1.10, 256 x 30 MiB 1.05 to 1.07, but 0.93 to 0.97 of 6 MiB.
inline StoreHow back_how(bool update, bool adds, int64_t B, int64_t L, int64_t d, bool lines) {
  const int64_t weights = L * d, Mi = (int64_t)1 << 20;
  if (weights * (update ? 4 : 6) > (update ? 144 : 224) * Mi)
    return lines || (!update && !adds && B >= 64 && weights <= 100 * Mi) ? PAST : CACHED;
  return update && weights * 4 <= (lines ? 64 : 8) * Mi ? THROUGH : CACHED;
}

// Whether dX and a gradient that is written out take two passes instead of the joint one (back_step.hpp).  Whole micro-batches, time by
// the joint pass over that by two:
//   Up to 48 rows of up to 64 dims, which leave half of the joint pass's slice empty: 5 rows 0.9 at 46 Mi weights and 1.12 to 1.16 above, 9 rows
//   1.13 to 1.17, 33 rows 1.13 and at 100 Mi 1.05.  A gradient that is added to from 8 Mi on, 1.04 to 1.18, but 33 and 48 rows 0.93 to 1.03 from 52 Mi on.
//   33 to 64 rows of 256 to 383 dims, or 512, up to 110 Mi weights: 256 dims 1.02 to 1.09 from 26 Mi on, 320 dims 1.06 to 1.14, 512 dims 0.87 to 1.05
//   up to 56 Mi and 33 and 48 rows 1.09 at 100.  Of 33 to 128 rows of 384 to 512 up to 52 Mi only: 0.86 to 1.11 there, 0.87 to 1.05 above.
//   129 rows and more on long axes where the slices do not come out even with the CUs (768 dims, six of them on 240 CUs: 192 rows x 1,500,001
//   1.69 against 1.58 ms, 256 rows 1.98 against 1.77; 1024 dims, all CUs: 192 x 700,001 1.00 against 1.04).
// The last two for a gradient that is only written, which leaves the joint pass little to save, the second reading of G; of one that is
// added to it takes 0.7 to 0.9 from 46 Mi on.  Elsewhere it is the faster, or the same: up to 32 rows of 256, 512, 768 or 1024 dims x 46 Mi and
// more 0.83 to 0.96, 33 to 64 rows of 768 or 1024 dims 0.83 to 1.0.  (65 to 128 rows of less than 5 Mi up to 1.2, 2 to 5 us.)
inline bool gradients_apart(int64_t B, int64_t L, int64_t d, bool adds, int64_t cus) {
  const int64_t weights = L * d, Mi = (int64_t)1 << 20;
  if (d <= 64 && B <= 48) return adds ? weights > 8 * Mi && (B <= 32 || weights <= 48 * Mi) : weights > 48 * Mi;
  if (adds || B <= 32) return false;
  if (B <= 128) {
    const int64_t most = B <= 64 && (d < 384 || d == 512) ? 110 : B <= 64 || d >= 384 ? 52 : 0;
    return d >= 256 && d <= 512 && weights > 20 * Mi && weights <= most * Mi;
  }
  const bool even = (cus / 8) % ceil_div(d, BACK_DIMS) == 0;
  return d % 256 == 0 && !even && weights > 400 * Mi;
}

}  // namespace xfc
