// Which tiles the forward pass and dW take, on how many workgroups, and how dW's outputs are stored, as arithmetic on sizes and the number of
// CUs: the launches take it from here, and tests/test_tile_plan.py goes through it on the host.  Plain C++, nothing of the GPU.
#pragma once
#include <math.h>
#include <stdint.h>

namespace xfc {

inline int ceil_div(int64_t a, int64_t b) { return (int)((a + b - 1) / b); }
inline int64_t round_up(int64_t a, int64_t b) { return (a + b - 1) / b * b; }

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

}  // namespace xfc
