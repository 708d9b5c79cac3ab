// The order of back_wide.hpp's fetches, stores and counted waits, as arithmetic on a slot's number, and the lengths of its sums: the
// kernel and its launch take both from here, and tests/test_back_wide_order.py goes through them on the host.  Plain C++, nothing of the GPU.
#pragma once

namespace xfc {

// Into how many partial sums of dX a range of labels is divided: a tile's labels are part of one chain of MFMAs, as in xfc_dx, and
// there are as many chains as xfc_dx has (`sums`) or more, but none without a tile.
constexpr int back_wide_parts(int tiles, int ranges, int sums) {
  const int want = (sums + ranges - 1) / ranges, most = (tiles + ranges - 1) / ranges;
  return want < most ? want : most;
}

// For up to 64 RB rows.
template <int RB_>
struct BackWideOrder {
  static constexpr int RB = RB_, RP = 2 * RB;
  static constexpr int G_FETCH = 2 * RB;  // fetch instructions (8 rows x 64 labels of G) of a wave per tile
  // The slots of half a tile: a wave's MFMAs, dW's and then dX's.
  static constexpr int DW = 4 * RP, N = DW + 8 * RB;
  static constexpr int BAR = N - 18;                // the barrier stands before this one
  static constexpr int AHEAD = 3;                   // fragments of G are read so many groups of four slots ahead
  static constexpr int TAIL = (N - BAR - 3) / 3 + 1;  // fetches behind the barrier: every third slot has one
  static constexpr int PACE = RB >= 6 ? 1 : RB == 5 ? 2 : 3;      // pieces of the update per slot, 16 for each 16 labels, then their stores
  static constexpr int UPD = DW + 10, STORE0 = UPD + 16 / PACE, STORE1 = UPD + 33 / PACE;
  static_assert(TAIL >= 4 && 3 * (G_FETCH + 3) - (N - BAR - 2) < BAR && STORE1 < N && STORE0 - 4 < BAR && 4 * AHEAD < N - BAR, "schedule");

  // What is fetched in slot n of a tile's half h, -1 if nothing.  Behind a half's barrier the same half of the next tile's weights (0, 1) and
  // momentum (2, 3); then G, of the tile after the next behind the second half's barrier, of the next one before the first half's.
  static constexpr int fetches(int n) { return n > BAR ? n - BAR - 2 : n + N - BAR - 2; }  // slots from the barrier's first fetch on
  static constexpr bool fetch_at(int n) { return n != BAR && fetches(n) >= 0 && fetches(n) % 3 == 0; }
  static constexpr int w_fetch(int n) { return n > BAR && fetch_at(n) && fetches(n) / 3 < 4 ? fetches(n) / 3 : -1; }
  static constexpr int g_fetch(int h, int n) {
    const int j = fetches(n) / 3 - 4;
    return fetch_at(n) && (n > BAR ? h == 1 && j >= 0 : h == 0 && j < G_FETCH) ? j : -1;
  }

  // A wave waits at half h's barrier until at most so many vector-memory operations are outstanding: those that it has issued at least
  // behind the fetches that the next half reads, weights and momentum, which are the last of them.  Two stores for each
  // 16 labels are counted where they are made, that is, not in the tile that is not whole (`edge`): there a wave branches round those
  // whose labels are none.  That tile is a range's first where the pass runs from the last labels on, and another one follows it.
  static constexpr int STORES = (STORE0 < BAR ? 2 : 0) + (STORE1 < BAR ? 2 : 0);
  static constexpr int wait(int h, bool edge) { return (h == 0 ? G_FETCH : 0) + (edge ? 0 : STORES); }
};

}  // namespace xfc
