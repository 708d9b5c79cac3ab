"""Which tiles the forward pass and dW take, how dW's outputs are stored, and when two gradients take two passes (renee_amd/csrc/tile_plan.hpp, where the launches take it from), on
256 CUs unless said otherwise; tests that run on the GPU take from here what their sizes lead to."""
import pytest
from test_back_wide_order import _compiled

TEXT = r'''
#include <cstdio>
#include "tile_plan.hpp"
int main() {
  using namespace xfc;
  long long what, cus, M, n, d, more, lines;
  while (scanf("%lld %lld %lld %lld %lld %lld %lld", &what, &cus, &M, &n, &d, &more, &lines) == 7) {
    if (what == 0) {
      const long long most = more ? 512 : ANY_GRID;  // 4096 bytes of doubles
      const FwdPlan p = fwd_plan(M, n, d, more != 0, cus);
      printf("%d %lld %lld %lld %lld %lld\n", (int)p.tile, (long long)p.first, (long long)fwd_ids(p.tile, M, p.first), (long long)fwd_grid(p, M, cus, most),
             (long long)(p.first < n ? fwd_ids(FWD_WIDE128, M, n - p.first) : 0), (long long)fwd_rest_grid(p, M, n, cus, most));
    } else if (what == 2) {
      printf("%d\n", (int)gradients_apart(M, n, d, more != 0, cus));
    } else if (what == 4) {
      printf("%d\n", (int)dx_how(M, d, n, more, lines != 0));
    } else if (what == 3) {
      printf("%d\n", (int)back_how(more == 1, more == 2, M, n, d, lines != 0));
    } else {
      const DwPlan p = dw_plan((DwMode)more, n, d, M, lines != 0, cus);
      printf("%d %d\n", (int)p.small, (int)p.how);
    }
  }
}
'''
TILES = ("64", "128", "wide", "wide128")
OUT, UPDATE, MASTER = 0, 1, 2  # of dW
ADD = 2  # of the joint pass, beside OUT and UPDATE
CACHED, PAST, THROUGH = 0, 1, 2


class Plans:
    def __init__(self, tmp_path_factory):
        self.tmp = tmp_path_factory

    def forward(self, sizes, cus=256):
        """(rows, labels, dims, with the loss) -> tile, labels it takes, tiles, workgroups; tiles and workgroups of the labels after them."""
        lines = _compiled(self.tmp, TEXT, [int(v) for s in sizes for v in (0, cus, *s, 0)])
        return [(TILES[int(line.split()[0])], *map(int, line.split()[1:])) for line in lines]

    def dw(self, sizes, cus=256, whole=True):
        """(rows, labels, dims, mode) -> whether by small tiles, how what is written is stored; `whole`: its rows are whole lines."""
        lines = _compiled(self.tmp, TEXT, [int(v) for s in sizes for v in (1, cus, *s, whole)])
        return [(line.split()[0] == "1", int(line.split()[1])) for line in lines]

    def gradients_apart(self, sizes, cus=256):
        """(rows, labels, dims, whether the gradient is added to) -> whether the two gradients take two passes."""
        return [line == "1" for line in _compiled(self.tmp, TEXT, [int(v) for s in sizes for v in (2, cus, *s, 0)])]

    def back(self, sizes, whole=True):
        """(rows, labels, dims, mode: UPDATE, OUT, or ADD) -> how the joint pass stores weights and momentum, or the gradient."""
        return [int(line) for line in _compiled(self.tmp, TEXT, [int(v) for s in sizes for v in (3, 256, *s, whole)])]

    def dx(self, sizes, whole=True):
        """(rows, labels, dims, bytes of partial sums) -> how these are stored."""
        return [int(line) for line in _compiled(self.tmp, TEXT, [int(v) for s in sizes for v in (4, 256, *s, whole)])]


@pytest.fixture(scope="session")
def plans(tmp_path_factory):
    return Plans(tmp_path_factory)


def test_every_place_that_the_plan_prices_is_taken(plans):
    """The plan counts two small tiles to a CU, one of any other: so many workgroups must run, with the loss and without, and for the
    labels that whole rounds of large tiles leave over."""
    sizes = [(M, n, d, loss) for M in (1, 64, 65, 100, 128, 129, 200, 256, 300, 512, 700, 1024) for d in (64, 384, 768, 1024) for loss in (0, 1)
             for n in (8, 1000, 8192, 16384, 32768, 31752, 60008, 72008, 80008, 100008, 131080, 196616, 320008, 655368, 2812288)]
    small = rest = 0
    for size, (tile, first, ids, grid, rest_ids, rest_grid) in zip(sizes, plans.forward(sizes)):
        places = 512 if tile == "wide128" else 256
        assert grid == min(ids, places) and ids % 8 == 0 and 0 < first <= size[1], size
        assert rest_grid == min(rest_ids, 512) and (rest_ids == 0) == (first == size[1]), size
        small += tile == "wide128" and ids >= 512
        rest += rest_ids > 256
    assert small > 50 and rest > 5


def test_gradients_take_the_pass_that_measured_faster(plans):
    """Sizes where one of the two ways took at least a twentieth longer than the other."""
    joint = [(9, 81921, 512, 0), (16, 163841, 256, 0), (33, 61441, 1024, 0), (64, 122881, 1024, 0), (5, 62805, 768, 0), (64, 62805, 768, 0),
             (33, 81921, 768, 1), (64, 163841, 768, 1), (9, 1720321, 256, 1), (64, 245761, 256, 1), (48, 114689, 512, 1), (100, 131072, 384, 1),
             (64, 1638401, 64, 1), (48, 1638401, 64, 1), (9, 262145, 64, 0), (5, 753665, 64, 0), (100, 1638401, 64, 0)]
    apart = [(9, 917505, 64, 0), (33, 1638401, 64, 0), (9, 294913, 64, 1), (33, 655361, 64, 1), (33, 131073, 256, 0), (64, 229377, 256, 0),
             (48, 183501, 320, 0), (48, 204801, 512, 0)]
    assert plans.gradients_apart(joint) == [False] * len(joint)
    assert plans.gradients_apart(apart) == [True] * len(apart)


def test_dw_takes_the_tiles_that_measured_faster(plans):
    """Sizes where one of the two tiles took at least a thirtieth longer than the other, whole calls."""
    large = [(16, 450561, 256, MASTER), (35, 451991, 256, MASTER), (64, 450561, 256, MASTER), (16, 386599, 256, MASTER), (9, 614401, 256, MASTER),
             (64, 1638401, 128, OUT), (40, 1228801, 128, OUT), (128, 450561, 256, OUT), (128, 225281, 512, OUT), (128, 112641, 1024, OUT),
             (256, 655363, 768, OUT), (512, 131072, 768, OUT)]
    small = [(16, 1000000, 128, MASTER), (200, 450561, 256, MASTER), (48, 286721, 256, MASTER), (35, 184321, 384, MASTER), (128, 131073, 768, OUT),
             (600, 4097, 768, UPDATE), (384, 700001, 384, UPDATE), (300, 20001, 1024, MASTER), (128, 409601, 128, OUT)]
    assert [p[0] for p in plans.dw(large)] == [False] * len(large)
    assert [p[0] for p in plans.dw(small)] == [True] * len(small)


def test_rows_that_are_not_whole_lines_are_stored_as_usual(plans):
    """Stored past the L2 they took 1.1 to 1.6 times as long; those of 129 to 255 dims go by tiles that share no line."""
    sizes = [(B, mi * (1 << 20) // d, d, mode) for B in (1, 16, 128, 600) for mi in (20, 50, 200) for d in (72, 136, 200, 776, 1000) for mode in (OUT, UPDATE, MASTER)]
    assert {how for _, how in plans.dw(sizes, whole=False)} == {CACHED}
    assert {how for _, how in plans.dw(sizes)} == {CACHED, PAST, THROUGH}
    joint = [(B, mi * (1 << 20) // d, d, mode) for B in (1, 16, 128, 256) for mi in (4, 15, 30, 120) for d in (72, 136, 200, 776) for mode in (OUT, UPDATE, ADD)]
    assert set(plans.back(joint, whole=False)) == {CACHED}
    assert set(plans.back(joint)) == {CACHED, PAST, THROUGH}
    large = [(16, 80 * (1 << 20) // d, d, mode) for d in (136, 200, 248) for mode in (OUT, UPDATE, MASTER)]
    assert {small for small, _ in plans.dw(large, whole=False)} == {False}
    ours = [(100, 20001, 768, UPDATE), (100, 40001, 768, UPDATE), (100, 80001, 768, UPDATE), (100, 40001, 768, OUT), (100, 80001, 768, ADD)]
    assert plans.back(ours) == [THROUGH, CACHED, PAST, CACHED, PAST]
    small = [(100, 2001, 776, UPDATE), (100, 90001, 776, OUT), (9, 90001, 776, OUT), (100, 90001, 776, ADD), (100, 200001, 776, OUT)]
    assert plans.back(small, whole=False) == [THROUGH, PAST, CACHED, CACHED, CACHED]


def test_partial_sums_of_shared_lines_are_stored_as_usual(plans):
    """Tiles of 256 rows x 256 dims, two waves to a row: 1.05 to 1.36 times as long through the L2s from 129 rows and dims on."""
    sizes = [(B, L, d, 1 << 20) for B in (129, 200, 512, 1024) for L in (1001, 20001) for d in (136, 200, 328, 776, 1000)]
    assert set(plans.dx(sizes, whole=False)) == {CACHED} and set(plans.dx(sizes)) == {THROUGH}
    assert set(plans.dx([(128, 1001, 776, 1 << 20), (512, 1001, 72, 1 << 20)], whole=False)) == {THROUGH}
    assert set(plans.dx([(128, 40001, 768, 1 << 20), (512, 1001, 768, 49 << 20)])) == {CACHED}
