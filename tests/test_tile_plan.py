"""Which tiles the forward pass and dW take (renee_amd/csrc/tile_plan.hpp, where the launches take it from), on 256 CUs."""
import pytest
from test_back_wide_order import _compiled

TEXT = r'''
#include <cstdio>
#include "tile_plan.hpp"
int main() {
  using namespace xfc;
  long long M, n, d, loss;
  while (scanf("%lld %lld %lld %lld", &M, &n, &d, &loss) == 4) {
    const long long most = loss ? 512 : ANY_GRID;  // 4096 bytes of doubles
    const FwdPlan p = fwd_plan(M, n, d, loss != 0, 256);
    printf("%d %lld %lld %lld %lld %lld\n", (int)p.tile, (long long)p.first, (long long)fwd_ids(p.tile, M, p.first), (long long)fwd_grid(p, M, 256, most),
           (long long)(p.first < n ? fwd_ids(FWD_WIDE128, M, n - p.first) : 0), (long long)fwd_rest_grid(p, M, n, 256, most));
  }
}
'''
TILES = ("64", "128", "wide", "wide128")


@pytest.fixture(scope="module")
def forward(tmp_path_factory):
    """(rows, labels, dims, with the loss) -> tile, labels it takes, tiles, workgroups; tiles and workgroups of the labels after them."""
    def plans(sizes):
        lines = _compiled(tmp_path_factory, TEXT, [int(v) for s in sizes for v in s])
        return [(TILES[int(line.split()[0])], *map(int, line.split()[1:])) for line in lines]
    return plans


def test_every_place_that_the_plan_prices_is_taken(forward):
    """The plan counts two small tiles to a CU, one of any other: so many workgroups must run, with the loss and without, and for the
    labels that whole rounds of large tiles leave over."""
    sizes = [(M, n, d, loss) for M in (1, 64, 65, 100, 128, 129, 200, 256, 300, 512, 700, 1024) for d in (64, 384, 768, 1024) for loss in (0, 1)
             for n in (8, 1000, 8192, 16384, 32768, 31752, 60008, 72008, 80008, 100008, 131080, 196616, 320008, 655368, 2812288)]
    small = rest = 0
    for size, (tile, first, ids, grid, rest_ids, rest_grid) in zip(sizes, forward(sizes)):
        places = 512 if tile == "wide128" else 256
        assert grid == min(ids, places) and ids % 8 == 0 and 0 < first <= size[1], size
        assert rest_grid == min(rest_ids, 512) and (rest_ids == 0) == (first == size[1]), size
        small += tile == "wide128" and ids >= 512
        rest += rest_ids > 256
    assert small > 50 and rest > 5
