"""The counted waits of renee_amd/csrc/back_wide.hpp: its order of fetches, stores and waits (back_wide_order.hpp, which the kernel takes
its schedule from) is replayed for a wave, tile by tile, for every row count and direction and every length of the tile that is not
whole.  Of the hardware only what holds is assumed: vector-memory operations retire in the order of their issue, and s_waitcnt
vmcnt(N) proves those done that have N or more behind them.  Checked: what a half tile reads has landed when its wave passes the
barrier before it."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "renee_amd", "csrc")


def _compiled(tmp_path_factory, text, numbers):
    """The lines that the program `text`, compiled beside the kernels' sources, prints when it reads `numbers`."""
    gxx = shutil.which("g++") or shutil.which("clang++", path="/opt/rocm/llvm/bin:/opt/rocm/lib/llvm/bin")
    if gxx is None:
        pytest.skip("no host compiler")
    tmp = tmp_path_factory.mktemp("order")
    src, exe = tmp / "order.cpp", tmp / "order"
    src.write_text(text)
    subprocess.run([gxx, "-std=c++17", "-Wall", "-Werror", "-I", CSRC, str(src), "-o", str(exe)], check=True)
    return subprocess.run([str(exe)], check=True, input=" ".join(map(str, numbers)), stdout=subprocess.PIPE, text=True).stdout.splitlines()


@pytest.fixture(scope="module")
def orders(tmp_path_factory):
    """Per RB: G's fetches of a tile, how many of them stand behind the second half's barrier, wait[half][edge] and, slot by slot of
    the two halves, what happens there."""
    src_text = ('#include <cstdio>\n#include "back_wide_order.hpp"\n'
                   'template <int RB> void show() {\n'
                   '  using S = xfc::BackWideOrder<RB>;\n'
                   '  printf("order %d %d %d %d %d %d %d\\n", RB, S::G_FETCH, S::TAIL - 4, S::wait(0, false), S::wait(0, true), S::wait(1, false), S::wait(1, true));\n'
                   '  for (int h = 0; h < 2; ++h)\n'
                   '    for (int n = 0; n < S::N; ++n) {  // in the order of a slot\'s statements\n'
                   '      if (n == S::BAR) printf("%d wait 0\\n", h);\n'
                   '      if (S::w_fetch(n) >= 0) printf("%d w %d\\n", h, S::w_fetch(n));\n'
                   '      if (S::g_fetch(h, n) >= 0) printf("%d g %d\\n", h, S::g_fetch(h, n));\n'
                   '      if (n == S::STORE0) printf("%d store 0\\n", h);\n'
                   '      if (n == S::STORE1) printf("%d store 1\\n", h);\n'
                   '    }\n}\n'
                   'int main() { show<5>(); show<6>(); show<7>(); show<8>(); }\n')
    out = {}
    for line in _compiled(tmp_path_factory, src_text, []):
        v = line.split()
        if v[0] == "order":
            rb, g_fetch, tail, w0, e0, w1, e1 = (int(x) for x in v[1:])
            out[rb] = dict(g_fetch=g_fetch, tail=tail, wait=((w0, e0), (w1, e1)), slots=([], []))
        else:
            out[rb]["slots"][int(v[0])].append((v[1], int(v[2])))
    return out


def _replay(order, tiles, edge, whole):
    """What a wave reads before it is certain to have landed: (tile, half, what).  `edge`: the tile of `whole` labels, or -1."""
    issued, landed, late = [], 0, []  # operations in order; those before `landed` are done

    def read(tile, half, what):
        if tile < tiles and any(op == what for op in issued[landed:]):
            late.append((tile, half, what))

    # before the first tile everything of it is fetched and waited for, then the first fetches of the next one's G
    issued += [("g", 1, j) for j in range(order["tail"])]
    for tile in range(tiles):
        for h in (0, 1):
            for what, number in order["slots"][h]:
                if what == "wait":
                    landed = max(landed, len(issued) - order["wait"][h][0])
                    if tile == edge:
                        landed = max(landed, len(issued) - order["wait"][h][1])
                    at = (tile, 1) if h == 0 else (tile + 1, 0)  # what is read behind this barrier
                    for f in range(4):
                        read(*at, ("w", *at, f))
                    if h == 1:
                        for j in range(order["g_fetch"]):
                            read(*at, ("g", at[0], j))
                elif what == "w":
                    issued.append(("w", tile + 1, h, number))
                elif what == "g":
                    issued.append(("g", tile + (2 if h == 1 else 1), number))
                elif tile != edge or 32 * h + 16 * number < whole:  # else no lane has a label: the wave branches round the stores
                    issued += [("store",)] * 2
    return late


def test_the_replay_has_the_whole_order(orders):
    """Each half tile fetches two pieces of weights and two of momentum, each tile every piece of G once, and stores 64 labels."""
    assert sorted(orders) == [5, 6, 7, 8]
    for order in orders.values():
        first, second = order["slots"]
        for half in order["slots"]:
            assert [n for what, n in half if what == "w"] == [0, 1, 2, 3]
            assert [n for what, n in half if what == "store"] == [0, 1]
            assert [what for what, _ in half].count("wait") == 1
        assert [n for what, n in second if what == "g"] + [n for what, n in first if what == "g"] == list(range(order["g_fetch"]))
        assert len([n for what, n in second if what == "g"]) == order["tail"]
        assert max(max(w) for w in order["wait"]) < 64  # a six-bit counter
    src = open(os.path.join(CSRC, "back_wide.hpp")).read()
    # the replay mirrors these statements of the kernel; if they change, so must the replay
    for statement in ("struct BackWide : BackWideOrder<RB_> {",
                      "if (tile == edge) wait_vmcnt<S::wait(h, true)>();",
                      "wait_lds_vmcnt_barrier<S::wait(h, false)>();",
                      "if constexpr (constexpr int f = S::w_fetch(n); f >= 0) fetch_w(",
                      "if constexpr (constexpr int j = S::g_fetch(h, n); j >= 0) {",
                      "if (32 * h + 16 * lb + (lane_ & 15) < whole) out();",
                      "if constexpr (n == S::STORE0) store(",
                      "if constexpr (n == S::STORE1) store("):
        assert src.count(statement) == 1, statement


@pytest.mark.parametrize("rb", [5, 6, 7, 8])
def test_what_a_half_tile_reads_has_landed(orders, rb):
    order = orders[rb]
    for tiles in range(1, 7):
        assert _replay(order, tiles, -1, 64) == []
        for edge in {0, tiles - 1}:  # from the last labels on, from the first
            for whole in range(1, 64):
                assert _replay(order, tiles, edge, whole) == [], (tiles, edge, whole)


def test_the_replay_finds_stores_that_were_counted_but_not_made(orders):
    """With the whole tiles' counts in the tile that is not whole, too: what follows it is late where its labels make fewer stores, and
    the rows of 449 on lose weights, the others momentum."""
    late = {}
    for rb, order in orders.items():
        counted = dict(order, wait=tuple((whole, whole) for whole, _ in order["wait"]))
        late[rb] = {whole: {op[2][3] for op in _replay(counted, 3, 0, whole) if op[:2] == (1, 0)} for whole in range(1, 64)}
    assert all(late[8][whole] == {0, 1, 2, 3} for whole in range(1, 33)) and all(late[8][whole] == {2, 3} for whole in range(33, 49))
    assert all(late[rb][whole] == {2, 3} for rb, most in ((5, 32), (6, 16), (7, 32)) for whole in range(1, most + 1))
    assert not any(late[rb][whole] for rb in late for whole in range(49, 64))


def test_no_chain_of_dx_is_longer_than_xfc_dx_has_and_none_is_empty(tmp_path_factory):
    """Rows, labels and dims of up to 32 slices of 128: the longest chain of MFMAs of a partial sum of dX against xfc_dx's, whose number of
    sums is that of its workspace.  (Sums without a tile made a step of 512 rows x 64 labels x 768 dims take 108 us, 67 as two passes.)"""
    from renee_amd._lib import lib

    shapes = [(B, L, 128 * slices) for B in (257, 300, 384, 400, 449, 512) for slices in (1, 2, 3, 4, 5, 6, 8, 10, 12, 24, 32)
              for L in (1, 63, 64, 65, 200, 448, 513, 1396, 1827, 1912, 4097, 20011, 131073, 320001, 655363, 1310720, 1537820, 2080392, 2812281)]
    sums = [lib().xfc_gemm_workspace_bytes(B, d, L) // (B * d * 4) for B, L, d in shapes]
    tiles = [-(-L // 64) for _, L, _ in shapes]
    ranges = [min(256 // (d // 128), t) for (_, _, d), t in zip(shapes, tiles)]  # a workgroup per CU
    text = ('#include <cstdio>\n#include "back_wide_order.hpp"\n'
            'int main() { int t, r, s; while (scanf("%d %d %d", &t, &r, &s) == 3) printf("%d\\n", xfc::back_wide_parts(t, r, s)); }\n')
    parts = [int(line) for line in _compiled(tmp_path_factory, text, [n for trs in zip(tiles, ranges, sums) for n in trs])]
    assert len(parts) == len(shapes)
    for shape, t, r, s, p in zip(shapes, tiles, ranges, sums, parts):
        most = -(-t // r)  # tiles of a range; part q of it has those from most * q / p on
        lengths = [most * (q + 1) // p - most * q // p for q in range(p)]
        assert p >= 1 and min(lengths) >= 1 and sum(lengths) == most, shape
        assert 64 * max(lengths) <= -(-(-(-shape[1] // s)) // 64) * 64, shape
    src = open(os.path.join(CSRC, "xfc_kernels.hip")).read()
    assert src.count("return {(int)ranges, back_wide_parts((int)tiles, (int)ranges, sums)};") == 1
