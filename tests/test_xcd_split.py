"""How launches over token tiles deal (expert, token tile, row block) triples to the XCDs (``csrc/bp_xcd.h``), compiled for the
host: every triple once, equal eighths, and no pattern of hot experts that leaves most XCDs idle."""

import ctypes as C
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parent.parent / "deepseekternarized_amd" / "csrc"

SOURCE = """
#include "bp_xcd.h"
extern "C" long items(long E, long max_rows, int rows, long blocks) { return bp::tile_items(bp::tile_split(E, max_rows, rows, blocks)); }
extern "C" void deal(long E, long max_rows, int rows, long blocks, int* out) {  // per workgroup: expert, tile, row block, or -1s
  bp::TileSplit s = bp::tile_split(E, max_rows, rows, blocks);
  const unsigned n = (unsigned)bp::tile_items(s);
  s.eighth = n / 8;
  for (unsigned i = 0; i < n; ++i) {
    unsigned e = 0, t = 0, b = 0;
    const bool any = bp::tile_item(s, i, e, t, b);
    out[3 * i] = any ? (int)e : -1, out[3 * i + 1] = any ? (int)t : -1, out[3 * i + 2] = any ? (int)b : -1;
  }
}
extern "C" unsigned over(unsigned n, unsigned d) { return bp::quotient(n, bp::divisor(d)); }
extern "C" long listed(long cap, int rows, long blocks) { return bp::list_items(rows, cap, blocks); }
extern "C" void deal_list(long cap, int rows, long blocks, int* out) {  // per workgroup: position in the list, row block
  const unsigned n = (unsigned)bp::list_items(rows, cap, blocks);
  const bp::TileSplit s = bp::tile_split(1, 1, rows, blocks);
  for (unsigned i = 0; i < n; ++i) {
    unsigned b = 0;
    out[2 * i] = (int)bp::list_item(s, rows, i, b);
    out[2 * i + 1] = (int)b;
  }
}
"""


@pytest.fixture(scope="module")
def deal(tmp_path_factory):
    d = tmp_path_factory.mktemp("xcd")
    (d / "x.cpp").write_text(SOURCE)
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-Wall", "-Werror", f"-I{CSRC}", str(d / "x.cpp"), "-o", str(d / "x.so")], check=True)
    lib = C.CDLL(str(d / "x.so"))
    lib.items.restype, lib.items.argtypes = C.c_long, [C.c_long, C.c_long, C.c_int, C.c_long]
    lib.deal.argtypes = [C.c_long, C.c_long, C.c_int, C.c_long, C.POINTER(C.c_int)]

    def run(E, max_rows, rows, blocks):
        n = lib.items(E, max_rows, rows, blocks)
        out = (C.c_int * (3 * n))()
        lib.deal(E, max_rows, rows, blocks, out)
        return [(i & 7, out[3 * i], out[3 * i + 1], out[3 * i + 2]) for i in range(n) if out[3 * i] >= 0], n

    def run_list(cap, rows, blocks):
        n = lib.listed(cap, rows, blocks)
        out = (C.c_int * (2 * n))()
        lib.deal_list(cap, rows, blocks, out)
        return [(i & 7, out[2 * i], out[2 * i + 1]) for i in range(n)]

    lib.listed.restype, lib.listed.argtypes = C.c_long, [C.c_long, C.c_int, C.c_long]
    lib.deal_list.argtypes = [C.c_long, C.c_int, C.c_long, C.POINTER(C.c_int)]
    lib.over.restype, lib.over.argtypes = C.c_uint, [C.c_uint, C.c_uint]
    run.items, run.list, run.over = lib.items, run_list, lib.over
    return run


@pytest.mark.parametrize("rows", [32, 128])
@pytest.mark.parametrize("E", [1, 2, 7, 8, 9, 15, 16, 20, 64, 385])
def test_every_triple_once_in_equal_eighths(deal, rows, E):
    for max_rows in (1, 32, 33, 129, 257, 600):
        for blocks in (1, 3, 8):
            got, n = deal(E, max_rows, rows, blocks)
            tiles = -(-max_rows // rows)
            assert n % 8 == 0
            assert sorted(g[1:] for g in got) == [(e, t, b) for e in range(E) for t in range(tiles) for b in range(blocks)]
            # the grid holds no more than the items, those that fill up an expert's last run (none with fewer than eight
            # experts) and the rounding to eighths
            runs = 1 if E < 8 else -(-tiles // max(1, 64 // rows))
            assert n - 8 < E * runs * -(-tiles // runs) * blocks <= n


# E experts, those of `hot` with rows: work items of the busiest XCD against an even split
@pytest.mark.parametrize("E,hot,rows_each,worst", [
    (64, range(0, 8), 512, 1), (64, range(8, 16), 512, 1), (64, range(4, 12), 512, 1), (64, range(16, 32), 256, 1), (384, range(96, 104), 64, 1),
    (64, range(0, 64, 8), 512, 1), (64, range(0, 64, 8), 256, 2), (64, [17], 512, 1), (20, range(2, 10), 96, 1.5), (1, [0], 777, 1.1), (3, [1], 2048, 3.1)])
def test_hot_experts_are_spread(deal, E, hot, rows_each, worst):
    got, _ = deal(E, rows_each, 32, 8)
    live = [g for g in got if g[1] in set(hot)]
    per = [sum(1 for g in live if g[0] == x) for x in range(8)]
    assert max(per) <= worst * -(-len(live) // 8)


def test_more_workgroups_than_a_grid_holds(deal):
    assert deal.items(65535, 1 << 20, 32, 64) == -1 and deal.items(1, 1 << 31, 32, 1 << 10) == -1
    assert 0 < deal.items(1, 1 << 20, 32, 32) <= 0x7FFFFFF8


@pytest.mark.parametrize("rows", [32, 128])
def test_lists_of_tiles(deal, rows):
    """Every position of a list once with every row block; 128 token rows in a row on one XCD, the next 128 on the next."""
    for cap in (1, 7, 16, 100):
        got = deal.list(cap, rows, 3)
        assert sorted(g[1:] for g in got) == [(p, b) for p in range(len(got) // 3) for b in range(3)] and len(got) // 3 >= cap
        assert all(xcd == p * rows // 128 % 8 for xcd, p, _ in got)


def test_quotients(deal):
    most = 2**31 - 1
    for d in [*range(1, 70), 127, 128, 1000, 4095, 4097, 65535, 10**6 + 3, 2**30 - 1, 2**30, 2**30 + 1, most]:
        for n in (0, 1, d - 1, d, d + 1, 7 * d - 1, 7 * d, most // d * d - 1, most // d * d, most - 1, most):
            if 0 <= n <= most:
                assert deal.over(n, d) == n // d, (n, d)
