"""The tile sides that batches and servers choose
(charming_amd/csrc/jacobi2d/tile_rules.h, compiled for the host)."""
import ctypes
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "charming_amd", "csrc", "jacobi2d")
SRC = r"""
#include "tile_rules.h"
// probs: width, height, iters, tolerance (0 or 1), side (0: not given)
extern "C" void batch_sides(const int* probs, int n, int n_wg, long max_tiles,
                            int* sides) {
  std::vector<chm_batch_problem> p(n);
  std::vector<int> b(n);
  for (int i = 0; i < n; i++) {
    const int* q = probs + 5 * i;
    p[i] = {q[0], q[1], q[2], 0, q[3] ? 1e-3 : 0.0, 0, 0, 1.0};
    b[i] = q[4];
  }
  chm::eng::pick_blocks(p.data(), n, n_wg, max_tiles, b);
  for (int i = 0; i < n; i++) sides[i] = b[i];
}
// requests in order: the side of each with all before it resident
extern "C" void serve_sides(const int* wh, int n, int n_wg, long max_tiles,
                            int* sides, int iters) {
  chm::eng::ServeLoad load;
  for (int i = 0; i < n; i++) {
    const int w = wh[2 * i], h = wh[2 * i + 1];
    const int bs =
        chm::eng::serve_block_pipe(w, h, iters, n_wg, load, max_tiles);
    const long tiles = (long)((w + bs - 1) / bs) * ((h + bs - 1) / bs);
    load.requests++;
    load.tiles += tiles;
    load.us += chm::eng::serve_round_us(w, h, iters, tiles, bs);
    sides[i] = bs;
  }
}
"""
CUS, MAX_TILES = 256, 1 << 18


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    d = tmp_path_factory.mktemp("rules")
    (d / "r.cpp").write_text(SRC)
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-I",
                           CSRC, "-I", os.path.join(ROOT, "include"),
                           str(d / "r.cpp"), "-o", str(d / "r.so")])
    L = ctypes.CDLL(str(d / "r.so"))
    L.batch_sides.argtypes = [ctypes.c_void_p, ctypes.c_int, ctypes.c_int,
                              ctypes.c_long, ctypes.c_void_p]
    L.serve_sides.argtypes = L.batch_sides.argtypes + [ctypes.c_int]

    def batch(probs, n_wg=CUS, max_tiles=MAX_TILES):
        flat = (ctypes.c_int * (5 * len(probs)))(*[v for p in probs for v in p])
        out = (ctypes.c_int * len(probs))()
        L.batch_sides(flat, len(probs), n_wg, max_tiles, out)
        return list(out)

    def serve(wh, n_wg=CUS, max_tiles=MAX_TILES, iters=1500):
        flat = (ctypes.c_int * (2 * len(wh)))(*[v for p in wh for v in p])
        out = (ctypes.c_int * len(wh))()
        L.serve_sides(flat, len(wh), n_wg, max_tiles, out, iters)
        return list(out)
    return batch, serve


def test_caps_do_not_tell_where_a_tolerance_stops(rules):
    batch, _ = rules
    sizes = [(889, 857), (400, 1100), (1187, 300), (64, 500), (700, 700)]
    for n in (1, 2, 5):
        same = batch([(w, h, 400, 1, 0) for w, h in sizes[:n]])
        assert batch([(w, h, 400 - 95 * i, 1, 0)
                      for i, (w, h) in enumerate(sizes[:n])]) == same
    # few problems on many workgroups: none is left in large tiles
    assert max(same) == 96
    # fixed counts do count: a short one costs less in large tiles
    mixed = batch([(889, 857, 400, 0, 0), (889, 857, 16, 0, 0)])
    assert mixed[0] < mixed[1]


def test_large_batches_keep_large_tiles(rules):
    batch, _ = rules
    for tol in (0, 1):
        assert set(batch([(1500, 1500, 200, tol, 0)] * 300)) == {544}
        few = batch([(300, 300, 200, tol, 0)] * 4)
        assert few == [few[0]] * 4 and few[0] == 96


def test_given_sides_and_the_tile_limit(rules):
    batch, _ = rules
    assert batch([(900, 900, 50, 0, 33), (900, 900, 50, 1, 8192)]) == [33, 8192]
    # 5000 x 5000 in tiles of 96 would be 2809
    side, = batch([(5000, 5000, 500, 0, 0)], n_wg=100000, max_tiles=2000)
    assert side == 160


def test_a_lone_request_is_spread(rules):
    # small ones in the finest tiles, larger ones in finer ones than 288 as
    # long as the card has room, the largest in few turns of the card
    _, serve = rules
    for side, want in [(100, 64), (300, 64), (600, 64), (1000, 96), (2000, 192),
                       (2048, 192), (3000, 160), (4000, 288), (6000, 288),
                       (8000, 544), (20000, 544)]:
        assert serve([(side, side)]) == [want], side
    assert max(serve([(3000, 50)]) + serve([(50, 3000)]) + serve([(9, 9)])) <= 160


def test_a_few_small_requests_are_spread_too(rules):
    _, serve = rules
    assert set(serve([(300, 300)] * 6)) <= {64, 96}
    assert set(serve([(148, 148)] * 30)) <= {64, 96}


def test_sides_grow_with_the_load(rules):
    _, serve = rules
    for side in (300, 600, 1000, 2000, 5000):
        got = serve([(side, side)] * 60)
        assert got[0] == min(got) and got[-1] == max(got) >= 160
    assert set(serve([(2000, 2000)] * 60)[30:]) == {544}
    # a tile of 300 x 300 would make its round three times as long as four of
    # 160: not even then
    assert serve([(300, 300)] * 100)[-1] == 160


def test_few_sweeps_take_finer_tiles(rules):
    # to seed and hash a tile of 288 takes as long as three of its rounds
    _, serve = rules
    few = serve([(500, 500)] * 11, iters=5)
    many = serve([(500, 500)] * 11, iters=1500)
    assert max(few) < max(many) and all(f <= m for f, m in zip(few, many))


def test_request_tile_limit(rules):
    _, serve = rules
    assert serve([(2000, 2000)], max_tiles=100) == [288]
    assert serve([(2000, 2000)], max_tiles=1) == [544]


def test_partial_tiles_cost_their_own_size(rules):
    # with the card full what counts is the work: two tiles of 544 where the
    # second is a strip cost less than three of 288
    _, serve = rules
    full = [(2000, 2000)] * 60
    for wh in [(584, 1329), (597, 283), (668, 1210), (740, 571), (3323, 1102)]:
        assert serve(full + [wh])[-1] == 544, wh
