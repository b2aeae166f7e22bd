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
extern "C" int serve_side(int w, int h, int n_wg, int resident,
                          long max_tiles) {
  return chm::eng::serve_block_pipe(w, h, n_wg, resident, max_tiles);
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
    L.serve_side.argtypes = [ctypes.c_int] * 4 + [ctypes.c_long]

    def batch(probs, n_wg=CUS, max_tiles=MAX_TILES):
        flat = (ctypes.c_int * (5 * len(probs)))(*[v for p in probs for v in p])
        out = (ctypes.c_int * len(probs))()
        L.batch_sides(flat, len(probs), n_wg, max_tiles, out)
        return list(out)
    return batch, L.serve_side


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
