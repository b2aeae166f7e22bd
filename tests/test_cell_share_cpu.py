"""How the fill, hash and residual kernels' workgroups share a grid's cells
(charming_amd/csrc/jacobi2d/cell_share.h, compiled for the host): every cell
exactly once at any shape, and no thread with many more cells than the
average, so that low, wide and narrow, tall grids keep a launch busy too."""
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                    "charming_amd", "csrc", "jacobi2d")
SRC = r"""
#define __host__
#define __device__
#include "cell_share.h"
#include <stdio.h>
#include <stdlib.h>
#include <vector>
// rows cols n_wg threads -> 1 if every cell is taken once, the most cells of
// a thread, cell_wgs
int main(int argc, char** argv) {
  for (int a = 1; a + 3 < argc; a += 4) {
    const int rows = atoi(argv[a]), cols = atoi(argv[a + 1]);
    const int n_wg = atoi(argv[a + 2]), T = atoi(argv[a + 3]);
    std::vector<char> seen((size_t)rows * cols, 0);
    long long most = 0, sum = 0;
    bool once = true;
    for (int w = 0; w < n_wg; w++)
      for (int t = 0; t < T; t++) {
        const chm::jac::CellShare s =
            chm::jac::cell_share(rows, cols, w, n_wg, T, t);
        long long n = 0;
        for (int i = s.row; i < rows; i += s.row_step)
          for (int j = s.col; j < cols; j += s.col_step, n++)
            if (seen[(size_t)i * cols + j]++) once = false;
        sum += n;
        if (n > most) most = n;
      }
    once = once && sum == (long long)rows * cols;
    printf("%d %lld %d\n", (int)once, most,
           rows * cols ? chm::jac::cell_wgs(rows, cols, T, n_wg) : 0);
  }
}
"""


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    d = tmp_path_factory.mktemp("cell_share")
    (d / "main.cpp").write_text(SRC)
    subprocess.check_call(["g++", "-O2", "-std=c++17", "-I", CSRC,
                           str(d / "main.cpp"), "-o", str(d / "main")])
    return str(d / "main")


SHAPES = [(1, 1), (1, 270001), (4, 130000), (16, 100001), (18, 1500), (17, 17),
          (64, 64), (100, 1023), (683, 1021), (1023, 1025), (1500, 300),
          (2801, 257), (100003, 1), (65537, 4), (40000, 16), (30000, 33),
          (5000, 255), (3, 1 << 20)]


@pytest.mark.parametrize("n_wg,threads", [(1, 256), (8, 256), (64, 256),
                                          (1024, 256), (2048, 256), (341, 64),
                                          (16384, 64)])
def test_every_cell_once_and_evenly(exe, n_wg, threads):
    args = [str(v) for r, c in SHAPES for v in (r, c, n_wg, threads)]
    out = subprocess.check_output([exe] + args, text=True).splitlines()
    for (rows, cols), line in zip(SHAPES, out):
        once, most, wgs = map(int, line.split())
        assert once, (rows, cols)
        # lanes are a power of two (half of them idle at worst), rows come in
        # whole turns and row parts are a whole number: a factor of two each;
        # a row is cut no finer than four cells a thread, eight with the rest
        even = -(-rows * cols // (n_wg * threads))
        assert most <= 8 * even + 8, (rows, cols, most, even)
        assert 1 <= wgs <= n_wg


def test_empty_regions_take_no_cell(exe):
    out = subprocess.check_output(
        [exe] + [str(v) for s in ((0, 7), (7, 0)) for v in (*s, 64, 256)],
        text=True).split()
    assert out == ["1", "0", "0"] * 2


SUM_SRC = r"""
#define __host__
#define __device__
#include "cell_share.h"
#include <stdio.h>
#include <stdlib.h>
int main(int argc, char** argv) {
  for (int a = 1; a + 2 < argc; a += 3)
    printf("%d\n", chm::jac::sum_wgs(atoi(argv[a]), atoi(argv[a + 1]), 256,
                                     atof(argv[a + 2])));
}
"""


def test_workgroups_of_a_sum(tmp_path):
    """At least one, at most 1024, no more than have a cell; and where rows
    are few, not so many that their atomics outlast the cells."""
    (tmp_path / "main.cpp").write_text(SUM_SRC)
    exe = str(tmp_path / "main")
    subprocess.check_call(["g++", "-O2", "-std=c++17", "-I", CSRC,
                           str(tmp_path / "main.cpp"), "-o", exe])
    shapes = SHAPES + [(0, 7), (7, 0), (16384, 16384), (1, 1 << 30),
                       (1 << 30, 1)]
    out = subprocess.check_output(
        [exe] + [str(v) for s in shapes for c in (2.5, 5) for v in (*s, c)],
        text=True).split()
    for (rows, cols), a, b in zip(shapes, out[::2], out[1::2]):
        for n in (int(a), int(b)):
            assert 1 <= n <= 1024, (rows, cols, n)
            assert n <= max(1, rows * cols), (rows, cols, n)
    few = subprocess.check_output(
        [exe] + "500 2800 2.5 500 2800 5 200 2800 2.5 200 2800 5".split(),
        text=True).split()
    assert all(int(n) <= 512 for n in few), few
