"""The pieces in which a grid is read back
(charming_amd/csrc/jacobi2d/read_plan.h, compiled for the host): every cell
once, in order, and no piece longer than a pinned buffer at any shape."""
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                    "charming_amd", "csrc", "jacobi2d")
SRC = r"""
#include "read_plan.h"
#include <stdio.h>
#include <stdlib.h>
int main(int argc, char** argv) {
  const int rows = atoi(argv[1]), cols = atoi(argv[2]);
  const chm::jac::ReadPlan p = chm::jac::read_plan(rows, cols);
  size_t at = 0;
  bool whole = true;
  for (int k = 0; k < p.n; k++) {
    whole = whole && p.first(k) == at && p.rows_of(k) >= 1 &&
            p.cols_of(k) >= 1 && (p.rows_of(k) == 1 || p.cols_of(k) == cols) &&
            p.rows_of(k) <= p.rows && p.cols_of(k) <= p.cols;
    at += (size_t)p.rows_of(k) * p.cols_of(k);
  }
  whole = whole && at == (size_t)rows * cols;
  printf("%d %zu %d\n", (int)whole, (size_t)p.rows * p.cols * 8, p.n);
}
"""


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    d = tmp_path_factory.mktemp("read")
    (d / "main.cpp").write_text(SRC)
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-I", CSRC,
                           str(d / "main.cpp"), "-o", str(d / "main")])
    return str(d / "main")


@pytest.mark.parametrize("rows,cols", [
    (3, 3), (512, 256), (513, 256), (512, 257), (1102, 1502), (3, 131072),
    (3, 131073), (7, 140003), (18, 1000002), (3, 2**30 + 2), (2**30 + 2, 3),
    (2**30 + 2, 4)])
def test_pieces(exe, rows, cols):
    whole, nbytes, n = map(int, subprocess.check_output(
        [exe, str(rows), str(cols)], text=True).split())
    assert whole and nbytes <= 1 << 20
    assert n <= 3 * (rows * cols * 8 / (1 << 20) + rows * (cols > 131072)) + 1
