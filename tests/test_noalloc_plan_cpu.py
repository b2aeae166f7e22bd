"""The launches of a no-alloc solve (charming_amd/csrc/jacobi2d/noalloc_plan.h,
compiled for the host): the sweeps they add up to, their order, and the
largest sweep counts, which take no memory."""
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                    "charming_amd", "csrc", "jacobi2d")
SRC = r"""
#include "noalloc_plan.h"
#include <stdio.h>
#include <stdlib.h>
int main(int argc, char** argv) {
  const int H = atoi(argv[1]);
  for (int a = 2; a < argc; a++) {
    const chm::jac::NoallocPlan p = chm::jac::noalloc_plan(H, atoi(argv[a]));
    printf("%d", p.n);
    for (int i = 0; i < p.n && i < 64; i++) printf(" %d", p[i]);
    if (p.n > 64) printf(" %d %d", p[p.n - 2], p[p.n - 1]);
    puts("");
  }
}
"""


@pytest.fixture(scope="module")
def plan(tmp_path_factory):
    d = tmp_path_factory.mktemp("plan")
    (d / "main.cpp").write_text(SRC)
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-I", CSRC,
                           str(d / "main.cpp"), "-o", str(d / "main")])

    def lines(H, iters):
        out = subprocess.check_output([str(d / "main"), str(H)] +
                                      [str(i) for i in iters], text=True)
        return [list(map(int, l.split())) for l in out.splitlines()]
    return lines


def expected(H, iters):
    left, l = iters - 1, []
    while H >= 16 and left >= 4:
        l.append(min(16, left // 4 * 4))
        left -= l[-1]
    k = len(l)
    l += [1] * (left + 1)
    if len(l) % 2 and k and l[k - 1] > 4:
        l[k - 1:k] = [l[k - 1] - 4, 4]
    elif len(l) % 2 and k and l[0] > 4:
        l[:1] = [l[0] - 4, 4]
    return l


@pytest.mark.parametrize("H", [1, 15, 16, 2800])
def test_every_count(plan, H):
    iters = range(1, 64 if H < 16 else 700)
    for it, got in zip(iters, plan(H, iters)):
        want = expected(H, it)
        assert sum(want) == it and want[-1] == 1
        assert got == [len(want)] + want, (H, it)


def test_largest_counts(plan):
    big = 2**31 - 1
    low, = plan(15, [big])
    assert low[0] == big and set(low[1:]) == {1}
    high, = plan(16, [big])   # 2^31 - 2 = 16 * 134217727 + 14: 12, 1, 1, 1
    assert high[0] % 2 == 0 and high[1] == 16 and high[-1] == 1
    assert high[0] == 134217727 + 2 + 2 + 1
