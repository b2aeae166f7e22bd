"""The stop filter of tolerance rounds that sum their last sweep only
(charming_amd/csrc/jacobi2d/stop_filter.h, compiled for the host), against the
exact residuals of every sweep: a round that holds the stop is never passed
over, whatever the boundary, the initial grid, the tolerance and the order of
the FP64 sum, and rounds far from the stop mostly are."""
import ctypes
import math
import os
import subprocess

import numpy as np
import pytest

from oracle import oracle as O

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                    "charming_amd", "csrc", "jacobi2d")


@pytest.fixture(scope="module")
def may_stop(tmp_path_factory):
    d = tmp_path_factory.mktemp("filter")
    (d / "f.cpp").write_text(
        "#define __host__\n#define __device__\n#include \"stop_filter.h\"\n"
        "extern \"C\" int may_stop(double thr, double a, double n, double d,"
        " double m) { return chm::jac::last_sum_may_stop(thr, a, n, d, m); }\n")
    subprocess.check_call(["g++", "-O2", "-std=c++17", "-shared", "-fPIC",
                           "-ffp-contract=off", "-I", CSRC, str(d / "f.cpp"),
                           "-o", str(d / "f.so")])
    f = ctypes.CDLL(str(d / "f.so")).may_stop
    f.argtypes = [ctypes.c_double] * 5
    return lambda *a: f(*a) != 0


def _sweeps(W, H, n, **kw):
    """Exact residuals S_1 .. S_n and the FP64 sums of squared changes."""
    u = O.init_grid(W, H, **kw)
    S, T = [], []
    with np.errstate(over="ignore"):
        for _ in range(n):
            v = O.step(u)
            S.append(O.residual_fixed(v, u))
            d = (v - u)[1:-1, 1:-1]
            T.append(float(np.sum(d * d)))
            u = v
    return S, T


@pytest.mark.parametrize("W,H,n,kw", [
    (13, 12, 2400, dict(seed=1, boundary=1.0)),
    (12, 40, 3000, dict(seed=2, boundary=0.0)),
    (31, 23, 3000, dict(seed=3, boundary=-1e3)),
    (31, 23, 3000, dict(seed=4, boundary=1e6)),
    (13, 12, 2400, dict(seed=5, boundary=-1e12)),
    (23, 19, 6000, dict(seed=9, boundary=1e14)),
    (16, 16, 2400, dict(seed=6, boundary=1e100)),
    (24, 30, 3000, dict(mode=1)),
    (120, 90, 600, dict(seed=7, boundary=1.0)),
    (120, 90, 600, dict(seed=8, boundary=1e6)),
])
def test_no_stop_is_passed_over(may_stop, W, H, n, kw):
    # the sweeps go on until the residuals are down to rounding, where they
    # may rise again and the error term decides
    S, T = _sweeps(W, H, n, **kw)
    m = 10.0 if kw.get("mode") else max(1.0, abs(kw["boundary"]))
    s0 = O.u128_to_double(S[0])
    levels = sorted(set(S))
    tols = [1e-1, 1e-2, 1e-3, 1e-6, 1e-9]
    # and tolerances just at, below and above sweeps' own residuals
    for s in levels[::max(1, len(levels) // 60)]:
        t = math.sqrt(O.u128_to_double(s) / s0) if s0 else 0.0
        tols += [t, t * (1 - 1e-12), t * (1 + 1e-12)]
    passed = looked = 0
    for tol in tols:
        thr = tol * tol * s0
        for k in range(12, n - 11, 12):       # a round: sweeps k+1 .. k+12
            holds = any(O.u128_to_double(s) <= thr for s in S[k:k + 12])
            for slack in (1.0, 1 - 2.0**-23, 1 + 2.0**-23):
                may = may_stop(thr, T[k + 11] * slack, W * H, 12, m)
                assert may or not holds, (tol, k, slack)
            looked += 1
            passed += not may
            if holds:
                break
    assert passed > 0 and looked > passed


def test_the_error_term_is_needed(may_stop):
    # plant a mistake: no rounding (m = 0).  At the rounding floor a round's
    # last residual may be larger than one before it, and stops are missed
    S, T = _sweeps(13, 12, 2400, seed=5, boundary=-1e12)
    missed = [0, 0]
    for k in range(12, 2400 - 11, 12):
        for s in set(S[k:k + 12]):
            thr = O.u128_to_double(s)   # the round holds a stop
            for i, m in enumerate((0.0, 1e12)):
                missed[i] += not may_stop(thr, T[k + 11], 13 * 12, 12, m)
    assert missed[0] > 0 and missed[1] == 0


@pytest.mark.parametrize("a", [0.0, float("inf"), float("nan"), 1e-300, 1.0])
def test_values_out_of_range_go_to_the_exact_sums(may_stop, a):
    big, nan = float("inf"), float("nan")
    assert may_stop(2.0**62, a, 1e4, 12, 1.0)
    assert may_stop(big, a, 1e4, 12, 1.0) and may_stop(nan, a, 1e4, 12, 1.0)
    assert may_stop(1.0, a, 1e4, 12, nan)
    if math.isfinite(a):
        assert may_stop(1.0, a, 1e4, 12, big)
    if a < 1e-10 or math.isnan(a):
        assert may_stop(0.0, a, 1e4, 12, 1.0)
