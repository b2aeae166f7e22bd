"""Tolerance requests served one after another in the same slot: a first or
last round of nine to sixteen sweeps finds no sums of the request before."""
import time

import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("iters", [8, 9, 12, 23])
def test_same_slot(iters):
    import charming_amd as cam
    with cam.Server("engine", budget_bytes=1 << 28, max_active=1) as srv:
        for seed in (1, 2, 3):
            p = dict(width=300, height=280, iters=iters, tol=1e-12, seed=seed)
            t = srv.submit(p)
            done, until = [], time.time() + 20
            while not done and time.time() < until:
                done = srv.poll()
            g, n, last, first = O.jacobi_solve_tol(300, 280, iters, 1e-12,
                                                   seed=seed)
            c, = done
            assert (c["ticket"], c["hash"], c["iters"], c["residual"],
                    c["residual0"]) == (t, O.grid_hash(g), n, last, first)
