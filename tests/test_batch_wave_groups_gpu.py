"""Rounds that groups of waves run in the task engine (512-thread workgroups):
several full rounds of sixteen sweeps at the tile sides their windows give and
at odd ones, which other rounds take, rings of any size, and tolerance rounds
of twelve, whose filter sums the last sweep only; against the CPU oracle, in a
batch and served from memory that held other problems."""
import time

import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _fixed(p):
    g, res = O.jacobi_run(p["width"], p["height"], p["iters"], seed=p["seed"],
                          mode=p.get("init_mode", 0),
                          boundary=p.get("boundary", 1.0))
    return O.grid_hash(g), p["iters"], res


def _tol(p):
    g, n, last, first = O.jacobi_solve_tol(p["width"], p["height"], p["iters"],
                                           p["tol"], seed=p["seed"],
                                           mode=p.get("init_mode", 0),
                                           boundary=p.get("boundary", 1.0))
    return O.grid_hash(g), n, last


def _check(probs, out):
    for i, p in enumerate(probs):
        want = (_tol if p.get("tol") else _fixed)(p)
        assert (out["hashes"][i], out["iters"][i], out["residuals"][i]) == \
            want, (i, p)


@pytest.mark.parametrize("w,h,iters,kw", [
    (700, 450, 33, dict(boundary=1e6)), (1200, 1101, 49, dict(init_mode=1)),
    (577, 600, 64, dict(boundary=-0.375)), (545, 33, 35, dict())])
def test_tile_sides(w, h, iters, kw):
    # 33, 65 and 545 are odd: their windows would start on even columns, so
    # only a problem of one tile column runs by groups
    import charming_amd as cam
    probs = [dict(width=w, height=h, iters=iters, seed=w + h, block=b, **kw)
             for b in (0, 16, 33, 65, 96, 160, 162, 288, 544, 545, 1024)]
    out = cam.batch_run(probs, wg_threads=512)
    assert len({(out["hashes"][i], out["residuals"][i])
                for i in range(len(probs))}) == 1
    _check(probs[:1], out)


def _tol_problems():
    probs = []
    for i, (b, m) in enumerate([(1e6, 0), (-3e9, 0), (1.0, 1), (0.0, 0)]):
        for k, (side, w, h) in enumerate([(96, 230, 200), (33, 150, 100),
                                          (0, 300, 170), (161, 161, 90),
                                          (16, 60, 41), (288, 12, 40)]):
            for tol in (0.2, 3e-2, 4e-3):
                probs.append(dict(width=w, height=h, iters=600, tol=tol,
                                  block=side, seed=10 * i + k, boundary=b,
                                  init_mode=m))
    return probs


def test_tolerance_rounds_with_any_ring():
    import charming_amd as cam
    probs = _tol_problems()
    out = cam.batch_run(probs, wg_threads=512)
    _check(probs, out)
    stops = {n % 12 for p, n in zip(probs, out["iters"]) if 12 < n < 600}
    assert len(stops) >= 8   # inside rounds, at most places of one


def test_converged_to_the_rounding_floor():
    # the residuals of small grids end at or near zero: there the filter's
    # error term keeps the exact sums in use
    import charming_amd as cam
    probs = [dict(width=13 + i, height=12 + 3 * i, iters=3000, tol=tol, seed=i,
                  boundary=b, block=16 * (i % 2))
             for i, (b, tol) in enumerate([(1.0, 1e-9), (1e6, 1e-12),
                                           (-1e12, 1e-12), (3e9, 1e-11)])]
    _check(probs, cam.batch_run(probs, wg_threads=512))


def test_served_from_memory_that_held_other_problems():
    import charming_amd as cam
    dirty = [dict(width=900, height=700, iters=40, seed=i, boundary=1e300)
             for i in range(6)]
    probs = [dict(width=500, height=300, iters=50, seed=1),
             dict(width=300, height=280, iters=400, seed=2, tol=1e-2,
                  boundary=-7.0),
             dict(width=40, height=700, iters=37, seed=3, init_mode=1),
             dict(width=161, height=100, iters=500, seed=4, tol=5e-3)]

    def serve(srv, ps):
        tickets = {srv.submit(p): p for p in ps}
        assert None not in tickets
        got, until = [], time.time() + 30
        while len(got) < len(ps) and time.time() < until:
            got += srv.poll()
        return {c["ticket"]: c for c in got}, tickets

    cam.batch_run(dirty)
    for _ in range(2):   # the second server takes the first one's memory
        with cam.Server("engine", budget_bytes=1 << 28) as srv:
            serve(srv, dirty[:4])
            done, tickets = serve(srv, probs)
        for t, p in tickets.items():
            c = done[t]
            assert (c["hash"], c["iters"], c["residual"]) == \
                (_tol if p.get("tol") else _fixed)(p), p
        _check(probs, cam.batch_run(probs))
