"""Performance cases of the FP64 Jacobi2D solver through its public entry
points: the single solves (message-driven chares, and the default per-launch
form), the solve on a caller-owned device grid, batches of uneven problems,
and the solve server's request loop.

A pass is what a program does with a problem it already holds: re-seed u_0 on
the device where the form solves from u_0, solve, and read the solution back
where the case says so (`fetch`).  The batched and served forms return a
hash, the exact residual and the sweep count per problem; they have no other
output.
"""
import ctypes as C
import math

import numpy as np
import torch

import charming_amd as cam
from charming_amd import serve as SV
from charming_amd import workloads as WL

BOUNDARY = 1.0
NOALLOC_SIDE = 2800  # about the largest square the no-alloc solve takes


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
def _noalloc(w, h, iters, **kw):
    return dict(kind="noalloc", width=w, height=h, iters=iters, **kw)


def _single(form, w, h, iters, rows=0, cols=0, fetch=True, **kw):
    return dict(kind="single", form=form, width=w, height=h, iters=iters,
                chare_rows=rows, chare_cols=cols, fetch=fetch, **kw)


def _batch(n, lo, hi, it_lo, it_hi, tol=0.0, shape=WL.BATCH_SEED, **kw):
    return dict(kind="batch", n=n, side_lo=lo, side_hi=hi, it_lo=it_lo,
                it_hi=it_hi, tol=tol, shape=shape, **kw)


def _serve(n, lo, hi, iters, tol=1e-6, budget_gb=16, shape=WL.SERVE_SEED, **kw):
    return dict(kind="serve", n=n, side_lo=lo, side_hi=hi, iters=iters, tol=tol,
                budget_gb=budget_gb, shape=shape, **kw)


def listed():
    return [
        # a small grid advanced a few sweeps inside a caller's own stream
        # (a smoother step): launches and latency are all there is
        _noalloc(64, 64, 10, name="noalloc 64x64 x10"),
        # the same at an ordinary, odd size
        _noalloc(1021, 683, 100, name="noalloc 1021x683 x100"),
        # and near the largest grid that entry point takes
        _noalloc(2800, 2800, 200, name="noalloc 2800x2800 x200"),
        # the constructor's default form, one launch per sweep, solution read
        _single("plain", 1500, 1100, 250, name="plain 1500x1100 x250"),
        # the smallest message-driven configuration: 4x4 chares of 128^2
        _single("persistent", 512, 512, 100, 4, 4,
                name="chares 512x512 4x4 x100"),
        # a ragged grid on the automatic decomposition (every PE has a chare)
        _single("persistent", 3001, 1777, 250, name="chares 3001x1777 x250"),
        # 8x8 chares of 512^2; the residual and hash are enough here
        _single("persistent", 4096, 4096, 200, 8, 8, fetch=False,
                name="chares 4096x4096 8x8 x200"),
        # the headline configuration of bench.py: 16x16 chares of 1024^2,
        # whose result is the solve's residual and hash
        _single("persistent", 16384, 16384, 1000, 16, 16, fetch=False,
                name="chares 16384x16384 16x16 x1000"),
        # a few small uneven problems in one call: setup and latency
        _batch(24, 64, 512, 50, 500, name="batch 24 of 64..512"),
        # uneven problems that stop on a relative residual (48..1024 per side)
        _batch(64, 48, 1024, 1000, 1000, tol=1e-3,
               name="batch 64 of 48..1024 to 1e-3"),
        # the 512-problem batch of bench.py at the default configuration
        _batch(512, 64, 4096, 50, 500, name="batch 512 of 64..4096"),
        # a burst of requests into a fresh server, run until all are done
        _serve(24, 256, 8192, 2000, name="serve 24 of 256..8192"),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(math.exp(rng.uniform(math.log(lo),
                                                    math.log(hi + 1))))))


def draw(rng):
    kind = rng.choice(("noalloc", "plain", "chares", "chares", "batch",
                       "batch_tol", "serve"))
    if kind == "noalloc":
        return _noalloc(_log_int(rng, 16, NOALLOC_SIDE),
                        _log_int(rng, 16, NOALLOC_SIDE), _log_int(rng, 1, 300))
    if kind == "plain":
        return _single("plain", _log_int(rng, 64, 6000),
                       _log_int(rng, 64, 6000), _log_int(rng, 10, 400))
    if kind == "chares":
        w, h = _log_int(rng, 256, 12000), _log_int(rng, 256, 12000)
        rows = cols = 0
        if rng.random() < 0.6:
            # chares of about 100 .. 1100 cells a side, at most 16 a side
            rows = max(1, min(16, h // rng.randint(100, 1100)))
            cols = max(1, min(16, w // rng.randint(100, 1100)))
        iters = _log_int(rng, 30, 1000)
        return _single("persistent", w, h, iters, rows, cols,
                       fetch=w * h <= 8 << 20)
    shape = rng.randrange(1 << 40)
    if kind == "batch":
        hi = _log_int(rng, 128, 4096)
        return _batch(_log_int(rng, 4, 256), max(32, hi // 64), hi,
                      rng.randint(20, 100), rng.randint(101, 500), shape=shape)
    if kind == "batch_tol":
        hi = _log_int(rng, 96, 2048)
        return _batch(_log_int(rng, 4, 96), max(24, hi // 24), hi, 1000, 1000,
                      tol=10.0 ** -rng.uniform(1.5, 3.5), shape=shape)
    hi = _log_int(rng, 512, 8192)
    return _serve(_log_int(rng, 1, 24), max(64, hi // 32), hi,
                  rng.choice((200, 500, 1000, 2000)),
                  tol=10.0 ** -rng.uniform(4.0, 6.0), shape=shape)


# ---------------------------------------------------------------------------
# what a program holds before the call
# ---------------------------------------------------------------------------
def _pitch(w):
    return (w + 18 + 15) // 16 * 16


def _random_grid(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    h, w = case["height"], case["width"]
    u = torch.full((h + 2, w + 2), BOUNDARY, dtype=torch.float64, device="cuda")
    u[1:-1, 1:-1] = torch.rand(h, w, dtype=torch.float64, device="cuda",
                               generator=g)
    return u


def _problems(case, seed):
    """The batch's or the stream's problems: sizes and sweep counts by the
    case, initial values by the seed."""
    if case["kind"] == "batch":
        arrivals = None
        probs = WL.batch_problems(case["n"], case["side_lo"], case["side_hi"],
                                  case["it_lo"], case["it_hi"],
                                  seed=case["shape"])
        if case["tol"]:
            probs = [dict(p, tol=case["tol"]) for p in probs]
    else:
        arrivals, probs = WL.serve_requests(
            case["n"], 2000.0, case["side_lo"], case["side_hi"], case["tol"],
            case["iters"], seed=case["shape"])
    return arrivals, [dict(p, seed=(seed * 1000003 + i) & (2**63 - 1))
                      for i, p in enumerate(probs)]


def prepare(case, seed):
    if case["kind"] == "noalloc":
        h, w = case["height"], case["width"]
        buf = torch.zeros(h + 2, _pitch(w), dtype=torch.float64, device="cuda")
        buf[:, 15:17 + w] = _random_grid(case, seed)
        out3 = torch.zeros(3, dtype=torch.int64, device="cuda")
        fn = cam.jacobi_lib().chm_jacobi2d_solve_noalloc
        fn.argtypes = [C.c_void_p, C.c_int, C.c_int, C.c_int, C.c_void_p,
                       C.c_void_p]
        return {"case": case, "fn": fn, "buf": buf, "out3": out3,
                "grid": buf[:, 15:17 + w]}
    if case["kind"] == "single":
        chares = None
        if case["chare_rows"] and case["chare_cols"]:
            chares = (case["chare_rows"], case["chare_cols"])
        j = cam.Jacobi2D(case["width"], case["height"], case["iters"],
                         form=case["form"], seed=seed, boundary=BOUNDARY,
                         chares=chares)
        return {"case": case, "solver": j}
    arrivals, probs = _problems(case, seed)
    return {"case": case, "problems": probs, "arrivals": arrivals}


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def _words(*values):
    """Unsigned 64-bit words as an int64 array."""
    return np.array(values, dtype=np.uint64).view(np.int64)


def _halves(residuals):
    return [v for r in residuals for v in (r & (2**64 - 1), r >> 64)]


def run(state):
    case = state["case"]
    if case["kind"] == "noalloc":
        rc = state["fn"](state["buf"].data_ptr(), case["width"], case["height"],
                         case["iters"], torch.cuda.current_stream().cuda_stream,
                         state["out3"].data_ptr())
        if rc != 0:
            raise RuntimeError(f"no-alloc solve: {rc}")
        return {"grid": state["grid"], "words": state["out3"]}
    if case["kind"] == "single":
        j = state["solver"]
        j.reset()
        r = j.solve()
        out = {"words": _words(r.hash, r.residual_lo, r.residual_hi,
                               r.iters_done)}
        if case["fetch"]:
            out["grid"] = j.grid()
        return out
    if case["kind"] == "batch":
        o = cam.batch_run(state["problems"])
        return {"hashes": _words(*o["hashes"]),
                "residuals": _words(*_halves(o["residuals"])),
                "iters": np.array(o["iters"], dtype=np.int64)}
    r = SV.run_stream("engine", state["arrivals"], state["problems"],
                      budget_bytes=case["budget_gb"] << 30)["results"]
    return {"hashes": _words(*[c["hash"] for c in r]),
            "residuals": _words(*_halves([c["residual"] for c in r])),
            "iters": np.array([c["iters"] for c in r], dtype=np.int64)}


# ---------------------------------------------------------------------------
# the work of a pass, and its result in 64 bits
# ---------------------------------------------------------------------------
def _cells(case):
    """(cells, cell updates) of a pass; with a tolerance the sweep cap
    counts."""
    if case["kind"] in ("noalloc", "single"):
        cells = case["width"] * case["height"]
        return cells, cells * case["iters"]
    _, probs = _problems(case, 0)
    return (sum(p["width"] * p["height"] for p in probs), WL.cell_updates(probs))


def work(case):
    cells, updates = _cells(case)
    # u_0 read once and the result written once; five operations an update
    return {"bytes": 16.0 * cells, "flops": 5.0 * updates}


def _u01(seed, h, w):
    """The seeded interior (a counter-based splitmix64 per cell) in int64
    arithmetic modulo 2^64."""
    def s64(v):
        return v - (1 << 64) if v >= 1 << 63 else v

    def srl(x, k):  # logical shift of a signed word
        return (x >> k) & ((1 << (64 - k)) - 1)
    rows = torch.arange(1, h + 1, dtype=torch.int64, device="cuda")[:, None]
    cols = torch.arange(1, w + 1, dtype=torch.int64, device="cuda")[None, :]
    z = s64(seed) + (rows * (1 << 32) + cols + 1) * s64(0x9E3779B97F4A7C15)
    z = (z ^ srl(z, 30)) * s64(0xBF58476D1CE4E5B9)
    z = (z ^ srl(z, 27)) * s64(0x94D049BB133111EB)
    return srl(z ^ srl(z, 31), 11).double() * 2.0**-53


def exact(case, seed):
    if case["kind"] == "noalloc":
        u = _random_grid(case, seed)
    elif case["kind"] == "single" and case["fetch"]:
        h, w = case["height"], case["width"]
        u = torch.full((h + 2, w + 2), BOUNDARY, dtype=torch.float64,
                       device="cuda")
        u[1:-1, 1:-1] = _u01(seed, h, w)
    else:
        return None  # whole numbers only
    for _ in range(case["iters"]):
        c = u[1:-1, 1:-1]
        u[1:-1, 1:-1] = (c + u[1:-1, :-2] + u[1:-1, 2:] + u[:-2, 1:-1] +
                         u[2:, 1:-1]) * 0.2
    return {"grid": u if case["kind"] == "noalloc" else u.cpu().numpy(),
            "words": None}
