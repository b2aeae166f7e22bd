"""CPU model of the sweeps that a group of four waves shares
(charming_amd/csrc/jacobi2d/pipeline.h): the windows of a block, the rows each
sweep keeps (the newest input row and the sum that waits for its south
neighbour), the row handed from sweep to sweep, the grid's ring rows and
columns, and the LDS links between waves with every wave stepping at random.
The model restates the device code's arithmetic and counters, so a wrong
window, ring cell, step or link slot shows up here before any GPU run."""
import numpy as np
import pytest

from oracle import oracle as O

RING, LINK, NONE = 6, 2, 1 << 29


def split(c0, c1, left, right, flat, d, k):
    win = 64 * k
    stride = win - 2 * d
    rl, rr = left >= c0 - d and left != NONE, right < c1 + d
    lo = left + flat if rl else c0 - d
    first = lo if lo & 1 else lo - 1
    hi = right - (flat and right & 1) if rr else c1 - 1 + d
    over = hi - first + 1 - win
    n = 1 if over <= 0 else 1 + -(-over // stride)
    return n, first, stride, hi, win, rl, rr


def pick_k(c0, c1, left, right, flat, d):
    return min((9, 5, 3), key=lambda k: split(c0, c1, left, right, flat, d,
                                              k)[0] * (k + 2))


def windows(c0, c1, left, right, flat, d, k):
    """(w0, oc0, oc1, left, right, cols) of every window."""
    n, first, stride, hi, win, rl, rr = split(c0, c1, left, right, flat, d, k)
    out = []
    for i in range(n):
        w0, last = first + i * stride, i == n - 1
        ends = last and rr and flat and (n > 1 or not rl)
        if ends:
            w0 = hi + 1 - win
        assert w0 & 1
        wl = left if rl and i == 0 and not flat else NONE
        wr = right if rr and last and w0 + win > right else NONE
        cols = 0 if wl == wr == NONE else (2 if ends else 3)
        out.append((w0, c0 if i == 0 else first + i * stride + d,
                    c1 if last else min(c1, first + (i + 1) * stride + d),
                    wl, wr, cols))
    return out


class Wave:
    """Wave `role` of a group: one call of step() is one step of the device
    code, which returns False while it would wait for another wave."""

    def __init__(self, role, nst, a, win, k, r0, r1, top, bottom, ring):
        self.role, self.nst, self.a = role, nst, a
        (self.w0, self.oc0, self.oc1, self.left, self.right, self.cols) = win
        self.k, self.r0, self.r1, self.top, self.bottom = k, r0, r1, top, bottom
        self.ns, self.d = nst + 2, 4 * nst
        ns = self.ns
        self.n_steps = -(-(r1 - r0 + 2 * self.d + 1) // ns) * ns
        z = np.full(64 * k, np.nan)
        self.p = [z.copy() for _ in range(nst)]
        self.c = [z.copy() for _ in range(ns)]
        self.ring = ring
        self.n, self.pre = 0, True
        col = self.w0 + np.arange(64 * k)
        self.col = col
        self.hold = (col == self.left) | (col == self.right)
        if self.cols == 0:
            assert not self.hold.any()
        if self.cols == 2:
            assert not self.hold[:-1].any()
        self.q0 = r0 - self.d - role * nst - 1

    def read(self, G, i):
        if self.role == 0:
            lo, hi = G.rows
            return G.cells(max(lo, min(self.r0 - self.d + i, hi)), self.col)
        if G.made[self.role - 1] < min(i + 1, self.n_steps):
            return None
        row = G.link[self.role - 1][i % LINK].copy()
        G.used[self.role - 1] = i + 1
        return row

    def step(self, G):
        if self.pre:
            row = self.read(G, 0)
            if row is None:
                return False
            self.c[0], self.pre, self.mid = row, False, False
            return True
        n, ns, nst = self.n, self.ns, self.nst
        e = (-n) % ns
        if not self.mid:  # the first sweep, then the next row
            self.sweep(0, e, n)
            self.mid = True
            return True
        if self.mid is True:
            row = self.read(G, n + 1)
            if row is None:
                return False
            self.c[(e + ns - 1) % ns] = row
            for s in range(1, nst):
                self.sweep(s, e, n)
            self.mid = 2
            return True
        out = self.c[(e + nst) % ns]
        if self.role < 3:
            if G.used[self.role] < n + 1 - LINK:
                return False
            G.link[self.role][n % LINK] = out.copy()
            G.made[self.role] = n + 1
        else:
            row = self.r0 - 2 * self.d + n
            if self.r0 <= row < self.r1:
                ok = (self.col >= self.oc0) & (self.col < self.oc1)
                G.store(row, self.col[ok], out[ok])
        self.n, self.mid = n + 1, False
        return True

    def sweep(self, s, e, n):
        ns, k = self.ns, self.k
        S, C, P = self.c[(e + s) % ns], self.c[(e + s + 1) % ns], self.p[s]
        w = np.concatenate(([self.ring], S[:-1]))   # lane 0 keeps its west
        x = np.concatenate((S[1:], [self.ring]))    # lane 63 its east
        t = P + S
        self.p[s] = ((S + w) + x) + C
        new = np.where(self.hold, C, t * 0.2)
        q = self.q0 + n - s
        # one ring row per turn of the row sets
        tA = self.top - self.q0 + self.nst if self.top != NONE else 0
        t0 = n // ns * ns
        special = self.top if t0 < tA else self.bottom
        if q in (self.top, self.bottom):
            assert q == special
        if q == special:
            new = self.a.cells(q, self.col)
        self.c[(e + s + 1) % ns] = new


class Array:
    """A block's array cut from the grid: cells outside it are NaN, so one
    that reaches a result is noticed."""

    def __init__(self, g, rows):
        self.g, self.rows = g, rows

    def cells(self, row, col):
        o = np.full(len(col), np.nan)
        if 0 <= row < self.g.shape[0]:
            ok = (col >= 0) & (col < self.g.shape[1])
            o[ok] = self.g[row, col[ok]]
        return o


class Group(Array):
    def __init__(self, g, rows, out, k, rng):
        super().__init__(g, rows)
        self.out, self.made, self.used = out, [0] * 3, [0] * 3
        self.link = [[np.full(64 * k, np.nan) for _ in range(LINK)]
                     for _ in range(3)]
        self.rng = rng

    def store(self, row, col, v):
        assert np.isnan(self.out[row, col]).all(), "a cell stored twice"
        self.out[row, col] = v

    def run(self, waves):
        left = list(waves)
        stuck = 0
        while left:
            w = left[self.rng.integers(len(left))]
            stuck = 0 if w.step(self) else stuck + 1
            assert stuck < 10000, "the waves wait for each other"
            left = [x for x in left if x.n < x.n_steps]


def block(g, r0, r1, c0, c1, flat, nst, seed):
    """pipe_block: the result of 4 nst sweeps on rows [r0, r1), columns
    [c0, c1) of the grid g (ring included)."""
    H, W, d = g.shape[0] - 2, g.shape[1] - 2, 4 * nst
    out = np.full_like(g, np.nan)
    k = pick_k(c0, c1, 0, W + 1, flat, d)
    wins = windows(c0, c1, 0, W + 1, flat, d, k)
    rng = np.random.default_rng(seed)
    half = (r1 - r0 + 1) // 2
    for i, win in enumerate(wins):
        parts = [(r0, r1)]
        if len(wins) % 2 and i == len(wins) - 1:
            parts = [(r0, r0 + half), (r0 + half, r1)]
        for a, b in parts:
            if a >= b or win[1] >= win[2]:
                continue
            t = 0 if 0 >= a - d else NONE
            u = H + 1 if H + 1 < b + d else NONE
            G = Group(g, (max(0, r0 - d), min(H + 1, r1 - 1 + d)), out, k, rng)
            G.run([Wave(r, nst, G, win, k, a, b, t, u,
                        g[0, 0] if flat else 0.5) for r in range(4)])
    return out[r0:r1, c0:c1]


@pytest.mark.parametrize("nst", [3, 4])
@pytest.mark.parametrize("flat", [True, False])
@pytest.mark.parametrize("W,H", [(16, 16), (17, 40), (160, 17), (190, 20),
                                 (192, 33), (193, 18), (320, 16), (321, 16),
                                 (577, 16), (1121, 16), (1090, 17)])
def test_whole_grids(W, H, flat, nst):
    g = O.init_grid(W, H, seed=W + H)
    if not flat:
        rng = np.random.default_rng(7)
        for edge in (g[0], g[-1], g[:, 0], g[:, -1]):
            edge[:] = rng.random(edge.shape)
    ref = g.copy()
    for _ in range(4 * nst):
        ref = O.step(ref)
    got = block(g, 1, H + 1, 1, W + 1, flat, nst, W)
    assert np.array_equal(got, ref[1:-1, 1:-1])


@pytest.mark.parametrize("c0,c1,r0,r1", [
    (1, 161, 1, 30), (129, 289, 30, 70), (1, 97, 20, 36), (641, 701, 20, 71),
    (97, 700, 1, 17), (1, 701, 30, 47), (545, 701, 1, 71),
    # the ring within reach beyond a thin neighbour
    (385, 690, 20, 60), (545, 689, 33, 70), (17, 690, 5, 9)])
def test_blocks_of_a_grid(c0, c1, r0, r1):
    W, H, nst = 700, 70, 4
    g = O.init_grid(W, H, seed=3)
    ref = g.copy()
    for _ in range(4 * nst):
        ref = O.step(ref)
    got = block(g, r0, r1, c0, c1, True, nst, c0)
    assert np.array_equal(got, ref[r0:r1, c0:c1])


def test_a_short_link_is_noticed(monkeypatch):
    # a producer that never waits for its rows to be used overwrites them
    g = O.init_grid(40, 40, seed=1)
    ref = g.copy()
    for _ in range(16):
        ref = O.step(ref)
    step = Wave.step

    def hasty(self, G):
        if self.role < 3:
            G.used[self.role] = 1 << 20
        return step(self, G)
    monkeypatch.setattr(Wave, "step", hasty)
    got = block(g, 1, 41, 1, 41, True, 4, 5)
    assert not np.array_equal(got, ref[1:-1, 1:-1])
