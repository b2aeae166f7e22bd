"""Low, wide and narrow, tall grids, whose rows several workgroups share (or
several of whose rows one takes): grid, hash, hashes of regions and the exact
residual against the CPU oracle in every form."""
import ctypes as C

import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu

SHAPES = [(200001, 1), (100003, 4), (70001, 17), (1, 50003), (3, 40000),
          (17, 30001), (255, 600), (257, 1500)]


@pytest.mark.parametrize("W,H", SHAPES)
@pytest.mark.parametrize("form", ["plain", "persistent"])
def test_forms(form, W, H):
    import charming_amd as cam
    seed, mode = W + 3 * H, (W + H) & 1
    ref, res = O.jacobi_run(W, H, 5, seed=seed, mode=mode)
    kw = {}
    if form == "persistent":  # chares of a few rows or columns, or one
        kw = dict(chares=(1, 7) if W > 1000 else (7, 1) if H > 1000 else (1, 1))
    with cam.Jacobi2D(W, H, 5, form=form, seed=seed, init_mode=mode, **kw) as j:
        r = j.solve()
        assert np.array_equal(j.grid(), ref)
        assert r.hash == O.grid_hash(ref) and r.residual == res
        # two halves of the columns, then of the rows, add up to the whole
        c, m = W // 2 + 1, H // 2 + 1
        for a, b in (((1, H + 1, 1, c), (1, H + 1, c, W + 1)),
                     ((1, m, 1, W + 1), (m, H + 1, 1, W + 1))):
            assert (j.hash_region(*a) + j.hash_region(*b)) % 2**64 == r.hash


@pytest.mark.parametrize("W,H", SHAPES)
@pytest.mark.parametrize("iters", [3, 4])
def test_noalloc(W, H, iters):
    import torch

    import charming_amd as cam
    fn = cam.jacobi_lib().chm_jacobi2d_solve_noalloc
    fn.argtypes = [C.c_void_p, C.c_int, C.c_int, C.c_int, C.c_void_p, C.c_void_p]
    u0, _ = O.jacobi_run(W, H, 0, seed=W + H)
    ref, res = O.jacobi_run(W, H, iters, seed=W + H)
    P = (W + 18 + 15) // 16 * 16
    buf = torch.zeros(H + 2, P, dtype=torch.float64, device="cuda")
    buf[:, 15:17 + W] = torch.from_numpy(u0).cuda()
    out3 = torch.zeros(3, dtype=torch.int64, device="cuda")
    torch.cuda.synchronize()
    assert fn(buf.data_ptr(), W, H, iters, None, out3.data_ptr()) == 0
    torch.cuda.synchronize()
    assert np.array_equal(buf[:, 15:17 + W].cpu().numpy(), ref)
    words = [int(x) & (2**64 - 1) for x in out3.cpu()]
    assert words == [O.grid_hash(ref), res & (2**64 - 1), res >> 64]


def test_batch():
    import charming_amd as cam
    probs = [dict(width=w, height=h, iters=3 + 6 * i, seed=i, init_mode=i & 1)
             for i, (w, h) in enumerate(SHAPES)]
    for some in (probs[:1], probs):
        out = cam.batch_run(some)
        for i, p in enumerate(some):
            ref, res = O.jacobi_run(p["width"], p["height"], p["iters"],
                                    seed=p["seed"], mode=p["init_mode"])
            assert out["hashes"][i] == O.grid_hash(ref)
            assert out["residuals"][i] == res
