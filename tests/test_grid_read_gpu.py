"""Reading the grid back, which goes in pieces of whole rows: one piece, an
odd number of pieces with a short last one, rows longer than a piece."""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("W,H,chares,mode", [
    (1, 1, (1, 1), 0), (254, 510, (3, 2), 1), (254, 511, (2, 3), 0),
    (1021, 300, (7, 5), 0), (140001, 5, (1, 9), 0), (131070, 3, (1, 1), 1)])
@pytest.mark.parametrize("form", ["plain", "persistent"])
def test_pieces(form, W, H, chares, mode):
    import charming_amd as cam
    kw = dict(chares=chares) if form == "persistent" else {}
    u0, _ = O.jacobi_run(W, H, 0, seed=W + H, mode=mode)
    ref, _ = O.jacobi_run(W, H, 2, seed=W + H, mode=mode)
    with cam.Jacobi2D(W, H, 2, form=form, seed=W + H, init_mode=mode,
                      **kw) as j:
        assert np.array_equal(j.grid(), u0)
        j.solve()
        assert np.array_equal(j.grid(), ref)
        assert np.array_equal(j.grid(), ref)
