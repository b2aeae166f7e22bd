"""Device memory kept between batches and servers: a kept block that held
something else changes no result, and what is kept goes back on request."""
import pytest
import torch

from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _probs(n, lo, seed):
    return [dict(width=lo + 37 * i, height=lo + 11 * (n - i), iters=9 + 5 * i,
                 seed=seed + i) for i in range(n)]


def _expect(probs):
    out = []
    for p in probs:
        g, res = O.jacobi_run(p["width"], p["height"], p["iters"],
                              seed=p["seed"])
        out.append((O.grid_hash(g), res))
    return out


def _run(cam, probs):
    r = cam.batch_run(probs)
    return list(zip(r["hashes"], r["residuals"]))


def test_reused_blocks_and_release():
    import charming_amd as cam
    small, large = _probs(3, 40, 1), _probs(5, 300, 50)
    ref_s, ref_l = _expect(small), _expect(large)
    for _ in range(2):
        assert _run(cam, large) == ref_l
        assert _run(cam, small) == ref_s  # in blocks that held other data
        with cam.Server("engine", budget_bytes=1 << 30) as srv:
            assert srv.submit(small[2]) is not None
    torch.cuda.synchronize()
    before = torch.cuda.mem_get_info()[0]
    cam.release_memory()
    after = torch.cuda.mem_get_info()[0]
    assert after >= before + (1 << 30)  # the server's pool at least
    assert _run(cam, large) == ref_l
