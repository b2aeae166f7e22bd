"""Kept device memory beside a running server: giving memory back waits for
every kernel of the device, and a server's engine ends only when its owner
stops it, so nothing may be given back while it runs."""
import threading
import time

import pytest
import torch

pytestmark = pytest.mark.gpu


def test_release_beside_a_server_returns():
    import charming_amd as cam
    probs = [dict(width=700, height=600, iters=20, seed=i) for i in range(9)]
    cam.batch_run(probs)  # (the first calls load code and take scratch)
    with cam.Server("engine", budget_bytes=1 << 28):
        pass
    cam.release_memory()
    torch.cuda.synchronize()
    before = torch.cuda.mem_get_info()[0]
    cam.batch_run(probs)
    kept = before - torch.cuda.mem_get_info()[0]
    assert kept > 9 * 3 * 700 * 600 * 8
    srv = cam.Server("engine", budget_bytes=1 << 28)
    # (the engine ends in any case, so that a wait for it would show as time)
    t0, guard = time.time(), threading.Timer(20, srv.stop)
    guard.start()
    try:
        # the batch's memory went back before the engine started
        used = before - torch.cuda.mem_get_info()[0]
        assert used < kept + (1 << 28) - 9 * 3 * 700 * 600 * 8
        cam.release_memory()
        t = srv.submit(probs[0])
        while not srv.poll():
            pass
        assert t is not None and time.time() - t0 < 10
    finally:
        guard.cancel()
        srv.stop()
    cam.release_memory()
