"""When kept device memory goes back: before a server's engine starts and not
while it runs (giving memory back waits for every kernel of the device, and
that engine ends only when its owner stops it), and by itself once it has not
been used for a while."""
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


def test_unused_memory_goes_back_by_itself():
    # after ten seconds, here while another thread captures a graph, which
    # the free must not end
    import charming_amd as cam
    probs = [dict(width=1500, height=1400, iters=20, seed=i) for i in range(9)]
    arena = 9 * 3 * 1500 * 1400 * 8
    want = cam.batch_run(probs)["hashes"]
    cam.release_memory()
    x = torch.zeros(1000, device="cuda")
    torch.cuda.synchronize()
    before = torch.cuda.mem_get_info()[0]
    assert cam.batch_run(probs)["hashes"] == want
    assert before - torch.cuda.mem_get_info()[0] >= arena
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        x.add_(1)
        time.sleep(13)
    for k in range(3):
        graph.replay()
        torch.cuda.synchronize()
        assert bool((x == k + 1).all())
    assert before - torch.cuda.mem_get_info()[0] < arena
    assert cam.batch_run(probs)["hashes"] == want


def test_kept_memory_counts_as_free():
    # a budget sized from the free memory is the same before and after a batch
    import charming_amd as cam
    probs = [dict(width=1500, height=1400, iters=20, seed=i) for i in range(9)]
    arena = 9 * 3 * 1500 * 1400 * 8
    cam.batch_run(probs)
    cam.release_memory()
    before = cam.device_memory()
    cam.batch_run(probs)
    after = cam.device_memory()
    assert before[1] == after[1] and abs(after[0] - before[0]) < arena // 2
    assert torch.cuda.mem_get_info()[0] <= after[0] - arena
    cam.release_memory()
