"""Broadcasts (invoke_all) of small payloads, which the sender's lanes write
side by side: thread 0's buffer alone counts, also where it lies in that
thread's own memory (charming_amd/csrc/examples/broadcast.hip)."""
import ctypes
import os
import re

import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "charming_amd", "lib")
_loaded = {}


def _run(capfd, args, **env):
    if not _loaded:
        rt = ctypes.CDLL(os.path.join(LIB, "libcharming_amd.so"),
                         mode=ctypes.RTLD_GLOBAL)
        rt.chm_main.argtypes = [ctypes.c_int, ctypes.POINTER(ctypes.c_char_p)]
        rt.chm_select_program.argtypes = [ctypes.c_char_p]
        _loaded["rt"] = rt
        _loaded["prog"] = ctypes.CDLL(os.path.join(LIB, "libchm_broadcast.so"))
    rt = _loaded["rt"]
    assert rt.chm_select_program(b"broadcast.hip") == 0
    env = dict(CHM_TIMEOUT_S=20, CHM_STATS=1, **env)
    saved = {k: os.environ.get(k) for k in env}
    argv = [b"broadcast"] + [str(a).encode() for a in args]
    print(f"running broadcast {args} {env}", flush=True)
    capfd.readouterr()
    os.environ.update({k: str(v) for k, v in env.items()})
    try:
        rc = rt.chm_main(len(argv), (ctypes.c_char_p * len(argv))(*argv))
    finally:
        for k, v in saved.items():
            if v is None:
                del os.environ[k]
            else:
                os.environ[k] = v
    out, err = capfd.readouterr()
    stats = dict(re.findall(r"(\w+)=([\d.]+)", out.split("[STATS]")[-1]))
    return rc, out, err, stats


@pytest.mark.parametrize("pes,count,nbytes", [
    (5, 3, 1), (5, 3, 4), (65, 2, 8), (200, 2, 24), (7, 40, 63), (130, 3, 64),
    (3, 2, 0)])
def test_thread_zeros_payload_counts(capfd, pes, count, nbytes):
    rc, out, err, st = _run(capfd, ["word", count, nbytes], CHM_N_PES=pes)
    assert rc == 0, err[-2000:]
    assert (f"{count} payloads of {nbytes} bytes to {pes} chares, 0 wrong"
            in out), out[-2000:]
    assert int(st["delivered"]) == 1 + pes * count + pes


RING = dict(CHM_RING_BYTES=65536, CHM_MAX_MSG_BYTES=32768)


def _still_works(capfd):
    rc, out, err, st = _run(capfd, ["word", 2, 12], CHM_N_PES=9)
    assert rc == 0 and "12 bytes to 9 chares, 0 wrong" in out, err[-2000:]


@pytest.mark.parametrize("pes,nbytes", [(3, 8), (70, 24)])
def test_lanes_wait_for_room(capfd, pes, nbytes):
    # chare 1's PE is busy and three quarters of its inbox taken: about 270 of
    # the 400 broadcasts fit, each later one waits for its one late lane
    rc, out, err, st = _run(capfd, ["full", 400, nbytes], CHM_N_PES=pes, **RING)
    assert rc == 0, err[-2000:]
    assert f"400 payloads of {nbytes} bytes to {pes} chares, 0 wrong" in out
    assert int(st["send_spins"]) > 0


def test_waiting_lane_gives_up_at_the_spin_limit(capfd):
    rc, out, err, st = _run(capfd, ["full", 400, 8], CHM_N_PES=70,
                            CHM_SPIN_LIMIT=2000, **RING)
    assert rc == 1
    assert "device error 8 (send spin limit reached" in err, err[-2000:]
    assert int(st["send_spins"]) >= 2000
    _still_works(capfd)


def test_own_inbox_full_fails_at_once(capfd):
    # 1024 messages of 64 bytes fill the sender's own ring
    rc, out, err, st = _run(capfd, ["self", 1100, 8], CHM_N_PES=3, **RING)
    assert rc == 1 and st["error"] == "2", err[-2000:]
    _still_works(capfd)
