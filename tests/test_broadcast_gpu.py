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
