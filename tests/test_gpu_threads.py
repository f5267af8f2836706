"""The native host side gives up the interpreter lock while it allocates, launches and multiplies: other Python threads run."""
import sys
import threading
import time

import pytest
import torch

from oracle.timemix_restated import ChannelMix6, TimeMix6

pytestmark = pytest.mark.gpu


def _turns_of_another_thread(call, n):
    """how often another thread gets its turn inside `call`, with the interpreter's own switching switched off (so that it runs
    only where this thread gives the lock up)"""
    turns, stop, previous = [0], threading.Event(), sys.getswitchinterval()

    def count():
        while not stop.is_set():
            turns[0] += 1
            time.sleep(0)          # gives the lock back
    thread = threading.Thread(target=count, daemon=True)
    call()
    torch.cuda.synchronize()
    sys.setswitchinterval(100)
    try:
        thread.start()
        got = 0
        for _ in range(n):
            before = turns[0]
            call()
            got += turns[0] - before
    finally:
        stop.set()
        sys.setswitchinterval(previous)
        thread.join()
    torch.cuda.synchronize()
    return got


def _cases():
    from rwkv_wkv_hip import _lib
    H, T = 4, 300
    C = 64 * H
    host = _lib.host()
    bf = lambda *s: torch.randn(*s, device="cuda", dtype=torch.bfloat16)
    tm, cm = TimeMix6(C, H, seed=1).cuda().bfloat16(), ChannelMix6(C, 4 * C, seed=2).cuda().bfloat16()
    x, shift, state = bf(1, T, C), bf(1, C), torch.randn(1, H, 64, 64, device="cuda")
    r, k, v, w = bf(1, T, C), bf(1, T, C), bf(1, T, C), bf(1, T, C)
    u = torch.randn(H, 64, device="cuda")
    v4 = [torch.randn(C, device="cuda"), torch.randn(C, device="cuda"), k, v, torch.zeros(1, C, 3, device="cuda")]
    return {"timemix": lambda: host.timemix(6, 0, tm, x, (shift, state)), "channelmix": lambda: host.channelmix(6, cm, x, shift),
            "wkv56": lambda: host.wkv56(6, 0, False, 1, T, C, H, r, k, v, w, u, state), "wkv4": lambda: host.wkv4(*v4),
            "forward56": lambda: host.forward56(6, 0, 1, T, C, H, r, k, v, w, u, state, None)}


@pytest.mark.parametrize("name", ["timemix", "channelmix", "wkv56", "wkv4", "forward56"])
def test_other_threads_run_meanwhile(name):
    call = _cases()[name]
    assert call() is not None
    assert _turns_of_another_thread(call, 1000) > 0
