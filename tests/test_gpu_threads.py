"""GPU: other Python threads run while the binding launches (a launch blocks on a full queue)."""

import sys
import threading

import pytest
import torch

from ssm_scan import _abi
from ssm_scan.hip_scan import scan_forward

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("entry", ["scan", "norm"])
def test_launches_release_the_interpreter_lock(dev, entry):
    """With forced switches off, a waiting thread gets in only where the launching thread lets go of the
    lock itself: during its launches.  (Freeing a tensor may let go of it too: all results are kept.)"""
    x, v = torch.randn(1, 8, 64, device=dev), torch.randn(64, device=dev)
    A, Bm = -torch.rand(64, 8, device=dev), torch.randn(1, 8, 8, device=dev)
    host = _abi.host()
    call = {"scan": lambda: scan_forward(x, x, A, Bm, Bm, None, None, None, None, 0, False),
            "norm": lambda: host.norm_forward(x, v, 1e-5)}[entry]
    call()
    torch.cuda.synchronize()
    go, ran, kept = threading.Event(), [], []
    t = threading.Thread(target=lambda: (go.wait(), ran.append(True)))
    t.start()
    interval = sys.getswitchinterval()
    sys.setswitchinterval(1000.0)
    try:
        go.set()
        for _ in range(5000):
            kept.append(call())
            if ran:
                break
        got_in = bool(ran)
    finally:
        sys.setswitchinterval(interval)
        t.join()
        torch.cuda.synchronize()
    assert got_in
