"""flou_hip_check and the time loops synchronise the handle's stream: nothing is pending on return.

The error flag reaches the host in pinned memory a few microseconds before the stream reports
its end; without the wait the stream is still busy in most of the repetitions.
"""
import ctypes

import pytest

import flouhip as F
from cases import random_euler_state
from flouhip import _capi as C
from test_gpu_reductions import build

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


def test_nothing_is_pending_on_return():
    disc, eq, orc = build(3, 4, [5, 4, 3])
    Qd = disc.to_device(random_euler_state(orc.coords()[0], 3, seed=2, amp=0.05))
    dQ = disc.new_state()
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        torch.cuda.synchronize()
        for _ in range(200):
            F.rhs_(dQ, Qd, F.EquationConfig(disc, eq))
            disc.check()
            assert s.query()
        t = ctypes.c_double(0.0)
        for _ in range(50):
            assert C.lib.flou_hip_timeintegrate(disc.h, C.SSPRK33, disc._dptr(Qd), 1e-6, 2, 0.0, ctypes.byref(t)) == C.OK
            assert s.query()
            assert C.lib.flou_hip_timeintegrate_until(disc.h, C.CK2N54, disc._dptr(Qd), 1e-6, t.value + 3e-6, 0.2,
                                                      ctypes.byref(t)) == C.OK
            assert s.query()
