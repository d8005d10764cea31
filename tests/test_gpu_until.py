"""The library's loop to a final time (flou_hip_timeintegrate_until, timeintegrate(.., cfl=..)).

Runs that end below zero, time steps that stop advancing the time, non-physical states met on the way,
interrupts.  Steps of 1/64 (exact in the time's arithmetic) so that a run and its shifted copy take the same
ones, bit for bit.
"""
import ctypes
import signal
import time

import numpy as np
import pytest

import flouhip as F
from cases import random_euler_state
from flouhip import _capi as C
from test_gpu_reductions import build

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


def start(amp=0.01):
    disc, eq, orc = build(2, 3, [2, 2])
    Q = random_euler_state(orc.coords()[0], 2, seed=3, amp=amp)
    return disc, eq, Q


@pytest.mark.parametrize("solver", [F.SSPRK33, F.CarpenterKennedy2N54])
@pytest.mark.parametrize("t0,tf", [(-1.0, -0.5), (-0.25, 0.25), (-0.5, 0.0)])
def test_final_times_of_any_sign(t0, tf, solver):
    disc, eq, Q = start()
    a, b = disc.to_device(Q), disc.to_device(Q)
    assert F.get_max_dt(a, disc, eq, 100.0) > 1 / 64
    F.timeintegrate(a, disc, eq, solver(), tf, dt=1 / 64, cfl=100.0, t0=t0)
    F.timeintegrate(b, disc, eq, solver(), tf - t0, dt=1 / 64, cfl=100.0)
    assert torch.equal(a, b) and torch.isfinite(a).all()


def test_step_that_no_longer_advances():
    disc, eq, Q = start()
    Qd = disc.to_device(Q)
    Qd[3, 5] = float("inf")  # an unbounded wave speed: the CFL step is 0
    with pytest.raises(F.DomainError, match="advance"):
        F.timeintegrate(Qd, disc, eq, F.SSPRK33(), 1.0, dt=1e-2, cfl=0.2)
    Qd = disc.to_device(Q)
    with pytest.raises(F.DomainError, match="advance"):  # 1 + 1e-17 == 1
        F.timeintegrate(Qd, disc, eq, F.SSPRK33(), 2.0, dt=1e-17, cfl=0.2, t0=1.0)
    assert np.array_equal(disc.to_host(Qd), Q)
    disc.check()


@pytest.mark.parametrize("cfl", [0.0, 0.2])
def test_no_step_after_a_non_physical_state(cfl):
    """The step that meets the state is the last: t stays where it ended."""
    disc, eq, Q = start()
    Q[7, 3] = -1.0  # negative pressure
    Qd = disc.to_device(Q)
    t = ctypes.c_double(0.0)
    rc = C.lib.flou_hip_timeintegrate_until(disc.h, C.SSPRK33, disc._dptr(Qd), 1e-4, 1.0, cfl, ctypes.byref(t))
    assert rc == C.EDOMAIN and 0 < t.value <= 1e-4
    disc.check()


class Alarm(Exception):
    pass


def test_a_run_can_be_interrupted():
    """A signal ends a run of many steps soon, and leaves a state between two steps."""
    disc, eq, Q = start()
    Qd = disc.to_device(Q)

    def ring(*_):
        raise Alarm

    old = signal.signal(signal.SIGALRM, ring)
    signal.setitimer(signal.ITIMER_REAL, 0.5)
    tic = time.perf_counter()
    try:
        with pytest.raises(Alarm):
            # 200,000 steps, some seconds
            F.timeintegrate(Qd, disc, eq, F.CarpenterKennedy2N54(), 0.2, dt=1e-6, cfl=0.2)
    finally:
        signal.setitimer(signal.ITIMER_REAL, 0)
        signal.signal(signal.SIGALRM, old)
    assert time.perf_counter() - tic < 2.0
    assert torch.isfinite(Qd).all() and F.get_max_dt(Qd, disc, eq, 0.2) > 1e-6


@pytest.mark.parametrize("scheme", [C.SSPRK33, C.CK2N54])
def test_slices_take_the_same_steps(scheme):
    disc, eq, Q = start(0.1)
    a, b = disc.to_device(Q), disc.to_device(Q)
    tf, dt = 7.3e-3, 1e-3
    ta, tb = ctypes.c_double(0.0), ctypes.c_double(0.0)
    assert C.lib.flou_hip_timeintegrate_until(disc.h, scheme, disc._dptr(a), dt, tf, 0.1, ctypes.byref(ta)) == C.OK
    calls, before = 0, -1.0
    while tb.value > before:
        before = tb.value
        assert C.lib.flou_hip_timeintegrate_slice(disc.h, scheme, disc._dptr(b), dt, tf, 0.1, 0.0, ctypes.byref(tb)) == C.OK
        calls += 1
    assert calls > 3 and ta.value == tb.value and torch.equal(a, b)
