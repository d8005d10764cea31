"""The one-kernel reductions (csrc/reduce.hip) and the CFL loop on the device state.

Sizes at the edges of the reductions' grids: one element (fewer nodes than a block, and more
nodes per element than a block's threads), a node count that is no multiple of a block, and
enough nodes for several iterations per thread.  get_max_dt equals the oracle bit for bit;
sums use another summation order than the oracle's: n FP64 roundings at most, 1e-13 as the
monitor tests allow.  The library's CFL loop equals single steps at the dt it would take, bit
for bit, and reports a non-physical state.
"""
import numpy as np
import pytest

import flouhip as F
import oracle_lib as O
from cases import GAMMA, random_euler_state
from test_gpu_curved import build_curved

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


def build(nd, n, nel):
    b = F.LagrangeBasis("GLL", n)
    std = [None, F.StdSegment, F.StdQuad, F.StdHex][nd](b, F.DGSEMrec(b), nd + 2)
    finish = [1.0, 1.5, 2.0][:nd]
    mesh = F.CartesianMesh(nd, [0.0] * nd, finish, nel)
    mesh.apply_periodicBCs(*[(str(2 * k + 1), str(2 * k + 2)) for k in range(nd)])
    eq = F.EulerEquation(nd, GAMMA)
    op = F.SplitDivOperator(F.KennedyGruber(), F.LxF(F.StdAverage(), 1.0))
    disc = F.MultielementDisc(mesh, std, eq, op)
    orc = O.OracleDisc(nd, n, nel, [0.0] * nd, finish, [1] * nd, O.build_ops(n, "GLL"), O.EQ_EULER, [GAMMA],
                       O.VOL_SPLIT, O.TP_KENNEDY_GRUBER, O.AVG_STD, O.DISS_LXF, 1.0)
    return disc, eq, orc


@pytest.mark.parametrize("nd,n,nel", [(1, 2, [1]), (1, 5, [331]), (2, 6, [1, 1]), (2, 5, [67, 31]), (3, 8, [1, 1, 1]),
                                      (3, 7, [1, 2, 1]), (3, 4, [23, 21, 27])])
def test_reductions_match_oracle(nd, n, nel):
    disc, eq, orc = build(nd, n, nel)
    Q = random_euler_state(orc.coords()[0], nd, seed=5, amp=0.3, smooth=False)
    Qd = disc.to_device(Q)
    for _ in range(2):  # the arrival counter is back at zero
        assert F.get_max_dt(Qd, disc, eq, 0.4) == orc.max_dt(Q, 0.4)
        for v in range(nd + 2):
            scale = np.sum(np.abs(Q[:, v])) / Q.shape[0] * np.prod([1.0, 1.5, 2.0][:nd])
            assert abs(F.integrate(Qd, disc, v) - orc.integrate(Q, v)) <= 1e-13 * scale
        for name, kind in (("kinetic_energy", O.MON_KINETIC_ENERGY), ("entropy", O.MON_ENTROPY)):
            assert F.get_monitor(disc, eq, name)(Qd, disc, eq) == pytest.approx(orc.monitor(Q, kind), rel=1e-13,
                                                                               abs=1e-13)


def test_max_dt_with_element_sizes():
    disc, orc, eq, X, J, std = build_curved(3, 5, 3)  # Δx differs between the elements
    Q = random_euler_state(X, 3, seed=6, amp=0.2)
    assert F.get_max_dt(disc.to_device(Q), disc, eq, 0.4) == orc.max_dt(Q, 0.4)


@pytest.mark.parametrize("solver", [F.SSPRK33, F.CarpenterKennedy2N54])
def test_cfl_loop_takes_the_single_steps(solver):
    disc, eq, orc = build(2, 5, [7, 5])
    Q = random_euler_state(orc.coords()[0], 2, seed=7, amp=0.2)
    loop, steps = disc.to_device(Q), disc.to_device(Q)
    dt0 = F.get_max_dt(loop, disc, eq, 0.2)
    tf = 3.6 * dt0
    F.timeintegrate(loop, disc, eq, solver(), tf, dt=2 * dt0, cfl=0.2)
    t = 0.0
    while t < tf * (1 - 1e-14):
        dt = min(F.get_max_dt(steps, disc, eq, 0.2), min(2 * dt0, tf - t))
        F.timeintegrate(steps, disc, eq, solver(), dt, dt=dt)
        t += dt
    assert torch.equal(loop, steps)


def test_cfl_loop_reports_a_non_physical_state():
    disc, eq, orc = build(2, 5, [4, 4])
    Q = random_euler_state(orc.coords()[0], 2, seed=8, amp=0.1)
    Q[17, 3] = -1.0  # negative pressure
    with pytest.raises(F.DomainError):
        F.timeintegrate(disc.to_device(Q), disc, eq, F.SSPRK33(), 1e-2, dt=1e-3, cfl=0.2)
    disc.check()  # the flag is clear again
