"""The FP64 split-form kernel of axis-aligned elements (csrc/rhs_split.hip) against the oracle.

Sizes at the edges of its blocks: every node count 2..8 in 1-D to 3-D, element counts that
leave the last block partial (and one element), spare lanes, one and several face rounds per
thread, walls on one axis.  It computes the plain kernel's values in the same order, so
Kennedy-Gruber and StdAverage must equal the oracle bit for bit; Chandrasekhar evaluates
logarithms, whose device and host libraries may differ by an ulp (the bound the parity tests
use for it).
"""
import numpy as np
import pytest

import flouhip as F
import oracle_lib as O
from cases import GAMMA, random_euler_state

pytestmark = pytest.mark.gpu
pytest.importorskip("torch")

TP = {"std": (F.StdAverage, O.TP_STDAVG), "ch": (F.ChandrasekharAverage, O.TP_CHANDRASEKHAR),
      "kg": (F.KennedyGruber, O.TP_KENNEDY_GRUBER)}
NEL = {1: [37], 2: [5, 3], 3: [3, 2, 2]}


def build(nd, n, nel, tp, lxf, walls):
    finish = [1.0, 1.5, 2.0][:nd]
    b = F.LagrangeBasis("GLL", n)
    std = [None, F.StdSegment, F.StdQuad, F.StdHex][nd](b, F.DGSEMrec(b), nd + 2)
    mesh = F.CartesianMesh(nd, [0.0] * nd, finish, nel)
    mesh.apply_periodicBCs(*[(str(2 * k + 1), str(2 * k + 2)) for k in range(0 if not walls else 1, nd)])
    bcs = {"1": F.EulerSlipBC(), "2": F.EulerOutflowBC()} if walls else {}
    surf = F.LxF(F.StdAverage(), 0.8) if lxf else F.StdAverage()
    eq = F.EulerEquation(nd, GAMMA)
    disc = F.MultielementDisc(mesh, std, eq, F.SplitDivOperator(TP[tp][0](), surf), bcs)
    orc = O.OracleDisc(nd, n, nel, [0.0] * nd, finish, [0 if walls and k == 0 else 1 for k in range(nd)],
                       O.build_ops(n, "GLL"), O.EQ_EULER, [GAMMA], O.VOL_SPLIT, TP[tp][1], O.AVG_STD,
                       O.DISS_LXF if lxf else O.DISS_NONE, 0.8 if lxf else 1.0)
    if walls:
        orc.set_bc(0, O.BC_SLIP)
        orc.set_bc(1, O.BC_OUTFLOW)
    return disc, eq, orc


def check(got, ref, tp):
    same = np.mean(got == ref)
    err = np.max(np.abs(got - ref) / np.max(np.abs(ref), axis=0))
    assert same == 1.0 if tp != "ch" else (same >= 0.9 and err <= 1e-13), (same, err)


@pytest.mark.parametrize("tp", ["std", "ch", "kg"])
@pytest.mark.parametrize("nd,n", [(nd, n) for nd in (1, 2, 3) for n in range(2, 9)])
def test_rhs_matches_oracle(nd, n, tp):
    disc, eq, orc = build(nd, n, NEL[nd], tp, n % 2 == 0, n in (2, 5, 6))
    Q = random_euler_state(orc.coords()[0], nd, seed=n, amp=0.3, smooth=n % 2 == 1)
    dQ = disc.new_state()
    F.rhs_(dQ, disc.to_device(Q), F.EquationConfig(disc, eq))
    disc.check()
    check(disc.to_host(dQ), orc.rhs(Q), tp)


@pytest.mark.parametrize("solver,scheme", [(F.SSPRK33, O.RK_SSPRK33), (F.CarpenterKennedy2N54, O.RK_CK2N54)])
def test_steps_match_oracle(solver, scheme):
    disc, eq, orc = build(3, 6, [1, 2, 1], "kg", True, False)
    Q = random_euler_state(orc.coords()[0], 3, seed=3, amp=0.2)
    Qd = disc.to_device(Q)
    F.timeintegrate(Qd, disc, eq, solver(), 3e-3, dt=1e-3)
    check(disc.to_host(Qd), orc.rk_run(scheme, Q, 1e-3, 3), "kg")
