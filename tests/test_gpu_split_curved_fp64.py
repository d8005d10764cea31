"""The FP64 split-form kernel of curved elements (csrc/rhs_split.hip) against the oracle.

Every node count 2..8 in 2-D and 3-D, partial last blocks and spare lanes, all three two-point
fluxes, with and without LxF, walls and outflow on one axis, smooth states and states on the
logarithm's branch.  Both sides round some 8 operations per flux over Σ_j |D_ij| ~ n², against
rates of 0.3 |F| or more: 8 · 2^-53 n² / 0.3 < 4e-15 n² of the largest value (n no less than 4:
the faces' share).
"""
import numpy as np
import pytest

import flouhip as F
import oracle_lib as O
from cases import GAMMA, random_euler_state
from flouhip import mesh as M
from test_gpu_curved import TP, rel_err, warp

pytestmark = pytest.mark.gpu
pytest.importorskip("torch")

NEL = {2: (5, 3), 3: (3, 2, 2)}


def build(nd, n, tp, lxf, walls, nel=None):
    nel = nel or NEL[nd]
    b = F.LagrangeBasis("GLL", n)
    std = [None, None, F.StdQuad, F.StdHex][nd](b, F.DGSEMrec(b), nd + 2)
    mesh = F.CartesianMesh(nd, (0.0,) * nd, (1.0,) * nd, nel)
    mesh.apply_periodicBCs(*[(str(2 * k + 1), str(2 * k + 2)) for k in range(1 if walls else 0, nd)])
    mesh.apply_mapping(warp)
    bcs = {"1": F.EulerSlipBC(), "2": F.EulerOutflowBC()} if walls else {}
    eq = F.EulerEquation(nd, GAMMA)
    surf = F.LxF(F.StdAverage(), 0.8) if lxf else F.StdAverage()
    disc = F.MultielementDisc(mesh, std, eq, F.SplitDivOperator(TP[tp][0](), surf), bcs)
    J, met, ev, fr, fj = M.curved_geometry(mesh, std)
    orc = O.OracleDisc(nd, n, list(nel), [0.0] * nd, [1.0] * nd, [0 if walls and k == 0 else 1 for k in range(nd)],
                       O.build_ops(n, "GLL"), O.EQ_EULER, [GAMMA], O.VOL_SPLIT, TP[tp][1], O.AVG_STD,
                       O.DISS_LXF if lxf else O.DISS_NONE, 0.8 if lxf else 1.0)
    orc.set_curved(met, J, fr.reshape(-1), fj, ev)
    if walls:
        orc.set_bc(0, O.BC_SLIP)
        orc.set_bc(1, O.BC_OUTFLOW)
    return disc, eq, orc, mesh.node_coords(std)


@pytest.mark.parametrize("tp", ["std", "ch", "kg"])
@pytest.mark.parametrize("nd,n", [(nd, n) for nd in (2, 3) for n in range(2, 9)])
def test_rhs_matches_oracle(nd, n, tp):
    disc, eq, orc, X = build(nd, n, tp, n != 5, n in (2, 4, 7))
    dQ = disc.new_state()
    for smooth in (True, False):
        Q = random_euler_state(X, nd, seed=n, amp=0.3, smooth=smooth)
        if not smooth:
            Q[::3] *= 2.5
        F.rhs_(dQ, disc.to_device(Q), F.EquationConfig(disc, eq))
        disc.check()
        assert rel_err(disc.to_host(dQ), orc.rhs(Q)) <= 4e-15 * max(n, 4) ** 2


@pytest.mark.parametrize("solver,scheme", [(F.SSPRK33, O.RK_SSPRK33), (F.CarpenterKennedy2N54, O.RK_CK2N54)])
def test_steps_match_oracle(solver, scheme):
    disc, eq, orc, X = build(3, 5, "ch", True, False)
    Q = random_euler_state(X, 3, seed=3, amp=0.2)
    Qd = disc.to_device(Q)
    F.timeintegrate(Qd, disc, eq, solver(), 3e-4, dt=1e-4)
    assert rel_err(disc.to_host(Qd), orc.rk_run(scheme, Q, 1e-4, 3)) <= 1e-13
