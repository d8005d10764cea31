"""The strong-form kernel of axis-aligned elements (csrc/rhs_strong.hip) against the oracle.

Every node count 2..8 in 1-D to 3-D, partial last blocks, spare lanes, one to three face nodes
per thread, own traces from LDS and from memory, walls, inflow and Dirichlet ends, Euler and
advection.  FP64 computes the plain kernel's values in the same order: bit for bit.  FP32
takes some 8 roundings of 2^-24 per flux, 3n terms of a node's sum with |D| ~ n²/2 and rates of
0.3 |F| or more: 40 n³ 2^-24, bounded by n³ 2^-18 of the largest value.
"""
import numpy as np
import pytest

import flouhip as F
import oracle_lib as O
from cases import GAMMA, random_euler_state

pytestmark = pytest.mark.gpu
pytest.importorskip("torch")

NEL = {1: [301], 2: [23, 9], 3: [5, 3, 4]}
INFLOW = {1: [1.1, 0.3, 2.5], 2: [1.1, 0.3, -0.1, 2.5], 3: [1.1, 0.3, -0.1, 0.2, 2.5]}


def build(nd, n, adv, lxf, ends, precision):
    finish, nel, nv = [1.0, 1.5, 2.0][:nd], NEL[nd], 1 if adv else nd + 2
    b = F.LagrangeBasis("GLL", n)
    std = [None, F.StdSegment, F.StdQuad, F.StdHex][nd](b, F.DGSEMrec(b), nv)
    mesh = F.CartesianMesh(nd, [0.0] * nd, finish, nel)
    mesh.apply_periodicBCs(*[(str(2 * k + 1), str(2 * k + 2)) for k in range(1 if ends else 0, nd)])
    state = [0.7] if adv else INFLOW[nd]
    first, code = {"": (None, None), "inflow": (F.EulerInflowBC(state) if not adv else None, O.BC_INFLOW),
                   "slip": (F.EulerSlipBC(), O.BC_SLIP)}[ends]
    bcs = {"1": first, "2": F.EulerOutflowBC()} if ends else {}
    surf = F.LxF(F.StdAverage(), 0.8) if lxf else F.StdAverage()
    vel = [3.0, 4.0, -2.0][:nd]
    eq = F.LinearAdvection(*vel) if adv else F.EulerEquation(nd, GAMMA)
    disc = F.MultielementDisc(mesh, std, eq, F.StrongDivOperator(surf), bcs, precision=precision)
    orc = O.OracleDisc(nd, n, nel, [0.0] * nd, finish, [0 if ends and k == 0 else 1 for k in range(nd)],
                       O.build_ops(n, "GLL"), O.EQ_ADVECTION if adv else O.EQ_EULER, vel if adv else [GAMMA],
                       O.VOL_STRONG, O.TP_STDAVG, O.AVG_STD, O.DISS_LXF if lxf else O.DISS_NONE, 0.8 if lxf else 1.0)
    if ends:
        orc.set_bc(0, code, np.array(state)) if ends == "inflow" else orc.set_bc(0, code)
        orc.set_bc(1, O.BC_OUTFLOW)
    return disc, eq, orc


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("ends", ["", "inflow", "slip"])
@pytest.mark.parametrize("nd,n", [(nd, n) for nd in (1, 2, 3) for n in range(2, 9)])
def test_euler_matches_oracle(nd, n, ends, precision):
    disc, eq, orc = build(nd, n, False, n % 2 == 0 or ends == "slip", ends, precision)
    Q = random_euler_state(orc.coords()[0], nd, seed=n, amp=0.3, smooth=n % 2 == 1)
    if precision == "fp32":
        Q = np.asfortranarray(Q.astype(np.float32).astype(np.float64))
    dQ = disc.new_state()
    F.rhs_(dQ, disc.to_device(Q), F.EquationConfig(disc, eq))
    disc.check()
    got, ref = disc.to_host(dQ).astype(np.float64), orc.rhs(Q)
    if precision == "fp64":
        assert np.array_equal(got, ref)
    else:
        assert np.max(np.abs(got - ref) / np.max(np.abs(ref))) <= n ** 3 * 2.0 ** -18


@pytest.mark.parametrize("nd,n", [(nd, n) for nd in (1, 2, 3) for n in range(2, 9)])
def test_advection_steps_match_oracle(nd, n):
    disc, eq, orc = build(nd, n, True, n != 4, "", "fp64")
    Q = np.asfortranarray(np.random.default_rng(n).standard_normal((orc.coords()[0].shape[0], 1)))
    Qd = disc.to_device(Q)
    solver, scheme = (F.SSPRK33, O.RK_SSPRK33) if n % 2 else (F.CarpenterKennedy2N54, O.RK_CK2N54)
    F.timeintegrate(Qd, disc, eq, solver(), 3e-4, dt=1e-4)
    assert np.array_equal(disc.to_host(Qd), orc.rk_run(scheme, Q, 1e-4, 3))
