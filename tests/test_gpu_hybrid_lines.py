"""The hybrid kernel of small axis-aligned meshes (csrc/rhs_hybrid.hip) against the oracle.

Every node count 2..8 in 1-D and 2-D with partial last blocks, walls and outflow on one axis,
all surface fluxes, and meshes of exactly the most blocks that take it and of one element more
(the other kernel).  Bound 1e-12 of the largest value, as the hybrid form's other tests.
"""
import numpy as np
import pytest

import flouhip as F
import oracle_lib as O
from cases import GAMMA, random_euler_state
from test_gpu_hybrid import TP, surface

pytestmark = pytest.mark.gpu
pytest.importorskip("torch")

SURF = [(O.AVG_STD, O.DISS_LXF), (O.AVG_CHANDRASEKHAR, O.DISS_MATRIX), (O.AVG_STD, O.DISS_MATRIX),
        (O.AVG_STD, O.DISS_NONE), (O.AVG_CHANDRASEKHAR, O.DISS_SCALAR)]


def check(nd, n, nel, tp, savg, sdiss, walls):
    finish = [1.0, 1.5][:nd]
    b = F.LagrangeBasis("GLL", n)
    std = [None, F.StdSegment, F.StdQuad][nd](b, F.DGSEMrec(b), nd + 2)
    mesh = F.CartesianMesh(nd, [0.0] * nd, finish, nel)
    mesh.apply_periodicBCs(*[(str(2 * k + 1), str(2 * k + 2)) for k in range(1 if walls else 0, nd)])
    bcs = {"1": F.EulerSlipBC(), "2": F.EulerOutflowBC()} if walls else {}
    eq = F.EulerEquation(nd, GAMMA)
    disc = F.MultielementDisc(mesh, std, eq, F.HybridDivOperator(TP[tp](), surface(savg, sdiss), 0.5), bcs)
    orc = O.OracleDisc(nd, n, nel, [0.0] * nd, finish, [0 if walls and k == 0 else 1 for k in range(nd)],
                       O.build_ops(n, "GLL"), O.EQ_EULER, [GAMMA], O.VOL_HYBRID, tp, savg, sdiss, 1.0)
    orc.set_blend(0.5)
    if walls:
        orc.set_bc(0, O.BC_SLIP)
        orc.set_bc(1, O.BC_OUTFLOW)
    Q = random_euler_state(orc.coords()[0], nd, seed=n, amp=0.3, smooth=False)
    dQ = disc.new_state()
    F.rhs_(dQ, disc.to_device(Q), F.EquationConfig(disc, eq))
    disc.check()
    ref = orc.rhs(Q)
    assert np.max(np.abs(disc.to_host(dQ) - ref) / np.max(np.abs(ref), axis=0)) <= 1e-12


@pytest.mark.parametrize("surf", range(len(SURF)))
@pytest.mark.parametrize("nd,n", [(nd, n) for nd in (1, 2) for n in range(2, 9)])
def test_small_meshes(nd, n, surf):
    tp = (O.TP_CHANDRASEKHAR, O.TP_KENNEDY_GRUBER, O.TP_STDAVG)[(n + surf) % 3]
    check(nd, n, [67] if nd == 1 else [7, 5], tp, *SURF[surf], walls=(n + surf) % 2 == 0)


@pytest.mark.parametrize("extra", [0, 1])
@pytest.mark.parametrize("n", [4, 6, 8])
def test_most_blocks(n, extra):
    epb = 128 // (n * (n + 1))
    check(2, n, [32 * epb + extra, 24], O.TP_CHANDRASEKHAR, O.AVG_CHANDRASEKHAR, O.DISS_MATRIX, False)
