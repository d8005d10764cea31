"""The 1-D FP64 split-form kernel (csrc/rhs_split.hip, k_split_1d) against the oracle.

Every node count 2..8, every surface flux, Dirichlet-like inflow, slip and outflow ends, partial last
blocks and one element, and meshes of exactly the most blocks that take it and of one element more.
The plain kernel's values in the same order: Kennedy-Gruber and StdAverage with LxF bit for bit,
otherwise logarithms, square roots and exponents of the device library within 1e-12.
"""
import numpy as np
import pytest

import flouhip as F
import oracle_lib as O
from cases import GAMMA, random_euler_state
from test_gpu_hybrid import TP, surface

pytestmark = pytest.mark.gpu
pytest.importorskip("torch")

SURF = [(O.AVG_STD, O.DISS_LXF), (O.AVG_CHANDRASEKHAR, O.DISS_MATRIX), (O.AVG_STD, O.DISS_NONE),
        (O.AVG_CHANDRASEKHAR, O.DISS_SCALAR)]


def check(n, ne, tp, savg, sdiss, ends):
    b = F.LagrangeBasis("GLL", n)
    std = F.StdSegment(b, F.DGSEMrec(b), 3)
    mesh = F.CartesianMesh(1, [0.0], [1.0], [ne])
    state = np.array([1.1, 0.3, 2.5])
    first, code = [(None, None), (F.EulerSlipBC(), O.BC_SLIP), (F.EulerInflowBC(state), O.BC_INFLOW)][ends]
    if not ends:
        mesh.apply_periodicBCs(("1", "2"))
    eq = F.EulerEquation(1, GAMMA)
    disc = F.MultielementDisc(mesh, std, eq, F.SplitDivOperator(TP[tp](), surface(savg, sdiss)),
                              {"1": first, "2": F.EulerOutflowBC()} if ends else {})
    orc = O.OracleDisc(1, n, [ne], [0.0], [1.0], [0 if ends else 1], O.build_ops(n, "GLL"), O.EQ_EULER, [GAMMA],
                       O.VOL_SPLIT, tp, savg, sdiss, 1.0)
    if ends:
        orc.set_bc(0, code, state)
        orc.set_bc(1, O.BC_OUTFLOW)
    Q = random_euler_state(orc.coords()[0], 1, seed=n, amp=0.3, smooth=False)
    dQ = disc.new_state()
    F.rhs_(dQ, disc.to_device(Q), F.EquationConfig(disc, eq))
    disc.check()
    got, ref = disc.to_host(dQ), orc.rhs(Q)
    if tp != O.TP_CHANDRASEKHAR and savg == O.AVG_STD:
        assert np.array_equal(got, ref)
    else:
        assert np.max(np.abs(got - ref) / np.max(np.abs(ref), axis=0)) <= 1e-12


@pytest.mark.parametrize("surf", range(len(SURF)))
@pytest.mark.parametrize("n", range(2, 9))
def test_rhs_matches_oracle(n, surf):
    tp = (O.TP_CHANDRASEKHAR, O.TP_KENNEDY_GRUBER, O.TP_STDAVG)[(n + surf) % 3]
    for ne, ends in ((1, 1), (20, 2), (131, 0)):
        check(n, ne, tp, *SURF[surf], ends)


@pytest.mark.parametrize("extra", [0, 1])
@pytest.mark.parametrize("n", [2, 5, 8])
def test_most_blocks(n, extra):
    epb = 64 if n == 2 else 128 // (n * (n - 1) // 2)
    for surf in SURF[:2]:
        check(n, 1024 * epb + extra, O.TP_KENNEDY_GRUBER, *surf, 1)
