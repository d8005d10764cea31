"""A node of exactly zero density under the Chandrasekhar two-point flux raises DomainError.

With a momentum its pressure is -inf and β = -0, and the logarithm's argument β₁/β₂ is -inf or -0: the
reference stops at the logarithm of a negative number.  The node lies inside an element, where no
surface flux looks at it.
"""
import numpy as np
import pytest

import flouhip as F
from cases import random_euler_state
from test_gpu_hybrid import surface
from test_gpu_split_curved_fp64 import build as build_curved
from test_gpu_split_fp64 import build as build_axis
import oracle_lib as O

pytestmark = pytest.mark.gpu
pytest.importorskip("torch")


def check(disc, eq, orc, X, nd, n):
    Q = random_euler_state(X, nd, seed=n, amp=0.3, smooth=False)
    Q[sum((n // 2) * n ** k for k in range(nd)), 0] = 0.0
    with pytest.raises(ArithmeticError):
        orc.rhs(Q)
    F.rhs_(disc.new_state(), disc.to_device(Q), F.EquationConfig(disc, eq))
    with pytest.raises(F.DomainError):
        disc.check()


@pytest.mark.parametrize("nd,n,nel", [(1, 4, [9]), (1, 8, [4200]), (2, 5, [4, 3]), (3, 5, [2, 2, 2])])
def test_axis_aligned(nd, n, nel):
    disc, eq, orc = build_axis(nd, n, nel, "ch", True, False)
    check(disc, eq, orc, orc.coords()[0], nd, n)


@pytest.mark.parametrize("nd,n,nel", [(2, 5, [4, 3]), (3, 5, [2, 2, 2])])
def test_curved(nd, n, nel):
    disc, eq, orc, X = build_curved(nd, n, "ch", True, False, nel)
    check(disc, eq, orc, X, nd, n)


def test_small_1d_mesh_with_matrix_dissipation():
    b = F.LagrangeBasis("GLL", 4)
    mesh = F.CartesianMesh(1, [0.0], [1.0], [9]).apply_periodicBCs(("1", "2"))
    eq = F.EulerEquation(1, 1.4)
    op = F.SplitDivOperator(F.ChandrasekharAverage(), surface(O.AVG_CHANDRASEKHAR, O.DISS_MATRIX))
    disc = F.MultielementDisc(mesh, F.StdSegment(b, F.DGSEMrec(b), 3), eq, op)
    assert disc.kernel_name() == "k_split_1d"
    orc = O.OracleDisc(1, 4, [9], [0.0], [1.0], [1], O.build_ops(4, "GLL"), O.EQ_EULER, [1.4], O.VOL_SPLIT,
                       O.TP_CHANDRASEKHAR, O.AVG_CHANDRASEKHAR, O.DISS_MATRIX, 1.0)
    check(disc, eq, orc, orc.coords()[0], 1, 4)
