"""The FP64 line adjoint of axis-aligned elements (csrc/vjp_split.hip) against the oracle.

<W, J V> from the oracle's dual-number JVP against <J^T W, V> from the kernel, three random
directions each, at every node count of the kernel (4..8; block sizes and spare lanes differ),
2-D and 3-D, partial last blocks, all three two-point fluxes, with and without LxF, walls,
states on the series and on the logarithm's branch of the means.  Bound 1e-12 of Σ|W·JV|, as the
adjoint's other dot-product tests.
"""
import numpy as np
import pytest

import flouhip as F
import oracle_lib as O
from cases import random_euler_state
from flouhip import adjoint as A
from test_gpu_split_fp64 import build

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")



def elements(nd, n, tp):
    """The fewest elements at which the kernel is taken, or a few; partial last blocks."""
    if tp != "std" and nd == 2 and n >= 6:
        return [53, 29] if n == 6 else [61, 51]
    if tp != "std" and nd == 3 and n == 6:
        return [5, 8, 7]
    return {2: [7, 3], 3: [3, 2, 1]}[nd]


def dots(disc, orc, Q, seed):
    rng = np.random.default_rng(seed)
    W = rng.standard_normal(Q.shape)
    acc0 = rng.standard_normal(Q.shape)
    Qbar = disc.to_device(acc0)  # rhs_vjp accumulates
    A.rhs_vjp(Qbar, disc.to_device(W), disc.to_device(Q), disc)
    JTW = disc.to_host(Qbar) - acc0
    for _ in range(3):
        V = rng.standard_normal(Q.shape)
        _, JV = orc.rhs_jvp(Q, V)
        assert abs(np.sum(W * JV) - np.sum(JTW * V)) <= 1e-12 * np.sum(np.abs(W * JV))


@pytest.mark.parametrize("tp", ["std", "ch", "kg"])
@pytest.mark.parametrize("nd,n", [(nd, n) for nd in (2, 3) for n in range(4, 9)])
def test_dot_product_with_oracle_jvp(nd, n, tp):
    disc, eq, orc = build(nd, n, elements(nd, n, tp), tp, n != 5, n in (4, 7))
    X = orc.coords()[0]
    dots(disc, orc, random_euler_state(X, nd, seed=n, amp=0.05), 3 * n)
    # neighbouring densities and pressures far apart: the logarithm's branch
    rough = random_euler_state(X, nd, seed=n, amp=0.2, smooth=False)
    rough[::3] *= 2.5
    dots(disc, orc, rough, 3 * n + 1)


def test_uniform_state():
    """Equal wave speeds on every face (the maximum's tie) and u = 0 in every mean."""
    disc, eq, orc = build(2, 5, [5, 4], "ch", True, False)
    Q = np.tile(np.array([1.1, 0.3, -0.2, 2.6]), (orc.coords()[0].shape[0], 1))
    dots(disc, orc, np.asfortranarray(Q), 1)


@pytest.mark.parametrize("solver,scheme", [(F.SSPRK33, O.RK_SSPRK33), (F.CarpenterKennedy2N54, O.RK_CK2N54)])
def test_rk_step(solver, scheme):
    disc, eq, orc = build(3, 5, [2, 3, 1], "ch", True, False)
    Q = random_euler_state(orc.coords()[0], 3, seed=4, amp=0.1)
    rng = np.random.default_rng(5)
    V, W = rng.standard_normal(Q.shape), rng.standard_normal(Q.shape)
    _, JV = orc.rk_run_jvp(scheme, Q, V, 1e-3, 1)
    stages = [disc.to_device(Q)] + [disc.new_state() for _ in range(solver.nstages - 1)]
    A.rk_step_record(disc, solver, 1e-3, stages, disc.new_state())
    ubar = disc.to_device(W)
    A.rk_step_vjp(disc, solver, 1e-3, stages, ubar)
    lhs, rhs = np.sum(W * JV), np.sum(disc.to_host(ubar) * V)
    assert abs(lhs - rhs) <= 1e-12 * np.sum(np.abs(W * JV))
