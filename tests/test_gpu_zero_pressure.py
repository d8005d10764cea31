"""A node of exactly zero pressure under the Chandrasekhar two-point flux, against the oracle.

The node's β = ρ/(2p) is infinite.  The reference's flux then has a finite mass and momentum (the mean
pressure is (ρ₁+ρ₂)/(2(β₁+β₂)) = 0) and NaN in its energy only: the kernels have to be NaN in the
same entries and agree in all others.  Sizes that reach the 1-D kernel of small meshes, the 1-D kernel
of large ones, the 2-D and 3-D kernels of axis-aligned elements and those of curved ones.
"""
import numpy as np
import pytest

import flouhip as F
from cases import random_euler_state
from test_gpu_split_curved_fp64 import build as build_curved
from test_gpu_split_fp64 import build as build_axis

pytestmark = pytest.mark.gpu
pytest.importorskip("torch")


@pytest.mark.parametrize("nd,n,nel,curved", [(1, 4, [9], False), (1, 8, [1024 * 4 + 3], False), (2, 5, [4, 3], False),
                                             (3, 4, [2, 2, 2], False), (2, 5, [4, 3], True), (3, 4, [2, 2, 2], True)])
def test_nan_in_the_energy_only(nd, n, nel, curved):
    if curved:
        disc, eq, orc, X = build_curved(nd, n, "ch", True, False, nel)
    else:
        disc, eq, orc = build_axis(nd, n, nel, "ch", True, False)
        X = orc.coords()[0]
    Q = random_euler_state(X, nd, seed=n, amp=0.3, smooth=False)
    node = X.shape[0] // 2
    Q[node, 0] = 1.0
    Q[node, 1:nd + 1] = 0.5
    Q[node, nd + 1] = 0.5 * nd * 0.25  # |m|²/(2ρ): no internal energy
    dQ = disc.new_state()
    F.rhs_(dQ, disc.to_device(Q), F.EquationConfig(disc, eq))
    disc.check()
    got, ref = disc.to_host(dQ), orc.rhs(Q)
    assert np.isfinite(ref[:, :nd + 1]).all() and np.isnan(ref[:, nd + 1]).any()
    assert np.array_equal(np.isnan(got), np.isnan(ref))
    assert np.nanmax(np.abs(got - ref) / np.nanmax(np.abs(ref), axis=0)) <= 4e-15 * max(n, 4) ** 2
