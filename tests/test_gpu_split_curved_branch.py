"""The curved FP64 split form at the branch point of the logarithmic mean, against the oracle.

Neighbouring nodes' densities (and β) are as 11 to 9, where u = 0.01 to rounding and the mean's two
branches are 1e-9 apart: the kernel has to take the reference's.  Bound as in test_gpu_split_curved_fp64.
"""
import numpy as np
import pytest

import flouhip as F
from cases import random_euler_state
from test_gpu_curved import rel_err
from test_gpu_split_curved_fp64 import NEL, build

pytestmark = pytest.mark.gpu
pytest.importorskip("torch")


@pytest.mark.parametrize("nd,n", [(2, 5), (3, 4), (3, 7)])
def test_takes_the_references_branch(nd, n):
    disc, eq, orc, X = build(nd, n, "ch", True, False)
    rng = np.random.default_rng(n)
    Q = random_euler_state(X, nd, seed=n, amp=0.1)
    u = Q[:, 1:nd + 1] / Q[:, :1]
    scale = np.repeat(rng.integers(1, 200, size=int(np.prod(NEL[nd]))), n ** nd)  # alike within an element
    rho = np.where(np.arange(X.shape[0]) % 2 == 0, 0.11, 0.09) * scale
    Q[:, 0] = rho
    Q[:, 1:nd + 1] = rho[:, None] * u
    Q[:, nd + 1] = 0.5 * scale / 0.4 + 0.5 * rho * np.sum(u * u, axis=1)
    dQ = disc.new_state()
    F.rhs_(dQ, disc.to_device(Q), F.EquationConfig(disc, eq))
    disc.check()
    assert rel_err(disc.to_host(dQ), orc.rhs(Q)) <= 4e-15 * max(n, 4) ** 2
