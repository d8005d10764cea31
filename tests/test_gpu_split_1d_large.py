"""k_split in 1-D (csrc/rhs_split.hip) against the oracle: meshes too large for the kernel of small ones.

Every node count and two-point flux, with and without LxF, walls, partial last blocks; bounds of
test_gpu_split_fp64.  (With few elements 1-D meshes run another kernel.)
"""
import pytest

import flouhip as F
from cases import random_euler_state
from test_gpu_split_fp64 import build, check

pytestmark = pytest.mark.gpu
pytest.importorskip("torch")


@pytest.mark.parametrize("tp", ["std", "ch", "kg"])
@pytest.mark.parametrize("n", range(2, 9))
def test_rhs_matches_oracle(n, tp):
    epb = 64 if n == 2 else 128 // (n * (n - 1) // 2)
    for lxf, walls in ((True, n % 2 == 0), (False, n % 2 == 1)):
        disc, eq, orc = build(1, n, [768 * epb + 1], tp, lxf, walls)
        assert disc.kernel_name() == "k_split"
        Q = random_euler_state(orc.coords()[0], 1, seed=n, amp=0.3, smooth=lxf)
        dQ = disc.new_state()
        F.rhs_(dQ, disc.to_device(Q), F.EquationConfig(disc, eq))
        disc.check()
        check(disc.to_host(dQ), orc.rhs(Q), tp)
