"""The FP64 line adjoint of curved elements (csrc/vjp_split.hip) against the oracle.

<W, J V> from the oracle's dual-number JVP against <J^T W, V> from the kernel, at every node count 4..8 in
2-D and 3-D, partial last blocks, all three two-point fluxes, with and without LxF, walls and outflow on
one axis, states on the series and on the logarithm's branch of the means.  Bound 1e-12 of
Σ|W·JV|, as the adjoint's other dot-product tests.
"""
import pytest

from cases import random_euler_state
from test_gpu_split_curved_fp64 import build
from test_gpu_split_vjp_fp64 import dots

pytestmark = pytest.mark.gpu
pytest.importorskip("torch")


@pytest.mark.parametrize("tp", ["std", "ch", "kg"])
@pytest.mark.parametrize("nd,n", [(nd, n) for nd in (2, 3) for n in range(4, 9)])
def test_dot_product_with_oracle_jvp(nd, n, tp):
    # 2-D with more than 4 nodes: the fewest elements that take the kernel, and a few over
    nel = None if nd == 3 or n == 4 else (67, 62)
    disc, eq, orc, X = build(nd, n, tp, n != 5, n in (4, 7), nel)
    dots(disc, orc, random_euler_state(X, nd, seed=n, amp=0.05), 3 * n)
    rough = random_euler_state(X, nd, seed=n, amp=0.2, smooth=False)
    rough[::3] *= 2.5
    dots(disc, orc, rough, 3 * n + 1)
