"""The FP64 line adjoint (csrc/vjp_split.hip) at the fewest elements that take it, against the oracle.

Dot products as in test_gpu_split_vjp_fp64 (bound 1e-12 of Σ|W·JV|), smooth states and states on the logarithm's
branch, with a partial last block where the element count leaves one.
"""
import pytest

from cases import random_euler_state
from test_gpu_split_curved_fp64 import build as build_curved
from test_gpu_split_fp64 import build as build_axis
from test_gpu_split_vjp_fp64 import dots

pytestmark = pytest.mark.gpu
pytest.importorskip("torch")


@pytest.mark.parametrize("nd,n,tp,nel,curved", [
    (2, 5, "ch", [96, 80], False), (2, 5, "kg", [83, 62], False), (2, 6, "ch", [88, 64], False),
    (2, 6, "kg", [61, 59], False), (2, 7, "ch", [83, 68], False), (2, 7, "kg", [61, 59], False),
    (2, 8, "ch", [83, 68], False), (2, 8, "kg", [61, 59], False), (3, 5, "ch", [11, 10, 7], False),
    (3, 6, "ch", [8, 8, 4], False), (3, 6, "kg", [11, 6, 4], False),
    (2, 5, "ch", [101, 77], True), (2, 5, "std", [80, 64], True), (2, 6, "ch", [83, 68], True),
    (2, 6, "kg", [64, 56], True), (2, 6, "std", [61, 59], True), (2, 7, "ch", [88, 64], True),
    (2, 7, "std", [61, 59], True), (3, 6, "kg", [3, 2, 1], True)])
def test_dot_product_with_oracle_jvp(nd, n, tp, nel, curved):
    if curved:
        disc, eq, orc, X = build_curved(nd, n, tp, True, n != 6, nel)
    else:
        disc, eq, orc = build_axis(nd, n, nel, tp, True, n != 6)
        X = orc.coords()[0]
    assert disc.kernel_name(adjoint=True) == "k_svjp"
    dots(disc, orc, random_euler_state(X, nd, seed=n, amp=0.05), 3 * n)
    rough = random_euler_state(X, nd, seed=n, amp=0.2, smooth=False)
    rough[::3] *= 2.5
    dots(disc, orc, rough, 3 * n + 1)
