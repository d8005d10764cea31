"""Which kernel a discretisation runs (flou_hip_kernel_name): the forms, geometries and precisions
that have a kernel of their own, and what falls to the general one."""
import pytest

import flouhip as F
from cases import warp

pytestmark = pytest.mark.gpu
pytest.importorskip("torch")

LXF = F.LxF(F.StdAverage(), 1.0)
MATRIX = F.MatrixDissipation(F.ChandrasekharAverage(), 1.0)
CH, KG, STD = F.ChandrasekharAverage(), F.KennedyGruber(), F.StdAverage()


def disc(nd, n, nel, op, precision="fp64", curved=False, nodes="GLL", eq=None):
    b = F.LagrangeBasis(nodes, n)
    eq = eq or F.EulerEquation(nd, 1.4)
    std = [None, F.StdSegment, F.StdQuad, F.StdHex][nd](b, F.DGSEMrec(b), 1 if isinstance(eq, F.LinearAdvection) else nd + 2)
    mesh = F.CartesianMesh(nd, (0.0,) * nd, (1.0,) * nd, nel)
    mesh.apply_periodicBCs(*[(str(2 * k + 1), str(2 * k + 2)) for k in range(nd)])
    if curved:
        mesh.apply_mapping(warp)
    return F.MultielementDisc(mesh, std, eq, op, precision=precision)


@pytest.mark.parametrize("rhs,adjoint,args", [
    ("k_split", "k_svjp", (2, 4, [3, 3], F.SplitDivOperator(CH, LXF))),
    ("k_split", "k_svjp", (3, 5, [2, 2, 2], F.SplitDivOperator(KG, LXF))),
    ("k_split", "k_vjp", (2, 6, [3, 3], F.SplitDivOperator(CH, LXF))),
    ("k_split_1d", "k_vjp", (1, 3, [20], F.SplitDivOperator(CH, MATRIX))),
    ("k_split", "k_vjp", (1, 8, [4200], F.SplitDivOperator(CH, LXF))),
    ("k_plain", "k_vjp", (1, 8, [4200], F.SplitDivOperator(CH, MATRIX))),
    ("k_plain", "k_vjp", (2, 4, [3, 3], F.SplitDivOperator(CH, MATRIX))),
    ("k_split_curved", "k_svjp", (3, 5, [2, 2, 2], F.SplitDivOperator(CH, LXF), "fp64", True)),
    ("k_split_curved", "k_vjp", (2, 6, [3, 3], F.SplitDivOperator(STD, LXF), "fp64", True)),
    ("k_strong", "k_vjp", (3, 5, [2, 2, 2], F.StrongDivOperator(LXF))),
    ("k_strong", "k_vjp", (3, 5, [2, 2, 2], F.StrongDivOperator(LXF), "fp32")),
    ("k_plain", "k_vjp", (3, 5, [2, 2, 2], F.StrongDivOperator(LXF), "fp64", True)),
    ("k_hybrid_lines", "", (2, 6, [5, 3], F.HybridDivOperator(CH, MATRIX, 1.0))),
    ("k_hybrid_lines", "", (1, 4, [30], F.HybridDivOperator(CH, MATRIX, 1.0), "fp32")),
    ("k_hybrid", "", (2, 6, [60, 60], F.HybridDivOperator(CH, MATRIX, 1.0))),
    ("k_hybrid", "", (3, 4, [2, 2, 2], F.HybridDivOperator(CH, MATRIX, 1.0))),
    ("k_plain", "", (2, 4, [3, 3], F.SplitDivOperator(CH, LXF), "fp64", False, "GL")),
    ("k_fast", "k_fvjp", (3, 6, [2, 2, 2], F.SplitDivOperator(CH, LXF), "fp32")),
    ("k_fastc", "k_fvjp", (3, 7, [2, 2, 2], F.SplitDivOperator(CH, LXF), "fp32", True)),
], ids=lambda x: str(x) if isinstance(x, str) else "-".join(map(str, x[:3])).replace(" ", ""))
def test_kernel_names(rhs, adjoint, args):
    d = disc(*args)
    assert (d.kernel_name(), d.kernel_name(adjoint=True)) == (rhs, adjoint)


def test_plain_option():
    d = disc(3, 6, [2, 2, 2], F.SplitDivOperator(CH, LXF), "fp32")
    d.set_option(1, 1)
    assert (d.kernel_name(), d.kernel_name(adjoint=True)) == ("k_plain", "k_vjp")
